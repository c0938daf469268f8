// k_acoustic.hip -- acoustic (fluid potential) element stiffness for NGLL=5.
//
// Restates compute_forces_acoustic.F90:35-726: chi'' -= div((1/rho) grad chi) in weak form. The lane
// layout is that of k_elastic_line (k_elastic.hip), for one component. Compiled twice like
// k_elastic.hip (SF_EXACT = 1: no fused multiply-add, the reference's rounding).
#include "elastic_point.h"

#ifndef SF_EXACT
#define SF_EXACT 1
#endif
#if SF_EXACT
#define SFX(name) name##_exact
#define SF_VNS v_exact
#else
#define SFX(name) name##_fast
#define SF_VNS v_fast
#endif

namespace sf {
namespace SF_VNS {

// The local forces are stored, one float per slot (gather_slot), and summed per global point by the
// update that follows (k_gather_update<1>). A 128-lane workgroup takes five elements, a lane one line
// of five points at a time: lane (el, c) holds the gamma column of c = i + 5 j in registers and the xi
// row 5 c .. 5 c + 4 and the eta row (c % 5) + 25 (c / 5) + 5 l in LDS, the coefficients in scalar
// registers. Plane A holds chi, then the xi derivatives, the xi products and their divergence, plane
// B the same for eta.
// Bound by HBM: 28 B per local point with the index and the density, 96 MB on 40x40x30 elements, 22 us
// (4.3 TB/s, near the rate of a large copy) where a lane per column with float atomics took 82 us;
// on 64x64x4 36 -> 12 us, on 19x17x4, in eight colour launches before, 53 -> 5. The sum, fused with the
// corrector, takes 18.6 us on 40x40x30 (20.9 with one element's slots after the other's); a corrector
// alone took 10.
__global__ void __launch_bounds__(128) k_acoustic(AcousticArgs A, GLLk G) {
  constexpr int PL = 626;
  __shared__ realw sA[PL], sB[PL];
  __shared__ realw sW[25];
  const int t = threadIdx.x;
  const bool lane = t < 125;                       // lanes 125..127 shadow the last element's first points
  const int el = lane ? t / 25 : 4, c = lane ? t - 25 * el : t - 125;
  const int i = c % 5, j = c / 5;
  // blocks b, b + 8, ... (one XCD) take one contiguous range of elements
  const int nb = gridDim.x, q = nb >> 3, r8 = nb & 7, xc = blockIdx.x & 7;
  const int ie = (xc * q + (xc < r8 ? xc : r8) + (int)(blockIdx.x >> 3)) * 5 + el;
  const bool active = lane && ie < A.nelem;
  const int e = A.elems[ie < A.nelem ? ie : A.nelem - 1];
  const int64_t ep = (int64_t)e * 125 + c;         // local point of k = 0
  const int irr = A.irregular[e];
  const int64_t jp = (int64_t)(irr ? irr - 1 : 0) * 125 + c;
  if (t < 25) sW[t] = G.wxy[t];
  realw rho[5], d3[5];
  {
    int g[5];
    realw chi[5];
#pragma unroll
    for (int k = 0; k < 5; k++) g[k] = A.ibool[ep + 25 * k];
#pragma unroll
    for (int k = 0; k < 5; k++) chi[k] = A.pot[g[k]];
#pragma unroll
    for (int k = 0; k < 5; k++) rho[k] = A.rho[ep + 25 * k];
    if (lane) {
#pragma unroll
      for (int k = 0; k < 5; k++) sA[el * 125 + c + 25 * k] = chi[k];
    }
    line_gradient(G, chi, d3);
  }
  lds_barrier();
  const int bx = el * 125 + 5 * c, by = el * 125 + i + 25 * j;  // first points of the lane's two rows
  realw x[5];
  {
    realw r[5], y[5];
#pragma unroll
    for (int l = 0; l < 5; l++) {
      r[l] = sA[bx + l];
      y[l] = sA[by + 5 * l];
    }
    line_gradient(G, r, x);
    line_gradient(G, y, r);
    if (lane) {
#pragma unroll
      for (int l = 0; l < 5; l++) sB[by + 5 * l] = r[l];
    }
  }
  lds_barrier();                                   // every row of chi has been read
  if (lane) {
#pragma unroll
    for (int l = 0; l < 5; l++) sA[bx + l] = x[l];
  }
  lds_barrier();
#pragma unroll
  for (int k = 0; k < 5; k++) {
    const int b = el * 125 + c + 25 * k;
    const realw a1 = sA[b], a2 = sB[b], a3 = d3[k];
    const realw rho_invl = (realw)1 / rho[k];
    realw t1, t2;
    if (irr) {
      const JacPt J = load_jac(A.jac, A.jac_plane, jp + 25 * k);
      const realw dpdx = sum3(J.xix, a1, J.etax, a2, J.gax, a3);
      const realw dpdy = sum3(J.xiy, a1, J.etay, a2, J.gay, a3);
      const realw dpdz = sum3(J.xiz, a1, J.etaz, a2, J.gaz, a3);
      t1 = rho_invl * J.jac * sum3(J.xix, dpdx, J.xiy, dpdy, J.xiz, dpdz);
      t2 = rho_invl * J.jac * sum3(J.etax, dpdx, J.etay, dpdy, J.etaz, dpdz);
      d3[k] = rho_invl * J.jac * sum3(J.gax, dpdx, J.gay, dpdy, J.gaz, dpdz);
    } else {
      const realw jl = A.jacobian_regular, xr = A.xix_regular;
      t1 = rho_invl * jl * xr * xr * a1;
      t2 = rho_invl * jl * xr * xr * a2;
      d3[k] = rho_invl * jl * xr * xr * a3;
    }
    if (lane) {
      sA[b] = t1;
      sB[b] = t2;
    }
  }
  lds_barrier();
  {
    realw r[5], y[5], o[5];
#pragma unroll
    for (int l = 0; l < 5; l++) {
      r[l] = sA[bx + l];
      y[l] = sB[by + 5 * l];
    }
    line_divergence(G, r, o);
    if (lane) {
#pragma unroll
      for (int l = 0; l < 5; l++) sA[bx + l] = o[l];
    }
    line_divergence(G, y, o);
    if (lane) {
#pragma unroll
      for (int l = 0; l < 5; l++) sB[by + 5 * l] = o[l];
    }
    line_divergence(G, d3, o);
#pragma unroll
    for (int k = 0; k < 5; k++) d3[k] = o[k];
  }
  lds_barrier();
  if (!active) return;
  const realw w3 = sW[i * 5 + j];
  const int slot = gather_slot(ie, j, i, A.eb);    // of k = 0
#pragma unroll
  for (int k = 0; k < 5; k++) {
    const int b = el * 125 + c + 25 * k;
    A.local_out[slot + k * 25 * A.eb] = sum3(sW[j * 5 + k], sA[b], sW[i * 5 + k], sB[b], w3, d3[k]);
  }
}

}  // namespace SF_VNS
using namespace SF_VNS;

void SFX(launch_acoustic)(hipStream_t s, const AcousticArgs& a) {
  if (a.nelem <= 0) return;
  hipLaunchKernelGGL(k_acoustic, dim3((a.nelem + 4) / 5), dim3(128), 0, s, a, g_gll_host);
  SF_LAUNCH_CHECK("k_acoustic");
}

}  // namespace sf
