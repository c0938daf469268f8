// k_elastic.hip -- isotropic elastic / viscoelastic (3 SLS) element stiffness for NGLL=5.
//
// Restates compute_forces_viscoelastic.F90:33-962 (with the memory update of
// compute_element_att_memory.f90:28-156) as two gfx950 kernels: k_elastic_line without attenuation
// (described there) and k_elastic_pt with it:
//   * a 128-thread workgroup (two wave64s) processes one element; lane p owns the GLL point
//     p = i + 5 j + 25 k (125 of the 128 lanes busy) and all three contractions read the element
//     tile staged in LDS;
//   * the local forces are stored, three floats per local point, and summed per global point by the
//     update that follows (k_gather_update): one launch over all elements, no atomics, no colours.
//     Against float atomics the viscoelastic launch on 64x64x32 elements (28 layers solid) went from
//     854 to 620 us (the atomics' write-back was 15 % of its traffic), and against eight colour
//     launches the elastic one from 277 to 187 us there and from 41 to 14 us on 20x20x20 (both of
//     them this kernel without attenuation, which k_elastic_line has replaced);
//   * workgroup ids are remapped so each XCD (8 per chip, dispatched round-robin) walks one
//     contiguous range of elements and keeps the shared points of neighbours in its own L2.
// The arithmetic order of every sum follows the reference (the five terms of each
// contraction left to right, etc.). This file is compiled twice: with -ffp-contract=off
// (SF_EXACT=1, same rounding as the CPU reference) and with FMA contraction (SF_EXACT=0).
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
// each build variant keeps its kernels in its own namespace (template instantiations of the
// two variants would otherwise be merged by the linker)
namespace SF_VNS {

__device__ __forceinline__ int xcd_remap(int b, int nb) {
  // bijection: blocks b, b+8, b+16, ... (one XCD) get one contiguous logical range
  const int q = nb >> 3, r = nb & 7, x = b & 7;
  return x * q + (x < r ? x : r) + (b >> 3);
}

// stored strain (6 planes) and SLS factors (table row or planes) of one point
__device__ __forceinline__ void load_factors(const ElasticArgs& A, int64_t ep, int64_t nl, realw fcv[3],
                                             realw fckv[3]) {
  if (A.fc_index) {
    const int r = A.fc_index[ep];
#pragma unroll
    for (int s = 0; s < 3; s++) {
      fcv[s] = A.fc_table[s * A.fc_rows + r];
      fckv[s] = A.fc_table[(3 + s) * A.fc_rows + r];
    }
  } else {
#pragma unroll
    for (int s = 0; s < 3; s++) {
      fcv[s] = A.fc[s * nl + ep];
      fckv[s] = A.fck[s * nl + ep];
    }
  }
}

__device__ __forceinline__ void load_att_state(const ElasticArgs& A, int e, int q, int64_t ep, int64_t nl, realw Sn[6],
                                               realw fcv[3], realw fckv[3]) {
#pragma unroll
  for (int cc = 0; cc < 6; cc++) Sn[cc] = A.eps[eps_idx(e, cc, q)];
  if (A.fc_index) {
    const int r = A.fc_index[ep];
#pragma unroll
    for (int s = 0; s < 3; s++) {
      fcv[s] = A.fc_table[s * A.fc_rows + r];
      fckv[s] = A.fc_table[(3 + s) * A.fc_rows + r];
    }
  } else {
#pragma unroll
    for (int s = 0; s < 3; s++) {
      fcv[s] = A.fc[s * nl + ep];
      fckv[s] = A.fck[s * nl + ep];
    }
  }
}

// Point-per-lane variant: a 128-thread workgroup (two wave64s) processes one element and lane p
// holds the GLL point p = i + 5 j + 25 k (lanes 125..127 shadow point 124 and store nothing).
// All three contractions read the element tile from LDS, so no lane carries a column of state
// between phases; the per-point state (memory variables, stored strain, SLS factors, moduli,
// Jacobian terms) is loaded before the first barrier and is in flight while the tile is
// gathered.
// AV selects how the attenuation state is scheduled (the "att_variant" tuning switch; same
// results):
// 0 every per-point array is loaded before the first barrier; 1 only the memory variables are,
// the stored strain and SLS factors are loaded where the memory update needs them (fewer live
// registers); 2 as 1 with the register budget capped for 5 waves per SIMD; 3 as 0 with that cap;
// 4 loads the memory variables and stored strain straight into LDS (global_load_lds, no
// registers held while they are in flight; each lane reads back its own point), which frees
// registers for 5 waves per SIMD; the stress products then reuse those LDS planes.
typedef __attribute__((address_space(3))) void* sf_lds_ptr;
typedef __attribute__((address_space(1))) void* sf_global_ptr;

template <int AV>
__global__ void __launch_bounds__(128) __attribute__((amdgpu_waves_per_eu(AV >= 2 ? 5 : 1)))
k_elastic_pt(ElasticArgs A, GLLk G) {
  constexpr bool LATE = AV == 1 || AV == 2;
  constexpr bool DL = AV == 4;
  __shared__ realw sU[6][128];            // u (0..2) and dt*v (3..5)
  __shared__ realw sX[DL ? 24 : 9][128];  // stress products (planes 0..8); with DL first the state
  realw(*const sT)[128] = sX;             // t1 (0..2), t2 (3..5), t3 (6..8)
  __shared__ realw sG[SF_NGLL_TABLE];     // hprime, hprimewgll, wgllwgll (+ folded, elastic_point.h)
  const int p = threadIdx.x;
  const bool active = p < 125;
  stage_gll(sG, G, p);
  const int ie = xcd_remap(blockIdx.x, gridDim.x);  // grid = one workgroup per listed element
  const int e = A.elems[ie];
  const int q = active ? p : 124;
  const int k = q / 25, j = (q / 5) % 5, i = q % 5;
  const int64_t ep = (int64_t)e * 125 + q;
  const int64_t nl = A.nloc;
  const int g = A.ibool[ep];
  const int irr = A.irregular[e];
  JacPt J = {};
  realw jacl = A.jacobian_regular;
  if (irr) {
    J = load_jac(A.jac, A.jac_plane, (int64_t)(irr - 1) * 125 + q);
    jacl = J.jac;
  }
  const float2 km = A.kappamu[ep];
  realw Rv[6][3], Sn[6], fcv[3], fckv[3];
  if (!DL) {
#pragma unroll
    for (int cc = 0; cc < 6; cc++)
#pragma unroll
      for (int s = 0; s < 3; s++) Rv[cc][s] = A.R[r_idx(e, cc * 3 + s, q)];
    if (!LATE) load_att_state(A, e, q, ep, nl, Sn, fcv, fckv);
  }
  if (DL) load_factors(A, ep, nl, fcv, fckv);
  {
    const realw* d = A.displ + 3 * (int64_t)g;
    const realw u0 = d[0], u1 = d[1], u2 = d[2];
    const realw* v = A.veloc + 3 * (int64_t)g;
    const realw v0 = v[0], v1 = v[1], v2 = v[2];
    sU[0][p] = u0; sU[1][p] = u1; sU[2][p] = u2;
    sU[3][p] = A.deltat * v0; sU[4][p] = A.deltat * v1; sU[5][p] = A.deltat * v2;
  }
  __syncthreads();
  if (DL) {
    // after the barrier (whose release would wait for them, as they write LDS): R planes 0..17 and
    // strain planes 0..5 of this element into sX[plane][lane], in flight during the gradient;
    // each lane reads back only its own slots, after its own wait
    __builtin_amdgcn_sched_barrier(0);
    const int w64 = p & 64;
#pragma unroll
    for (int pl = 0; pl < 18; pl++)
      __builtin_amdgcn_global_load_lds((sf_global_ptr)(A.R + r_idx(e, pl, q)), (sf_lds_ptr)&sX[pl][w64], 4, 0, 0);
#pragma unroll
    for (int c = 0; c < 6; c++)
      __builtin_amdgcn_global_load_lds((sf_global_ptr)(A.eps + eps_idx(e, c, q)), (sf_lds_ptr)&sX[18 + c][w64], 4,
                                       0, 0);
    __builtin_amdgcn_sched_barrier(0);
  }

  const realw ONE_THIRD = (realw)1 / (realw)3;
  const realw* hpg = gll_hp(sG, irr != 0);
  const Grad9 tg = tile_gradient<1>(sU[0], sU[1], sU[2], hpg, i, j, k);
  const Du9 du = map_gradient(tg, irr != 0, J, A.xix_regular);

  const Du9 st = map_gradient(tile_gradient_continue<1>(tg, sU[3], sU[4], sU[5], hpg, i, j, k), irr != 0, J,
                              A.xix_regular);
  const realw e_tr = (st.xx + st.yy + st.zz);
  const realw templ = ONE_THIRD * (st.xx + st.yy + st.zz);
  if (A.eps_tr3 && active) A.eps_tr3[ep] = templ;
  const realw e_xx = st.xx - templ;
  const realw e_yy = st.yy - templ;
  const realw e_xy = (realw)0.5 * (st.xy + st.yx);
  const realw e_xz = (realw)0.5 * (st.zx + st.xz);
  const realw e_yz = (realw)0.5 * (st.zy + st.yz);

  const realw kappal = km.x, mul = km.y;
  Sigma6 sg = iso_stress(du, kappal, mul);

  if (DL) {
    __builtin_amdgcn_s_waitcnt(0);  // the LDS-direct loads of this wave have landed
#pragma unroll
    for (int cc = 0; cc < 6; cc++)
#pragma unroll
      for (int s = 0; s < 3; s++) Rv[cc][s] = sX[cc * 3 + s][p];
#pragma unroll
    for (int c = 0; c < 6; c++) Sn[c] = sX[18 + c][p];
  }
  const realw rxx = (Rv[0][0] + Rv[0][1]) + Rv[0][2];
  const realw ryy = (Rv[1][0] + Rv[1][1]) + Rv[1][2];
  const realw rtr = (Rv[5][0] + Rv[5][1]) + Rv[5][2];
  sg.xx = sg.xx - rxx - rtr;
  sg.yy = sg.yy - ryy - rtr;
  sg.zz = sg.zz + rxx + ryy - rtr;
  sg.xy = sg.xy - ((Rv[2][0] + Rv[2][1]) + Rv[2][2]);
  sg.xz = sg.xz - ((Rv[3][0] + Rv[3][1]) + Rv[3][2]);
  sg.yz = sg.yz - ((Rv[4][0] + Rv[4][1]) + Rv[4][2]);
  if (active) {
    // memory-variable update (second-order RK) with old strain Sn and new strain Snp1
    if (LATE) load_att_state(A, e, q, ep, nl, Sn, fcv, fckv);
    const realw Snp1[6] = {e_xx, e_yy, e_xy, e_xz, e_yz, e_tr};
#pragma unroll
    for (int s = 0; s < 3; s++) {
      const realw flk = kappal * fckv[s];
      A.R[r_idx(e, 5 * 3 + s, q)] = A.alpha[s] * Rv[5][s] + flk * (A.beta[s] * Sn[5] + A.gamma[s] * Snp1[5]);
      const realw flm = mul * fcv[s];
#pragma unroll
      for (int cc = 0; cc < 5; cc++)
        A.R[r_idx(e, cc * 3 + s, q)] = A.alpha[s] * Rv[cc][s] + flm * (A.beta[s] * Sn[cc] + A.gamma[s] * Snp1[cc]);
    }
  }
  if (active) {
    realw* Ep = A.eps;
    Ep[eps_idx(e, 0, q)] = e_xx; Ep[eps_idx(e, 1, q)] = e_yy; Ep[eps_idx(e, 2, q)] = e_xy;
    Ep[eps_idx(e, 3, q)] = e_xz; Ep[eps_idx(e, 4, q)] = e_yz;
    Ep[eps_idx(e, 5, q)] = e_tr;
  }

  {
    realw t[9];
    stress_products<SF_FOLD, true>(sg, irr != 0, J, jacl, A.xix_regular, t);
#pragma unroll
    for (int m = 0; m < 9; m++) sT[m][p] = t[m];
  }
  lds_barrier();  // the memory-variable and strain stores drain during the divergence
  if (!active) return;

  realw f[3];
  tile_divergence<1>(&sT[0][0], 128, gll_hpw(sG, irr != 0), sG + 50, i, j, k, f);
  realw* o = A.local_out + 3 * (int64_t)gather_slot(ie, q / 5, i, A.eb);
  o[0] = f[0];
  o[1] = f[1];
  o[2] = f[2];
}

// Elastic stiffness without attenuation: a 128-lane workgroup takes five elements, a lane one line of
// five GLL points at a time (line_gradient, line_divergence). Lane (el, c) of 125 holds the gamma column
// of c = i + 5 j, whose contraction stays in its registers, and for the other two directions the xi row
// 5 c .. 5 c + 4 and the eta row (c % 5) + 25 (c / 5) + 5 l, read from and written back to LDS.
//
// k_elastic_pt reads 45 tile values and 15 coefficients from LDS per point and contraction stage,
// 123 reads in all; here it is 33 reads and 12 writes per point, and the coefficients sit in scalar
// registers. Planes A (u, then the xi derivatives, the xi products and their divergence) and B (the
// same for eta) are reused in place: a row is read and written by one lane, and a point's values are
// read and replaced by the lane of its column; only the xi derivatives need a barrier before they
// replace u. 15 KB of LDS per workgroup, 61 to 80 VGPRs, 5 waves per SIMD. Per launch against
// k_elastic_pt storing the same forces: 64x64x32 elements 187 -> 105 us (0.52 GB: the rate of a large
// copy), 20x20x20 14.3 -> 12.5, 24^3 with strain 22.2 -> 19.5, irregular 43x37x29 89 -> 87 (its 40 B of
// Jacobian terms per point were already the limit).
// REG: the regular elements of a mesh (FMA build: the mapping is folded into the tables, so that a regular
// element rounds the same whatever the mesh around it). A mesh with both kinds lists them before the
// irregular ones and its workgroups take one kind each. A step of 48x48x48 elements, half of them
// irregular: 294 us, with the choice per lane 325; 16x16x16: 22.1 and 21.5 (with a launch per kind 298 and
// 28.7).
constexpr int LINE_PL = 626;
template <bool STRAIN, bool REG>
__device__ __forceinline__ void elastic_line(const ElasticArgs& A, const GLLk& G, int n, const int* elems, int pos0,
                                             int block, int blocks, realw (&sA)[3][LINE_PL], realw (&sB)[3][LINE_PL],
                                             realw (&sW)[25]) {
  constexpr bool FOLD = REG && SF_FOLD;
  const int t = threadIdx.x;
  const bool lane = t < 125;                       // lanes 125..127 shadow the last element's first points
  const int el = lane ? t / 25 : 4, c = lane ? t - 25 * el : t - 125;
  const int i = c % 5, j = c / 5;
  const int ie = xcd_remap(block, blocks) * 5 + el;
  const bool active = lane && ie < n;
  const int e = elems[ie < n ? ie : n - 1];
  const int64_t ep = (int64_t)e * 125 + c;         // local point of k = 0
  const int irr = REG ? 0 : A.irregular[e];
  const int64_t jp = REG ? 0 : (int64_t)(irr ? irr - 1 : 0) * 125 + c;
  if (t < 25) sW[t] = G.wxy[t];
  float2 km[5];
  realw d3[5][3];
  {
    realw u[3][5];
    int g[5];
#pragma unroll
    for (int k = 0; k < 5; k++) g[k] = A.ibool[ep + 25 * k];
#pragma unroll
    for (int k = 0; k < 5; k++) {
      const realw* d = A.displ + 3 * (int64_t)g[k];
      u[0][k] = d[0]; u[1][k] = d[1]; u[2][k] = d[2];
    }
#pragma unroll
    for (int k = 0; k < 5; k++) km[k] = A.kappamu[ep + 25 * k];
    const int b = el * 125 + c;
#pragma unroll
    for (int a = 0; a < 3; a++) {
      if (lane) {
#pragma unroll
        for (int k = 0; k < 5; k++) sA[a][b + 25 * k] = u[a][k];
      }
      realw r[5];
      line_gradient(G, u[a], r);
#pragma unroll
      for (int k = 0; k < 5; k++) d3[k][a] = r[k];
    }
  }
  lds_barrier();
  const int bx = el * 125 + 5 * c, by = el * 125 + i + 25 * j;  // first points of the lane's two rows
  realw x[3][5];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    realw r[5], y[5];
#pragma unroll
    for (int l = 0; l < 5; l++) {
      r[l] = sA[a][bx + l];
      y[l] = sA[a][by + 5 * l];
    }
    line_gradient(G, r, x[a]);
    line_gradient(G, y, r);
    if (lane) {
#pragma unroll
      for (int l = 0; l < 5; l++) sB[a][by + 5 * l] = r[l];
    }
  }
  lds_barrier();                                   // every row of u has been read
  if (lane) {
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int l = 0; l < 5; l++) sA[a][bx + l] = x[a][l];
  }
  lds_barrier();
  const realw ONE_THIRD = (realw)1 / (realw)3;
#pragma unroll
  for (int k = 0; k < 5; k++) {
    const int b = el * 125 + c + 25 * k;
    const Grad9 tg = {sA[0][b], sA[1][b], sA[2][b], sB[0][b], sB[1][b], sB[2][b], d3[k][0], d3[k][1], d3[k][2]};
    JacPt J = {};
    realw jacl = A.jacobian_regular;
    if (!REG && irr) {
      J = load_jac(A.jac, A.jac_plane, jp + 25 * k);
      jacl = J.jac;
    }
    const Du9 du = map_gradient<FOLD>(tg, irr != 0, J, A.xix_regular);
    if (STRAIN) {
      const realw templ = ONE_THIRD * (du.xx + du.yy + du.zz);
      if (active) {
        if (A.eps_tr3) A.eps_tr3[ep + 25 * k] = templ;
        const int p = c + 25 * k;
        A.eps[eps_idx(e, 0, p)] = du.xx - templ;
        A.eps[eps_idx(e, 1, p)] = du.yy - templ;
        A.eps[eps_idx(e, 2, p)] = (realw)0.5 * (du.xy + du.yx);
        A.eps[eps_idx(e, 3, p)] = (realw)0.5 * (du.zx + du.xz);
        A.eps[eps_idx(e, 4, p)] = (realw)0.5 * (du.zy + du.yz);
      }
    }
    const Sigma6 sg = iso_stress(du, km[k].x, km[k].y);
    realw s[9];
    stress_products<FOLD>(sg, irr != 0, J, jacl, A.xix_regular, s);
#pragma unroll
    for (int a = 0; a < 3; a++) {
      if (lane) {
        sA[a][b] = s[a];
        sB[a][b] = s[3 + a];
      }
      d3[k][a] = s[6 + a];
    }
  }
  lds_barrier();
#pragma unroll
  for (int a = 0; a < 3; a++) {
    realw r[5], y[5], o[5];
#pragma unroll
    for (int l = 0; l < 5; l++) {
      r[l] = sA[a][bx + l];
      y[l] = sB[a][by + 5 * l];
    }
    line_divergence(G, r, o);
    if (lane) {
#pragma unroll
      for (int l = 0; l < 5; l++) sA[a][bx + l] = o[l];
    }
    line_divergence(G, y, o);
    if (lane) {
#pragma unroll
      for (int l = 0; l < 5; l++) sB[a][by + 5 * l] = o[l];
    }
#pragma unroll
    for (int k = 0; k < 5; k++) r[k] = d3[k][a];
    line_divergence(G, r, o);
#pragma unroll
    for (int k = 0; k < 5; k++) d3[k][a] = o[k];
  }
  lds_barrier();
  if (!active) return;
  const realw w3 = sW[i * 5 + j];
  const int slot = gather_slot(pos0 + ie, j, i, A.eb);  // of k = 0
#pragma unroll
  for (int k = 0; k < 5; k++) {
    const int b = el * 125 + c + 25 * k;
    const realw w1 = sW[j * 5 + k], w2 = sW[i * 5 + k];
    realw* o = A.local_out + 3 * (int64_t)(slot + k * 25 * A.eb);
#pragma unroll
    for (int a = 0; a < 3; a++) o[a] = sum3(w1, sA[a][b], w2, sB[a][b], w3, d3[k][a]);
  }
}

// R: tables of the regular elements, the first nreg; G: of the others
template <bool STRAIN, int KIND>
__global__ void __launch_bounds__(128) k_elastic_line(ElasticArgs A, GLLk R, GLLk G) {
  __shared__ realw sA[3][LINE_PL], sB[3][LINE_PL];
  __shared__ realw sW[25];
  const int nb = KIND == LINE_REG ? (int)gridDim.x : KIND == LINE_IRR ? 0 : (A.nreg + 4) / 5, b = (int)blockIdx.x;
  if (KIND != LINE_IRR && b < nb) elastic_line<STRAIN, true>(A, R, A.nreg, A.elems, 0, b, nb, sA, sB, sW);
  if (KIND != LINE_REG && b >= nb)
    elastic_line<STRAIN, false>(A, G, A.nelem - A.nreg, A.elems + A.nreg, A.nreg, b - nb, (int)gridDim.x - nb, sA, sB, sW);
}

// Elastic kernels of a run that recomputes the reconstructed field's strain from its displacement
// (A.displ; compute_kernels.f90:151-186 with the strain of compute_element_strain.F90:28-130): the
// gradient of k_elastic_line, then per point the sums of k_compute_kernels_el.
// Bound by HBM: 78 B per local point (index, acceleration, displacement and strain of the adjoint
// field, three sums read and written). The strain stored by one launch and read back by another
// took 16.5 + 30 us on 24^3 elements, and 2 us more in every stiffness launch that stored it;
// this launch takes 26.
// The operations are those of k_element_strain (the regular mapping is not folded into the tables) and
// of k_compute_kernels_el (products and sums rounded one by one, in FMA builds too: `rounded` keeps a
// product out of the sum that takes it).
__device__ __forceinline__ realw rounded(realw x) {
  asm("" : "+v"(x));
  return x;
}
__device__ __forceinline__ void kernel_sums(const KernelSums& S, int64_t q, int e, int p, realw dot, realw b1, realw b2,
                                            realw b3, realw b4, realw b5, realw btr3) {
  const realw e1 = S.eps[eps_idx(e, 0, p)], e2 = S.eps[eps_idx(e, 1, p)], e3 = S.eps[eps_idx(e, 2, p)],
              e4 = S.eps[eps_idx(e, 3, p)], e5 = S.eps[eps_idx(e, 4, p)];
  const realw shear = rounded(e3 * b3) + rounded(e4 * b4) + rounded(e5 * b5);
  S.rho_kl[q] = S.rho_kl[q] + rounded(S.deltat * dot);
  S.mu_kl[q] = S.mu_kl[q] + rounded(S.deltat * (rounded(e1 * b1) + rounded(e2 * b2) + rounded((e1 + e2) * (b1 + b2)) +
                                                (realw)2 * shear));
  S.kappa_kl[q] = S.kappa_kl[q] + rounded(S.deltat * ((realw)9 * S.eps_tr3[q] * btr3));
}

template <bool REG>
__global__ void __launch_bounds__(128) k_kernels_line(ElasticArgs A, KernelSums S, GLLk G) {
  constexpr int PL = 626;
  __shared__ realw sA[3][PL], sB[3][PL];
  const int t = threadIdx.x;
  const bool lane = t < 125;
  const int el = lane ? t / 25 : 4, c = lane ? t - 25 * el : t - 125;
  const int i = c % 5, j = c / 5;
  const int ie = xcd_remap(blockIdx.x, gridDim.x) * 5 + el;
  const bool active = lane && ie < A.nelem;
  const int e = A.elems[ie < A.nelem ? ie : A.nelem - 1];
  const int64_t ep = (int64_t)e * 125 + c;
  const int irr = REG ? 0 : A.irregular[e];
  const int64_t jp = REG ? 0 : (int64_t)(irr ? irr - 1 : 0) * 125 + c;
  realw d3[5][3], dot[5];
  {
    realw u[3][5];
    int g[5];
#pragma unroll
    for (int k = 0; k < 5; k++) g[k] = A.ibool[ep + 25 * k];
#pragma unroll
    for (int k = 0; k < 5; k++) {
      const realw* d = A.displ + 3 * (int64_t)g[k];
      const realw* a = S.accel + 3 * (int64_t)g[k];
      u[0][k] = d[0]; u[1][k] = d[1]; u[2][k] = d[2];
      dot[k] = rounded(a[0] * u[0][k]) + rounded(a[1] * u[1][k]) + rounded(a[2] * u[2][k]);
    }
    const int b = el * 125 + c;
#pragma unroll
    for (int a = 0; a < 3; a++) {
      if (lane) {
#pragma unroll
        for (int k = 0; k < 5; k++) sA[a][b + 25 * k] = u[a][k];
      }
      realw r[5];
      line_gradient(G, u[a], r);
#pragma unroll
      for (int k = 0; k < 5; k++) d3[k][a] = r[k];
    }
  }
  lds_barrier();
  const int bx = el * 125 + 5 * c, by = el * 125 + i + 25 * j;
  realw x[3][5];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    realw r[5], y[5];
#pragma unroll
    for (int l = 0; l < 5; l++) {
      r[l] = sA[a][bx + l];
      y[l] = sA[a][by + 5 * l];
    }
    line_gradient(G, r, x[a]);
    line_gradient(G, y, r);
    if (lane) {
#pragma unroll
      for (int l = 0; l < 5; l++) sB[a][by + 5 * l] = r[l];
    }
  }
  lds_barrier();                                   // every row of u has been read
  if (lane) {
#pragma unroll
    for (int a = 0; a < 3; a++)
#pragma unroll
      for (int l = 0; l < 5; l++) sA[a][bx + l] = x[a][l];
  }
  lds_barrier();
  if (!active) return;
  const realw ONE_THIRD = (realw)1 / (realw)3;
#pragma unroll
  for (int k = 0; k < 5; k++) {
    const int b = el * 125 + c + 25 * k, p = c + 25 * k;
    const int64_t q = ep + 25 * k;
    const Grad9 tg = {sA[0][b], sA[1][b], sA[2][b], sB[0][b], sB[1][b], sB[2][b], d3[k][0], d3[k][1], d3[k][2]};
    JacPt J = {};
    if (!REG && irr) J = load_jac(A.jac, A.jac_plane, jp + 25 * k);
    Du9 du = map_gradient<false>(tg, irr != 0, J, A.xix_regular);
    if (REG) {
      for (realw* d : {&du.xx, &du.xy, &du.xz, &du.yx, &du.yy, &du.yz, &du.zx, &du.zy, &du.zz}) *d = rounded(*d);
    }
    const realw templ = ONE_THIRD * (du.xx + du.yy + du.zz);
    kernel_sums(S, q, e, p, dot[k], du.xx - templ, du.yy - templ, (realw)0.5 * (du.xy + du.yx),
                (realw)0.5 * (du.zx + du.xz), (realw)0.5 * (du.zy + du.yz), templ);
  }
}

// element strain of a displacement field (compute_element_strain.F90:28-130); one lane per point
__global__ void __launch_bounds__(128) k_element_strain(ElasticArgs A, GLLk G, realw* eps, realw* eps_tr3,
                                                        int with_trace) {
  __shared__ realw s_buf[5][3][128];
  const int tid = threadIdx.x;
  const int el = tid / 25;
  const int c = tid - el * 25;
  const int i = c % 5, j = c / 5;
  const int ie = blockIdx.x * 5 + el;
  const bool active = (tid < 125) && (ie < A.nelem);
  const int e = active ? A.elems[ie] : 0;
  realw ux[5], uy[5], uz[5];
  if (active) {
#pragma unroll
    for (int k = 0; k < 5; k++) {
      const int g = A.ibool[(int64_t)e * 125 + c + 25 * k];
      ux[k] = A.displ[3 * (int64_t)g]; uy[k] = A.displ[3 * (int64_t)g + 1]; uz[k] = A.displ[3 * (int64_t)g + 2];
      s_buf[el][0][c + 25 * k] = ux[k]; s_buf[el][1][c + 25 * k] = uy[k]; s_buf[el][2][c + 25 * k] = uz[k];
    }
  }
  __syncthreads();
  if (!active) return;
  const int irr = A.irregular[e];
  const realw ONE_THIRD = (realw)1 / (realw)3;
#pragma unroll
  for (int k = 0; k < 5; k++) {
    const int p = c + 25 * k;
    const int b1 = 5 * j + 25 * k, b2 = i + 25 * k;
    const realw* sx = s_buf[el][0];
    const realw* sy = s_buf[el][1];
    const realw* sz = s_buf[el][2];
    realw tx1 = G.hp[i * 5] * sx[b1], ty1 = G.hp[i * 5] * sy[b1], tz1 = G.hp[i * 5] * sz[b1];
    realw tx2 = G.hp[j * 5] * sx[b2], ty2 = G.hp[j * 5] * sy[b2], tz2 = G.hp[j * 5] * sz[b2];
    realw tx3 = G.hp[k * 5] * ux[0], ty3 = G.hp[k * 5] * uy[0], tz3 = G.hp[k * 5] * uz[0];
#pragma unroll
    for (int l = 1; l < 5; l++) {
      tx1 = tx1 + G.hp[i * 5 + l] * sx[b1 + l]; ty1 = ty1 + G.hp[i * 5 + l] * sy[b1 + l];
      tz1 = tz1 + G.hp[i * 5 + l] * sz[b1 + l];
      tx2 = tx2 + G.hp[j * 5 + l] * sx[b2 + 5 * l]; ty2 = ty2 + G.hp[j * 5 + l] * sy[b2 + 5 * l];
      tz2 = tz2 + G.hp[j * 5 + l] * sz[b2 + 5 * l];
      tx3 = tx3 + G.hp[k * 5 + l] * ux[l]; ty3 = ty3 + G.hp[k * 5 + l] * uy[l]; tz3 = tz3 + G.hp[k * 5 + l] * uz[l];
    }
    realw duxdx, duxdy, duxdz, duydx, duydy, duydz, duzdx, duzdy, duzdz;
    if (irr) {
      const int64_t q = (int64_t)(irr - 1) * 125 + p;
      const int64_t P = A.jac_plane;
      const realw* J = A.jac;
      const realw xixl = J[q], xiyl = J[P + q], xizl = J[2 * P + q], etaxl = J[3 * P + q], etayl = J[4 * P + q];
      const realw etazl = J[5 * P + q], gaxl = J[6 * P + q], gayl = J[7 * P + q], gazl = J[8 * P + q];
      duxdx = xixl * tx1 + etaxl * tx2 + gaxl * tx3;
      duxdy = xiyl * tx1 + etayl * tx2 + gayl * tx3;
      duxdz = xizl * tx1 + etazl * tx2 + gazl * tx3;
      duydx = xixl * ty1 + etaxl * ty2 + gaxl * ty3;
      duydy = xiyl * ty1 + etayl * ty2 + gayl * ty3;
      duydz = xizl * ty1 + etazl * ty2 + gazl * ty3;
      duzdx = xixl * tz1 + etaxl * tz2 + gaxl * tz3;
      duzdy = xiyl * tz1 + etayl * tz2 + gayl * tz3;
      duzdz = xizl * tz1 + etazl * tz2 + gazl * tz3;
    } else {
      const realw xr = A.xix_regular;
      duxdx = xr * tx1; duxdy = xr * tx2; duxdz = xr * tx3;
      duydx = xr * ty1; duydy = xr * ty2; duydz = xr * ty3;
      duzdx = xr * tz1; duzdy = xr * tz2; duzdz = xr * tz3;
    }
    const realw templ = ONE_THIRD * (duxdx + duydy + duzdz);
    const int64_t ep = (int64_t)e * 125 + p;
    eps_tr3[ep] = templ;
    eps[eps_idx(e, 0, p)] = duxdx - templ;
    eps[eps_idx(e, 1, p)] = duydy - templ;
    eps[eps_idx(e, 2, p)] = (realw)0.5 * (duxdy + duydx);
    eps[eps_idx(e, 3, p)] = (realw)0.5 * (duzdx + duxdz);
    eps[eps_idx(e, 4, p)] = (realw)0.5 * (duzdy + duydz);
    // with attenuation the trace plane feeds the bulk memory variables (compute_strain_att,
    // compute_element_strain.F90:196: epsilondev_trace = 3 * epsilon_trace_over_3)
    if (with_trace) eps[eps_idx(e, 5, p)] = (realw)3 * templ;
  }
}

}  // namespace SF_VNS
using namespace SF_VNS;

void SFX(launch_elastic)(hipStream_t s, const ElasticArgs& a, bool strain, bool att, int att_variant) {
  if (a.nelem <= 0) return;
  GLLk G = g_gll_host;
  if (att && SF_FOLD) fold_gll(G, a.xix_regular, a.jacobian_regular);
  dim3 grid(a.nelem), block(128);
#define SF_K(V) hipLaunchKernelGGL((k_elastic_pt<V>), grid, block, 0, s, a, G)
  if (att) {
    if (att_variant == 1) SF_K(1);
    else if (att_variant == 2) SF_K(2);
    else if (att_variant == 3) SF_K(3);
    else if (att_variant == 4) SF_K(4);
    else SF_K(0);
  } else {
    GLLk R = G;
    if (SF_FOLD) regular_gll(R, a.xix_regular, a.jacobian_regular);
    const int nb = (a.nreg + 4) / 5 + (a.nelem - a.nreg + 4) / 5;
#define SF_L(S, K) hipLaunchKernelGGL((k_elastic_line<S, K>), dim3(nb), block, 0, s, a, R, G)
    if (a.nreg == a.nelem) {
      if (strain) SF_L(true, LINE_REG);
      else SF_L(false, LINE_REG);
    } else if (a.nreg == 0) {
      if (strain) SF_L(true, LINE_IRR);
      else SF_L(false, LINE_IRR);
    } else {
      if (strain) SF_L(true, LINE_BOTH);
      else SF_L(false, LINE_BOTH);
    }
#undef SF_L
  }
#undef SF_K
  SF_LAUNCH_CHECK("k_elastic_pt");
}

void SFX(launch_kernels_line)(hipStream_t s, const ElasticArgs& a, const KernelSums& k) {
  if (a.nelem <= 0) return;
  const dim3 grid((a.nelem + 4) / 5), block(128);
  if (a.jac_plane == 0) hipLaunchKernelGGL(k_kernels_line<true>, grid, block, 0, s, a, k, g_gll_host);
  else hipLaunchKernelGGL(k_kernels_line<false>, grid, block, 0, s, a, k, g_gll_host);
  SF_LAUNCH_CHECK("k_kernels_line");
}

void SFX(launch_element_strain)(hipStream_t s, const ElasticArgs& a, realw* eps, realw* eps_tr3, bool with_trace) {
  if (a.nelem <= 0) return;
  dim3 grid((a.nelem + 4) / 5), block(128);
  hipLaunchKernelGGL(k_element_strain, grid, block, 0, s, a, g_gll_host, eps, eps_tr3, with_trace ? 1 : 0);
  SF_LAUNCH_CHECK("k_element_strain");
}

}  // namespace sf
