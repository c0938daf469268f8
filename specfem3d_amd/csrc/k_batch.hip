// k_batch.hip -- element stiffness of the batched many-shot engine (elastic, isotropic).
//
// Many independent shots share one mesh. Their wavefields are kept in groups of eight shots
// (batch_idx): a point's three rows of a group are 96 contiguous bytes, and a run of points is a run
// of full cache lines that no other group touches, so a finished group costs nothing and leaves no
// holes in the rows of the others. A workgroup takes one element and SC
// shots (SC = 4 or 8): the element's ibool, moduli and Jacobian terms are loaded once for them, and
// the workgroups of one element's shots are adjacent in the grid, so they share those. The per-point
// arithmetic is elastic_point.h, the same code as the single-shot kernel, so a batched shot has the bits of
// its single-shot run in the same order of sums (FMA builds: without attenuation and under assembly 2, see
// batch.hip).
//
// Shots are stored in decreasing order of record length; a shot is live at step `it` while
// nstep[s] >= it, and a group whose first shot has finished exits at once (uneven record
// lengths cost nothing after a shot ends). `it` is read from device memory so a captured graph
// of the step can be replayed.
//
// The stiffness stores the local forces, and the update that starts the next step sums them per point
// (k_batch_gather in batch.hip), in the colour order of a single-shot run under assembly = 2.
//
// Compiled twice like k_elastic.hip: SF_EXACT=1 without FMA contraction, SF_EXACT=0 with it.
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

__device__ __forceinline__ realw c4(const float4& x, int r) { return r == 0 ? x.x : r == 1 ? x.y : r == 2 ? x.z : x.w; }

__device__ __forceinline__ int xcd_remap_b(int b, int nb) {
  const int q = nb >> 3, r = nb & 7, x = b & 7;
  return x * q + (x < r ? x : r) + (b >> 3);
}

// One element and SC = 4 or 8 shots per workgroup of 32 SC lanes, in two lane roles:
//   * global memory: lane = three units of 4 consecutive shots of one point and component, unit n =
//     (point, component, quad) with the quad fastest: with SC = 8 the units of a row of five points are
//     480 contiguous bytes, and the element's local forces one run of 12 KB;
//   * contractions: lane = (line of five points, shot), shot fastest, 25 SC lanes: the line scheme of
//     k_elastic_line (k_elastic.hip). The lane's gamma column stays in its registers, its xi and eta
//     rows go through LDS once each way, the coefficients sit in scalar registers.
// Both meet in LDS planes of the same order (point, component, shot). 61 VGPRs, 24 KB of LDS, six
// workgroups per CU. Two or three elements per workgroup fill the lanes better (25 SC of 32 SC work
// here) and are slower all the same (572 and 700 us against 523 for the whole step of 16 shots on
// 32x32x16 elements, same source otherwise): seven or ten waves wait for each other at each barrier.
// REG: the regular elements of a mesh (FMA build: the mapping is folded into the tables); workgroups take
// one kind each, as in k_elastic_line.
template <int SC, bool REG>
__device__ __forceinline__ void elastic_batch(const BatchArgs& B, const GLLk& G, const int* elems, int pos0, int block,
                                              int blocks, realw (&sA)[375 * SC], realw (&sB)[375 * SC], realw (&sW)[25]) {
  constexpr bool FOLD = REG && SF_FOLD;
  constexpr int NQ = SC / 4, NU = 375 * NQ, NT = 32 * SC, PS = 3 * SC;
  const int t = threadIdx.x;
  const int it = __hip_atomic_load(B.it, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int b = xcd_remap_b(block, blocks);
  const int ie = b / B.ngroups;
  const int s0 = B.s_first + (b - ie * B.ngroups) * SC;
  if (B.nstep[s0] < it) return;                   // every shot of this group has finished
  if (t < 25) sW[t] = G.wxy[t];
  const int e = elems[ie];
  const int irr = REG ? 0 : B.irregular[e];
  // memory role: units t, t + NT, t + 2 NT of 375 NQ
  const int q4 = t % NQ, sq = s0 + 4 * q4;        // NT is a multiple of NQ: one quad for all three
  const bool live0 = B.nstep[sq] >= it;           // shots sorted: later ones finish first
  int64_t row[3];
  bool mine[3];
#pragma unroll
  for (int m = 0; m < 3; m++) {
    const int n = t + m * NT, p = n < NU ? n / (3 * NQ) : 124;
    mine[m] = n < NU && live0;
    row[m] = batch_idx(B.nrow, 3 * (int64_t)B.ibool[(int64_t)e * 125 + p] + n / NQ % 3, sq);
  }
  // line role: column / rows of c, shot s (25 SC of the lanes; the rest shadow the first ones)
  const bool lane = t < 25 * SC;
  const int tt = lane ? t : t - 25 * SC;
  const int s = tt % SC, c = tt / SC;
  const int i = c % 5, j = c / 5;
  const int64_t ep = (int64_t)e * 125 + c;
  float2 km[5];
  {
    float4 u[3];
#pragma unroll
    for (int m = 0; m < 3; m++) {
      u[m] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (mine[m]) u[m] = *reinterpret_cast<const float4*>(B.u + row[m]);
    }
#pragma unroll
    for (int k = 0; k < 5; k++) km[k] = B.kappamu[ep + 25 * k];
#pragma unroll
    for (int m = 0; m < 3; m++)
      if (t + m * NT < NU) *reinterpret_cast<float4*>(&sA[4 * (t + m * NT)]) = u[m];
  }
  lds_barrier();
  const int bp = c * PS + s;                      // point k of the column at bp + 25 PS k
  const int bx = 5 * c * PS + s, by = (i + 25 * j) * PS + s;
  realw d3[5][3];
  {
    realw x[3][5];
#pragma unroll
    for (int a = 0; a < 3; a++) {
      realw r[5], y[5], z[5];
#pragma unroll
      for (int l = 0; l < 5; l++) {
        r[l] = sA[bx + PS * l + SC * a];
        y[l] = sA[by + 5 * PS * l + SC * a];
        z[l] = sA[bp + 25 * PS * l + SC * a];
      }
      line_gradient(G, r, x[a]);
      line_gradient(G, y, r);
      if (lane) {
#pragma unroll
        for (int l = 0; l < 5; l++) sB[by + 5 * PS * l + SC * a] = r[l];
      }
      line_gradient(G, z, r);
#pragma unroll
      for (int k = 0; k < 5; k++) d3[k][a] = r[k];
    }
    lds_barrier();                                // every row of u has been read
    if (lane) {
#pragma unroll
      for (int a = 0; a < 3; a++)
#pragma unroll
        for (int l = 0; l < 5; l++) sA[bx + PS * l + SC * a] = x[a][l];
    }
  }
  lds_barrier();
#pragma unroll
  for (int k = 0; k < 5; k++) {
    const int q = bp + 25 * PS * k;
    const Grad9 tg = {sA[q], sA[q + SC], sA[q + 2 * SC], sB[q], sB[q + SC], sB[q + 2 * SC], d3[k][0], d3[k][1], d3[k][2]};
    JacPt J = {};
    realw jacl = B.jacobian_regular;
    if (!REG && irr) {
      J = load_jac(B.jac, B.jac_plane, (int64_t)(irr - 1) * 125 + c + 25 * k);
      jacl = J.jac;
    }
    const Du9 du = map_gradient<FOLD>(tg, irr != 0, J, B.xix_regular);
    const Sigma6 sg = iso_stress(du, km[k].x, km[k].y);
    realw pr[9];
    stress_products<FOLD>(sg, irr != 0, J, jacl, B.xix_regular, pr);
#pragma unroll
    for (int a = 0; a < 3; a++) {
      if (lane) {
        sA[q + SC * a] = pr[a];
        sB[q + SC * a] = pr[3 + a];
      }
      d3[k][a] = pr[6 + a];
    }
  }
  lds_barrier();
#pragma unroll
  for (int a = 0; a < 3; a++) {
    realw r[5], y[5], o[5];
#pragma unroll
    for (int l = 0; l < 5; l++) {
      r[l] = sA[bx + PS * l + SC * a];
      y[l] = sB[by + 5 * PS * l + SC * a];
    }
    line_divergence(G, r, o);
    if (lane) {
#pragma unroll
      for (int l = 0; l < 5; l++) sA[bx + PS * l + SC * a] = o[l];
    }
    line_divergence(G, y, o);
    if (lane) {
#pragma unroll
      for (int l = 0; l < 5; l++) sB[by + 5 * PS * l + SC * a] = o[l];
    }
#pragma unroll
    for (int k = 0; k < 5; k++) r[k] = d3[k][a];
    line_divergence(G, r, o);
#pragma unroll
    for (int k = 0; k < 5; k++) d3[k][a] = o[k];
  }
  lds_barrier();
  if (lane) {
    const realw w3 = sW[i * 5 + j];
#pragma unroll
    for (int k = 0; k < 5; k++) {
      const int q = bp + 25 * PS * k;
      const realw w1 = sW[j * 5 + k], w2 = sW[i * 5 + k];
#pragma unroll
      for (int a = 0; a < 3; a++) sA[q + SC * a] = sum3(w1, sA[q + SC * a], w2, sB[q + SC * a], w3, d3[k][a]);
    }
  }
  lds_barrier();
  // finished shots of a live quad store what their last displacement gives; nothing reads it
  realw* o = B.local + (int64_t)(sq >> 3) * B.loc_group + (int64_t)(pos0 + ie) * 3000 + (sq & 7);
#pragma unroll
  for (int m = 0; m < 3; m++) {
    const int n = t + m * NT;
    if (mine[m]) *reinterpret_cast<float4*>(o + 8 * (n / NQ)) = *reinterpret_cast<const float4*>(&sA[4 * n]);
  }
}

// R: tables of the regular elements, the first nreg; G: of the others
template <int SC, int KIND>
__global__ void __launch_bounds__(32 * SC) k_elastic_batch(BatchArgs B, GLLk R, GLLk G) {
  __shared__ __attribute__((aligned(16))) realw sA[375 * SC], sB[375 * SC];  // (p, a, s) at (3 p + a) SC + s
  __shared__ realw sW[25];
  const int nb = KIND == LINE_REG ? (int)gridDim.x : KIND == LINE_IRR ? 0 : B.nreg * B.ngroups, b = (int)blockIdx.x;
  if (KIND != LINE_IRR && b < nb) elastic_batch<SC, true>(B, R, B.elems, 0, b, nb, sA, sB, sW);
  if (KIND != LINE_REG && b >= nb)
    elastic_batch<SC, false>(B, G, B.elems + B.nreg, B.nreg, b - nb, (int)gridDim.x - nb, sA, sB, sW);
}

// Viscoelastic (3-SLS) variant: each shot also carries its memory variables and stored strain
// (one block per element and shot: plane, point). The tile holds u and dt*v (6 rows per shot; they share the
// LDS of the stress products t2, t3, written after a barrier). Per shot, the arithmetic and its
// order are the single-shot point kernel's (k_elastic_pt): strain at u + dt v, isotropic stress
// minus the memory-variable sums, memory update, stress products.
// Per-shot state is one block per (element, shot), point-fastest within each plane: the lanes of a
// wave that read one shot read consecutive words (a shot-fastest row would spread a wave's reads
// of one shot over S times as many cache lines), and the planes of a block sit at fixed offsets
// from one base address.
__device__ __forceinline__ int64_t rb_idx(int64_t e, int plane, int p, int64_t S, int s) {
  return ((e * S + s) * 18 + plane) * 125 + p;
}
__device__ __forceinline__ int64_t eb_idx(int64_t e, int c, int p, int64_t S, int s) {
  return ((e * S + s) * 6 + c) * 125 + p;
}

template <int NQ>
__global__ void __launch_bounds__(128 * NQ) k_visco_batch(BatchArgs B, GLLk G) {
  constexpr int SC = 4 * NQ;
  // LDS rows (component or product, shot) of PST floats, point fastest: the rows of a lane's two quads
  // start 16 banks apart, so 16 consecutive points of two quads read 32 different banks
  constexpr int PST = 132;
  constexpr int CPL = SC * PST;
  __shared__ realw sBuf[9 * CPL];
  realw* const sT = sBuf;                         // stress products [m][s][p]
  realw* const sU = sBuf + 3 * CPL;               // u (rows 0..2) and dt*v (rows 3..5), [c][s][p]
  __shared__ realw sG[SF_NGLL_TABLE];
  stage_gll(sG, G, threadIdx.x);
  const int it = __hip_atomic_load(B.it, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int b = xcd_remap_b(blockIdx.x, gridDim.x);
  const int ie = b / B.ngroups;
  const int s0 = B.s_first + (b - ie * B.ngroups) * SC;
  if (B.nstep[s0] < it) return;
  const int q = threadIdx.x % NQ, p = threadIdx.x / NQ;
  const int sq = s0 + 4 * q;
  const bool live0 = B.nstep[sq] >= it;
  bool live[4];
#pragma unroll
  for (int r = 0; r < 4; r++) live[r] = B.nstep[sq + r] >= it;
  const bool active = p < 125;
  const int pp = active ? p : 124;
  const int e = B.elems[ie];
  const int irr = B.irregular[e];
  const int64_t S = B.S;
  const int64_t ep = (int64_t)e * 125 + pp;
  const int g = B.ibool[ep];
  const int64_t row = batch_idx(B.nrow, 3 * (int64_t)g, sq);
  const int ts = 4 * q;
  float4 u[3], V[3];                              // staged into the tile below
#pragma unroll
  for (int c = 0; c < 3; c++) {
    u[c] = make_float4(0.f, 0.f, 0.f, 0.f);
    V[c] = u[c];
    if (live0) {
      u[c] = *reinterpret_cast<const float4*>(B.u + row + c * 8);
      V[c] = *reinterpret_cast<const float4*>(B.v + row + c * 8);
    }
  }
  const bool mine = active && live0;
  JacPt J = {};
  realw jacl = B.jacobian_regular;
  if (irr) {
    J = load_jac(B.jac, B.jac_plane, (int64_t)(irr - 1) * 125 + pp);
    jacl = J.jac;
  }
  const float2 km = B.kappamu[ep];
  realw fcv[3], fckv[3];
  if (B.fc_index) {
    const int rrow = B.fc_index[ep];
#pragma unroll
    for (int s = 0; s < 3; s++) {
      fcv[s] = B.fc_table[s * B.fc_rows + rrow];
      fckv[s] = B.fc_table[(3 + s) * B.fc_rows + rrow];
    }
  } else {
#pragma unroll
    for (int s = 0; s < 3; s++) {
      fcv[s] = B.fc[s * B.nloc + ep];
      fckv[s] = B.fck[s * B.nloc + ep];
    }
  }
  if (active) {
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int c = 0; c < 3; c++) {
        sU[(c * SC + ts + r) * PST + p] = c4(u[c], r);
        sU[((3 + c) * SC + ts + r) * PST + p] = B.dt * c4(V[c], r);
      }
  }
  // memory variables and stored strain of the first shot, in flight with the tile gather; each
  // later shot's are loaded while the previous shot is computed (two register sets)
  realw Rc[18], Ec[6];
#pragma unroll
  for (int pl = 0; pl < 18; pl++) Rc[pl] = B.R[rb_idx(e, pl, pp, S, sq)];
#pragma unroll
  for (int cc = 0; cc < 6; cc++) Ec[cc] = B.eps[eb_idx(e, cc, pp, S, sq)];
  lds_barrier();

  const int k = pp / 25, j = (pp / 5) % 5, i = pp % 5;
  const realw ONE_THIRD = (realw)1 / (realw)3;
  const realw kappal = km.x, mul = km.y;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int s = sq + r;
    realw Rn[18], En[6];
    if (r < 3) {
#pragma unroll
      for (int pl = 0; pl < 18; pl++) Rn[pl] = B.R[rb_idx(e, pl, pp, S, s + 1)];
#pragma unroll
      for (int cc = 0; cc < 6; cc++) En[cc] = B.eps[eb_idx(e, cc, pp, S, s + 1)];
    }
    __builtin_amdgcn_sched_barrier(0);            // the next shot's loads are issued first
    const realw* su = sU + (ts + r) * PST;
    const Grad9 tg = tile_gradient<1>(su, su + CPL, su + 2 * CPL, gll_hp(sG, irr != 0), i, j, k);
    const Du9 du = map_gradient(tg, irr != 0, J, B.xix_regular);
    const Du9 st = map_gradient(tile_gradient_continue<1>(tg, su + 3 * CPL, su + 4 * CPL, su + 5 * CPL, gll_hp(sG, irr != 0), i, j, k),
                                irr != 0, J, B.xix_regular);
    const realw e_tr = (st.xx + st.yy + st.zz);
    const realw templ = ONE_THIRD * (st.xx + st.yy + st.zz);
    const realw Snp1[6] = {st.xx - templ, st.yy - templ, (realw)0.5 * (st.xy + st.yx), (realw)0.5 * (st.zx + st.xz),
                           (realw)0.5 * (st.zy + st.yz), e_tr};
    Sigma6 sg = iso_stress(du, kappal, mul);
    realw Rv[6][3], Sn[6];
#pragma unroll
    for (int cc = 0; cc < 6; cc++) {
#pragma unroll
      for (int sl = 0; sl < 3; sl++) Rv[cc][sl] = Rc[cc * 3 + sl];
      Sn[cc] = Ec[cc];
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
    if (mine && live[r]) {
#pragma unroll
      for (int sl = 0; sl < 3; sl++) {
        const realw flk = kappal * fckv[sl];
        B.R[rb_idx(e, 5 * 3 + sl, pp, S, s)] =
            B.alpha[sl] * Rv[5][sl] + flk * (B.beta[sl] * Sn[5] + B.gamma[sl] * Snp1[5]);
        const realw flm = mul * fcv[sl];
#pragma unroll
        for (int cc = 0; cc < 5; cc++)
          B.R[rb_idx(e, cc * 3 + sl, pp, S, s)] =
              B.alpha[sl] * Rv[cc][sl] + flm * (B.beta[sl] * Sn[cc] + B.gamma[sl] * Snp1[cc]);
      }
#pragma unroll
      for (int cc = 0; cc < 6; cc++) B.eps[eb_idx(e, cc, pp, S, s)] = Snp1[cc];
    }
    realw t[9];
    stress_products<SF_FOLD, true>(sg, irr != 0, J, jacl, B.xix_regular, t);
    if (active) {
#pragma unroll
      for (int m = 0; m < 3; m++) sT[(m * SC + ts + r) * PST + p] = t[m];
    }
    // products t2, t3 overlay this shot's u / dt*v rows: written once every lane is past them
    lds_barrier();
    if (active) {
#pragma unroll
      for (int m = 3; m < 9; m++) sT[(m * SC + ts + r) * PST + p] = t[m];
    }
    if (r < 3) {
#pragma unroll
      for (int pl = 0; pl < 18; pl++) Rc[pl] = Rn[pl];
#pragma unroll
      for (int cc = 0; cc < 6; cc++) Ec[cc] = En[cc];
    }
    __builtin_amdgcn_sched_barrier(0);            // at most two shots' state in registers
  }
  lds_barrier();
  if (!mine) return;

  const realw* hpw = gll_hpw(sG, irr != 0);
  const realw* wxy = sG + 50;
  realw* o = B.local + (int64_t)(sq >> 3) * B.loc_group + ((int64_t)ie * 125 + p) * 24 + (sq & 7);
#pragma unroll
  for (int c = 0; c < 3; c++) {
    float4 f;
    f.x = tile_divergence_c<1>(sT + ts * PST, CPL, hpw, wxy, i, j, k, c);
    f.y = tile_divergence_c<1>(sT + (ts + 1) * PST, CPL, hpw, wxy, i, j, k, c);
    f.z = tile_divergence_c<1>(sT + (ts + 2) * PST, CPL, hpw, wxy, i, j, k, c);
    f.w = tile_divergence_c<1>(sT + (ts + 3) * PST, CPL, hpw, wxy, i, j, k, c);
    *reinterpret_cast<float4*>(o + 8 * c) = f;
  }
}

// Batched acoustic stiffness (compute_forces_acoustic.F90:35-726; the arithmetic of k_acoustic per
// point and shot): chi'' -= div((1/rho) grad chi) for SC = 4 NQ shots of one element per
// workgroup. Lane = (GLL point p, quad of 4 consecutive shots) as in k_visco_batch; the
// potential tile and the three products (rho^-1 jacobian grad chi . grad xi, eta, gamma) go through
// LDS, one row of PST floats per (plane, shot). Every sum runs in k_acoustic's order (the gamma
// contraction reads the same values the column kernel holds in registers), so a batched shot
// reproduces the single-shot run with the same order of sums.
template <int NQ>
__global__ void __launch_bounds__(128 * NQ) k_acoustic_batch(BatchAcArgs B, GLLk G) {
  constexpr int SC = 4 * NQ;
  constexpr int PST = 132;
  constexpr int CPL = SC * PST;
  __shared__ realw sBuf[4 * CPL];                 // [0] potential tile, [1..3] products t1, t2, t3
  __shared__ realw sG[SF_NGLL_TABLE];
  stage_gll(sG, G, threadIdx.x);
  const int it = __hip_atomic_load(B.it, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int b = xcd_remap_b(blockIdx.x, gridDim.x);
  const int ie = b / B.ngroups;
  const int s0 = B.s_first + (b - ie * B.ngroups) * SC;
  if (B.nstep[s0] < it) return;
  const int q = threadIdx.x % NQ, p = threadIdx.x / NQ;
  const int sq = s0 + 4 * q;
  const bool live0 = B.nstep[sq] >= it;
  const bool active = p < 125;
  const int pp = active ? p : 124;
  const int e = B.elems[ie];
  const int irr = B.irregular[e];
  const int g = B.ibool[(int64_t)e * 125 + pp];
  const int64_t row = batch_idx(B.nrow, (int64_t)g - B.g0, sq);
  const int ts = 4 * q;
  float4 c0 = make_float4(0.f, 0.f, 0.f, 0.f);
  if (live0) c0 = *reinterpret_cast<const float4*>(B.pot + row);
  const realw rho_invl = (realw)1 / B.rho[(int64_t)e * 125 + pp];
  JacPt J = {};
  if (irr) J = load_jac(B.jac, B.jac_plane, (int64_t)(irr - 1) * 125 + pp);
  if (active) {
#pragma unroll
    for (int r = 0; r < 4; r++) sBuf[(ts + r) * PST + p] = c4(c0, r);
  }
  lds_barrier();
  const int k = pp / 25, j = (pp / 5) % 5, i = pp % 5;
  const int b1 = 5 * j + 25 * k, b2 = i + 25 * k, b3 = i + 5 * j;
  const realw* hp = sG;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const realw* s = sBuf + (ts + r) * PST;
    realw a1 = sum2(hp[i * 5], s[b1], hp[i * 5 + 1], s[b1 + 1]);
    realw a2 = sum2(hp[j * 5], s[b2], hp[j * 5 + 1], s[b2 + 5]);
    realw a3 = sum2(hp[k * 5], s[b3], hp[k * 5 + 1], s[b3 + 25]);
#pragma unroll
    for (int l = 2; l < 5; l++) {
      a1 = add_product(a1, hp[i * 5 + l], s[b1 + l]);
      a2 = add_product(a2, hp[j * 5 + l], s[b2 + 5 * l]);
      a3 = add_product(a3, hp[k * 5 + l], s[b3 + 25 * l]);
    }
    realw t1, t2, t3;
    if (irr) {
      const realw dpdx = sum3(J.xix, a1, J.etax, a2, J.gax, a3);
      const realw dpdy = sum3(J.xiy, a1, J.etay, a2, J.gay, a3);
      const realw dpdz = sum3(J.xiz, a1, J.etaz, a2, J.gaz, a3);
      t1 = rho_invl * J.jac * sum3(J.xix, dpdx, J.xiy, dpdy, J.xiz, dpdz);
      t2 = rho_invl * J.jac * sum3(J.etax, dpdx, J.etay, dpdy, J.etaz, dpdz);
      t3 = rho_invl * J.jac * sum3(J.gax, dpdx, J.gay, dpdy, J.gaz, dpdz);
    } else {
      const realw jl = B.jacobian_regular, xr = B.xix_regular;
      t1 = rho_invl * jl * xr * xr * a1;
      t2 = rho_invl * jl * xr * xr * a2;
      t3 = rho_invl * jl * xr * xr * a3;
    }
    if (active) {
      sBuf[(1 * SC + ts + r) * PST + p] = t1;
      sBuf[(2 * SC + ts + r) * PST + p] = t2;
      sBuf[(3 * SC + ts + r) * PST + p] = t3;
    }
  }
  lds_barrier();
  if (!active || !live0) return;
  const realw* hpw = sG + 25;
  const realw* wxy = sG + 50;
  float f[4];
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const realw* s1 = sBuf + (1 * SC + ts + r) * PST;
    const realw* s2 = sBuf + (2 * SC + ts + r) * PST;
    const realw* s3 = sBuf + (3 * SC + ts + r) * PST;
    realw n1 = sum2(hpw[i], s1[b1], hpw[5 + i], s1[b1 + 1]);
    realw n2 = sum2(hpw[j], s2[b2], hpw[5 + j], s2[b2 + 5]);
    realw n3 = sum2(hpw[k], s3[b3], hpw[5 + k], s3[b3 + 25]);
#pragma unroll
    for (int l = 2; l < 5; l++) {
      n1 = add_product(n1, hpw[l * 5 + i], s1[b1 + l]);
      n2 = add_product(n2, hpw[l * 5 + j], s2[b2 + 5 * l]);
      n3 = add_product(n3, hpw[l * 5 + k], s3[b3 + 25 * l]);
    }
    f[r] = sum3(wxy[j * 5 + k], n1, wxy[i * 5 + k], n2, wxy[i * 5 + j], n3);
  }
  realw* o = B.local + (int64_t)(sq >> 3) * B.loc_group + ((int64_t)ie * 125 + p) * 8 + (sq & 7);
  *reinterpret_cast<float4*>(o) = make_float4(f[0], f[1], f[2], f[3]);
}

}  // namespace SF_VNS
using namespace SF_VNS;

void SFX(launch_elastic_batch)(hipStream_t st, const BatchArgs& a, int sc) {
  if (a.nelem <= 0 || a.ngroups <= 0) return;
  if ((int64_t)a.nelem * a.ngroups > 0x7fffffff) fatal("launch_elastic_batch", "grid too large");
  if (sc != 4 && sc != 8) fatal("launch_elastic_batch", "shots per workgroup must be 4 or 8");
  GLLk G = g_gll_host, R = G;
  if (SF_FOLD) regular_gll(R, a.xix_regular, a.jacobian_regular);
  const unsigned nb = (unsigned)(a.nelem * a.ngroups);
#define SF_KB(SC, K) hipLaunchKernelGGL((k_elastic_batch<SC, K>), dim3(nb), dim3(32 * SC), 0, st, a, R, G)
  if (a.nreg == a.nelem) {
    if (sc == 4) SF_KB(4, LINE_REG);
    else SF_KB(8, LINE_REG);
  } else if (a.nreg == 0) {
    if (sc == 4) SF_KB(4, LINE_IRR);
    else SF_KB(8, LINE_IRR);
  } else {
    if (sc == 4) SF_KB(4, LINE_BOTH);
    else SF_KB(8, LINE_BOTH);
  }
#undef SF_KB
  SF_LAUNCH_CHECK("k_elastic_batch");
}

void SFX(launch_visco_batch)(hipStream_t st, const BatchArgs& a, int sc) {
  if (a.nelem <= 0 || a.ngroups <= 0) return;
  const int64_t nb = (int64_t)a.nelem * a.ngroups;
  if (nb > 0x7fffffff) fatal("launch_visco_batch", "grid too large");
  if (!a.R || !a.eps || !a.v) fatal("launch_visco_batch", "memory variables, strain and velocity are needed");
  const dim3 grid((unsigned)nb);
  GLLk G = g_gll_host;
  if (SF_FOLD) fold_gll(G, a.xix_regular, a.jacobian_regular);
  if (sc == 4) hipLaunchKernelGGL(k_visco_batch<1>, grid, dim3(128), 0, st, a, G);
  else if (sc == 8) hipLaunchKernelGGL(k_visco_batch<2>, grid, dim3(256), 0, st, a, G);
  else fatal("launch_visco_batch", "shots per workgroup must be 4 or 8");
  SF_LAUNCH_CHECK("k_visco_batch");
}

void SFX(launch_acoustic_batch)(hipStream_t st, const BatchAcArgs& a, int sc) {
  if (a.nelem <= 0 || a.ngroups <= 0) return;
  const int64_t nb = (int64_t)a.nelem * a.ngroups;
  if (nb > 0x7fffffff) fatal("launch_acoustic_batch", "grid too large");
  const dim3 grid((unsigned)nb);
  const GLLk G = g_gll_host;
  if (sc == 4) hipLaunchKernelGGL(k_acoustic_batch<1>, grid, dim3(128), 0, st, a, G);
  else if (sc == 8) hipLaunchKernelGGL(k_acoustic_batch<2>, grid, dim3(256), 0, st, a, G);
  else fatal("launch_acoustic_batch", "shots per workgroup must be 4 or 8");
  SF_LAUNCH_CHECK("k_acoustic_batch");
}

}  // namespace sf
