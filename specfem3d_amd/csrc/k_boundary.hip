// k_boundary.hip -- face-point kernels: Stacey absorbing boundaries, fluid-solid coupling,
// acoustic free surface.
//
// Faces are flattened at prepare time into face points carrying the global index, normal, weight and
// impedances, and sorted into "rounds" (the r-th occurrence of a global point in the host's face order).
// The terms of a step that add to one field (Stacey, coupling, sources, adjoint sources; k_terms_*) run as
// one launch over the points that any of them touches: a lane holds the point's sum and walks, term by
// term, the point's occurrences in round order (FacePoints::next), so shared points are summed in the
// reference's order of terms, faces and sources, without atomics.
// The launches are bound by the latency of their chain of loads, so fewer are better (us, rounds ->
// a launch per term): fluid Stacey on 40x40x30 elements 4 x 3.3 -> 6.1, on 19x17x4 4 x 2.5 -> 5.0; the
// coupling there 4 x 2.4 -> 3.9 and 4 x 2.2 -> 3.1; elastic Stacey with 0.63 M points 37 -> 21.7. One
// launch per term with float atomics: 65 us for the last, and 4.6 against 6.3 (fluid Stacey), 7.9 against
// 5.2 and 4.6 against 5.2 (coupling) on 64x64x32.
// Together: Stacey and source on 20x20x20 5.3 + 2.5 -> 4.9; Stacey, coupling and source on 19x17x16 under a
// sea 5.5 + 3.1 + 2.8 -> 5.9 in the solid and 5.0 + 3.9 -> 5.6 in the fluid.
// Built with -ffp-contract=off (reference rounding).
#include "kernels.h"

namespace sf {

// Stacey elastic (compute_stacey_viscoelastic.F90:85-118), the faces t, next[t], ... of one point:
//   t = rho vp (v.n) n + rho vs (v - (v.n) n);  a -= t w
// `store` (optional) receives t w at the face's record slot (SAVE_FORWARD boundary record).
__device__ __forceinline__ void stacey_el(const FacePoints& f, int t, realw vx, realw vy, realw vz, realw a[3],
                                          realw* store) {
  for (; t >= 0; t = f.next[t]) {
    const realw nx = f.normal[3 * t], ny = f.normal[3 * t + 1], nz = f.normal[3 * t + 2];
    const realw vn = vx * nx + vy * ny + vz * nz;
    const realw p = f.imp_p[t], s = f.imp_s[t];
    const realw tx = p * vn * nx + s * (vx - vn * nx);
    const realw ty = p * vn * ny + s * (vy - vn * ny);
    const realw tz = p * vn * nz + s * (vz - vn * nz);
    const realw w = f.jacw[t];
    const realw fx = tx * w, fy = ty * w, fz = tz * w;
    a[0] = a[0] - fx;
    a[1] = a[1] - fy;
    a[2] = a[2] - fz;
    if (store) {
      const int q = f.slot[t];
      store[3 * q] = fx;
      store[3 * q + 1] = fy;
      store[3 * q + 2] = fz;
    }
  }
}

// Stacey acoustic (compute_stacey_acoustic.f90:96-112): chi'' -= chi' w / c / rho.
// imp_p holds rho, imp_s holds c = sqrt(kappa/rho), both per face point.
__device__ __forceinline__ void stacey_ac(const FacePoints& f, int t, realw v, realw& a, realw* store) {
  for (; t >= 0; t = f.next[t]) {
    const realw absorbl = v * f.jacw[t] / f.imp_s[t] / f.imp_p[t];
    a = a - absorbl;
    if (store) store[f.slot[t]] = absorbl;
  }
}

__device__ __forceinline__ realw src_val(const SrcVals& a, int i) { return a.p ? a.p[i] : a.v[i]; }

// the terms of the solid, in the reference's order
__global__ void __launch_bounds__(128) k_terms_el(TermArgs A) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= A.n) return;
  const int4 h = reinterpret_cast<const int4*>(A.head)[t];
  const int st = A.terms & TERM_STACEY ? h.x : -1, co = A.terms & TERM_COUPLING ? h.y : -1;
  const int so = A.terms & TERM_SOURCE ? h.z : -1, ad = A.terms & TERM_ADJOINT ? h.w : -1;
  if (st < 0 && co < 0 && so < 0 && ad < 0) return;
  const int64_t g = A.iglob[t];
  realw a[3] = {A.out[3 * g], A.out[3 * g + 1], A.out[3 * g + 2]};
  if (st >= 0) stacey_el(A.stacey, st, A.in[3 * g], A.in[3 * g + 1], A.in[3 * g + 2], a, nullptr);
  if (co >= 0) {
    // compute_coupling_viscoelastic_ac.f90:84-160: a += w n (-chi'')
    realw pr = -A.other[g];
    if (A.flip) pr = -pr;
    for (int q = co; q >= 0; q = A.coupling.next[q]) {
      const realw w = A.coupling.jacw[q];
#pragma unroll
      for (int c = 0; c < 3; c++) a[c] = a[c] + w * A.coupling.normal[3 * q + c] * pr;
    }
  }
  // compute_add_sources_viscoelastic.F90:145-152: a(:,iglob) += sourcearray(isrc,:,i,j,k) * stf(isrc)
  for (int q = so; q >= 0; q = A.source.next[q]) {
    const int s = A.source.ispec[q];
    const realw* sa = A.src_array + ((int64_t)s * 125 + A.source.ploc[q]) * 3;
    const realw v = src_val(A.src, s);
#pragma unroll
    for (int c = 0; c < 3; c++) a[c] = a[c] + sa[c] * v;
  }
  // compute_add_sources_viscoelastic.F90:226-245: a += adj(:,irec) * hxi heta hgamma (CUSTOM_REAL)
  for (int q = ad; q >= 0; q = A.adjoint.next[q]) {
    const int r = A.adjoint.ispec[q];
    const realw hl = A.adj_h[(int64_t)r * 125 + A.adjoint.ploc[q]];
#pragma unroll
    for (int c = 0; c < 3; c++) a[c] = a[c] + src_val(A.adj, 3 * r + c) * hl;
  }
#pragma unroll
  for (int c = 0; c < 3; c++) A.out[3 * g + c] = a[c];
}

// the terms of the fluid
__global__ void __launch_bounds__(128) k_terms_ac(TermArgs A) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= A.n) return;
  const int4 h = reinterpret_cast<const int4*>(A.head)[t];
  const int st = A.terms & TERM_STACEY ? h.x : -1, co = A.terms & TERM_COUPLING ? h.y : -1;
  const int so = A.terms & TERM_SOURCE ? h.z : -1, ad = A.terms & TERM_ADJOINT ? h.w : -1;
  if (st < 0 && co < 0 && so < 0 && ad < 0) return;
  const int64_t g = A.iglob[t];
  realw a = A.out[g];
  if (st >= 0) stacey_ac(A.stacey, st, A.in[g], a, nullptr);
  if (co >= 0) {
    // compute_coupling_acoustic_el.f90:84-151: chi'' += w (u.n)
    realw ux = A.other[3 * g], uy = A.other[3 * g + 1], uz = A.other[3 * g + 2];
    if (A.flip) { ux = -ux; uy = -uy; uz = -uz; }
    for (int q = co; q >= 0; q = A.coupling.next[q]) {
      const realw* n = A.coupling.normal + 3 * q;
      const realw un = ux * n[0] + uy * n[1] + uz * n[2];
      a = a + A.coupling.jacw[q] * un;
    }
  }
  // compute_add_sources_acoustic.f90: chi'' -= sourcearray * stf / kappa (pressure source)
  for (int q = so; q >= 0; q = A.source.next[q]) {
    const int s = A.source.ispec[q];
    const int64_t i = (int64_t)s * 125 + A.source.ploc[q];
    a = a - A.src_array[3 * i] * src_val(A.src, s) / A.src_kappa[i];
  }
  // compute_add_sources_acoustic.f90:205-235 (adjoint sources in fluid elements): chi'' += adj(1, irec) *
  // hxi heta hgamma, the product of the CUSTOM_REAL interpolants, added as is (no 1/kappa, positive sign)
  for (int q = ad; q >= 0; q = A.adjoint.next[q]) {
    const int r = A.adjoint.ispec[q];
    a = a + src_val(A.adj, 3 * r) * A.adj_h[(int64_t)r * 125 + A.adjoint.ploc[q]];
  }
  A.out[g] = a;
}

// Stacey alone, with the boundary record
__global__ void k_stacey_el(int n0, FacePoints f, const realw* __restrict__ veloc, realw* accel, realw* store) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n0) return;
  const int64_t g = f.iglob[t];
  realw a[3] = {accel[3 * g], accel[3 * g + 1], accel[3 * g + 2]};
  stacey_el(f, t, veloc[3 * g], veloc[3 * g + 1], veloc[3 * g + 2], a, store);
#pragma unroll
  for (int c = 0; c < 3; c++) accel[3 * g + c] = a[c];
}
__global__ void k_stacey_ac(int n0, FacePoints f, const realw* __restrict__ potd, realw* potdd, realw* store) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n0) return;
  const int g = f.iglob[t];
  realw a = potdd[g];
  stacey_ac(f, t, potd[g], a, store);
  potdd[g] = a;
}

// replay of a stored boundary record on the backward field (compute_stacey_viscoelastic.F90:274-283)
__global__ void k_stacey_el_replay(int n0, const int* __restrict__ ig, const int* __restrict__ slot,
                                   const int* __restrict__ next, const realw* __restrict__ rec, realw* b_accel) {
  const int t0 = blockIdx.x * blockDim.x + threadIdx.x;
  if (t0 >= n0) return;
  const int64_t g = ig[t0];
  realw ax = b_accel[3 * g], ay = b_accel[3 * g + 1], az = b_accel[3 * g + 2];
  for (int t = t0; t >= 0; t = next[t]) {
    const int q = slot[t];
    ax = ax - rec[3 * q];
    ay = ay - rec[3 * q + 1];
    az = az - rec[3 * q + 2];
  }
  b_accel[3 * g] = ax;
  b_accel[3 * g + 1] = ay;
  b_accel[3 * g + 2] = az;
}

__global__ void k_stacey_ac_replay(int n0, const int* __restrict__ ig, const int* __restrict__ slot,
                                   const int* __restrict__ next, const realw* __restrict__ rec, realw* b_potdd) {
  const int t0 = blockIdx.x * blockDim.x + threadIdx.x;
  if (t0 >= n0) return;
  const int g = ig[t0];
  realw a = b_potdd[g];
  for (int t = t0; t >= 0; t = next[t]) a = a - rec[slot[t]];
  b_potdd[g] = a;
}

__global__ void k_free_surface(int n, const int* __restrict__ ig, realw* pot, realw* potd, realw* potdd) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int g = ig[t];
  pot[g] = 0.f;
  potd[g] = 0.f;
  potdd[g] = 0.f;
}

void launch_terms(hipStream_t s, const TermArgs& a, bool fluid) {
  if (a.n <= 0) return;
  hipLaunchKernelGGL(fluid ? k_terms_ac : k_terms_el, sf_grid(a.n, 128), dim3(128), 0, s, a);
  SF_LAUNCH_CHECK("k_terms");
}

void launch_stacey_elastic(hipStream_t s, const FacePoints& f, const realw* veloc, realw* accel, realw* b_absorb) {
  const int n0 = f.points();
  if (n0 <= 0) return;
  hipLaunchKernelGGL(k_stacey_el, sf_grid(n0, 128), dim3(128), 0, s, n0, f, veloc, accel, b_absorb);
  SF_LAUNCH_CHECK("k_stacey_el");
}

void launch_stacey_elastic_replay(hipStream_t s, const FacePoints& f, const realw* rec, realw* b_accel) {
  const int n0 = f.points();
  if (n0 <= 0) return;
  hipLaunchKernelGGL(k_stacey_el_replay, sf_grid(n0, 128), dim3(128), 0, s, n0, f.iglob, f.slot, f.next, rec, b_accel);
  SF_LAUNCH_CHECK("k_stacey_el_replay");
}

void launch_stacey_acoustic(hipStream_t s, const FacePoints& f, const realw* potd, realw* potdd, realw* b_absorb) {
  const int n0 = f.points();
  if (n0 <= 0) return;
  hipLaunchKernelGGL(k_stacey_ac, sf_grid(n0, 128), dim3(128), 0, s, n0, f, potd, potdd, b_absorb);
  SF_LAUNCH_CHECK("k_stacey_ac");
}

void launch_stacey_acoustic_replay(hipStream_t s, const FacePoints& f, const realw* rec, realw* b_potdd) {
  const int n0 = f.points();
  if (n0 <= 0) return;
  hipLaunchKernelGGL(k_stacey_ac_replay, sf_grid(n0, 128), dim3(128), 0, s, n0, f.iglob, f.slot, f.next, rec, b_potdd);
  SF_LAUNCH_CHECK("k_stacey_ac_replay");
}

void launch_free_surface(hipStream_t s, const FacePoints& f, realw* pot, realw* potd, realw* potdd) {
  if (f.n <= 0) return;
  hipLaunchKernelGGL(k_free_surface, sf_grid(f.n, 128), dim3(128), 0, s, f.n, f.iglob, pot, potd, potdd);
  SF_LAUNCH_CHECK("k_free_surface");
}

}  // namespace sf
