// k_boundary.hip -- face-point kernels: Stacey absorbing boundaries, fluid-solid coupling,
// acoustic free surface.
//
// Faces are flattened at prepare time into face points carrying the global index, normal, weight and
// impedances, and sorted into "rounds" (the r-th occurrence of a global point in the host's face order).
// One launch per term: a lane per point of round 0 (the first occurrence of each global point) walks
// the point's occurrences in round order (FacePoints::next) and applies each face's term to a register
// copy, so the sums at points shared by several faces are accumulated in the reference's face order and
// are deterministic. The launches are bound by the latency of their chain of loads, so one launch of
// chains beats a launch per round (us, rounds -> chain): fluid Stacey on 40x40x30 elements 4 x 3.3 ->
// 6.1, on 19x17x4 4 x 2.5 -> 5.0; the coupling there 4 x 2.4 -> 3.9 and 4 x 2.2 -> 3.1; elastic Stacey
// with 0.63 M points 37 -> 21.7. One launch with float atomics: 65 us for the last, and 4.6 against 6.3
// (fluid Stacey), 7.9 against 5.2 and 4.6 against 5.2 (coupling) on 64x64x32.
// Built with -ffp-contract=off (reference rounding).
#include "kernels.h"

namespace sf {

// Stacey elastic (compute_stacey_viscoelastic.F90:85-118):
//   t = rho vp (v.n) n + rho vs (v - (v.n) n);  a -= t w
// `store` (optional) receives t w at the point's record slot (SAVE_FORWARD boundary record).
__global__ void k_stacey_el(int n0, const int* __restrict__ ig, const realw* __restrict__ nrm,
                                  const realw* __restrict__ jw, const realw* __restrict__ rvp,
                                  const realw* __restrict__ rvs, const int* __restrict__ slot,
                                  const int* __restrict__ next, const realw* __restrict__ veloc, realw* accel,
                                  realw* __restrict__ store) {
  const int t0 = blockIdx.x * blockDim.x + threadIdx.x;
  if (t0 >= n0) return;
  const int64_t g = ig[t0];
  const realw vx = veloc[3 * g], vy = veloc[3 * g + 1], vz = veloc[3 * g + 2];
  realw ax = accel[3 * g], ay = accel[3 * g + 1], az = accel[3 * g + 2];
  for (int t = t0; t >= 0; t = next[t]) {
    const realw nx = nrm[3 * t], ny = nrm[3 * t + 1], nz = nrm[3 * t + 2];
    const realw vn = vx * nx + vy * ny + vz * nz;
    const realw p = rvp[t], s = rvs[t];
    const realw tx = p * vn * nx + s * (vx - vn * nx);
    const realw ty = p * vn * ny + s * (vy - vn * ny);
    const realw tz = p * vn * nz + s * (vz - vn * nz);
    const realw w = jw[t];
    const realw fx = tx * w, fy = ty * w, fz = tz * w;
    ax = ax - fx;
    ay = ay - fy;
    az = az - fz;
    if (store) {
      const int q = slot[t];
      store[3 * q] = fx;
      store[3 * q + 1] = fy;
      store[3 * q + 2] = fz;
    }
  }
  accel[3 * g] = ax;
  accel[3 * g + 1] = ay;
  accel[3 * g + 2] = az;
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

// Stacey acoustic (compute_stacey_acoustic.f90:96-112): chi'' -= chi' w / c / rho.
// imp_p holds rho, imp_s holds c = sqrt(kappa/rho), both per face point.
__global__ void k_stacey_ac(int n0, const int* __restrict__ ig, const realw* __restrict__ jw,
                            const realw* __restrict__ rho, const realw* __restrict__ cp, const int* __restrict__ slot,
                            const int* __restrict__ next, const realw* __restrict__ potd, realw* potdd,
                            realw* __restrict__ store) {
  const int t0 = blockIdx.x * blockDim.x + threadIdx.x;
  if (t0 >= n0) return;
  const int g = ig[t0];
  const realw v = potd[g];
  realw a = potdd[g];
  for (int t = t0; t >= 0; t = next[t]) {
    const realw absorbl = v * jw[t] / cp[t] / rho[t];
    a = a - absorbl;
    if (store) store[slot[t]] = absorbl;
  }
  potdd[g] = a;
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

// acoustic side of the coupling (compute_coupling_acoustic_el.f90:84-151): chi'' += w (u.n)
__global__ void k_coupling_ac_el(int n0, const int* __restrict__ ig, const realw* __restrict__ nrm,
                                 const realw* __restrict__ jw, const int* __restrict__ next,
                                 const realw* __restrict__ displ, realw* potdd, int flip) {
  const int t0 = blockIdx.x * blockDim.x + threadIdx.x;
  if (t0 >= n0) return;
  const int64_t g = ig[t0];
  realw ux = displ[3 * g], uy = displ[3 * g + 1], uz = displ[3 * g + 2];
  if (flip) { ux = -ux; uy = -uy; uz = -uz; }
  realw a = potdd[g];
  for (int t = t0; t >= 0; t = next[t]) {
    const realw un = ux * nrm[3 * t] + uy * nrm[3 * t + 1] + uz * nrm[3 * t + 2];
    a = a + jw[t] * un;
  }
  potdd[g] = a;
}

// elastic side (compute_coupling_viscoelastic_ac.f90:84-160): a += w n (-chi'')
__global__ void k_coupling_el_ac(int n0, const int* __restrict__ ig, const realw* __restrict__ nrm,
                                 const realw* __restrict__ jw, const int* __restrict__ next,
                                 const realw* __restrict__ potdd, realw* accel, int flip) {
  const int t0 = blockIdx.x * blockDim.x + threadIdx.x;
  if (t0 >= n0) return;
  const int64_t g = ig[t0];
  realw pr = -potdd[g];
  if (flip) pr = -pr;
  realw ax = accel[3 * g], ay = accel[3 * g + 1], az = accel[3 * g + 2];
  for (int t = t0; t >= 0; t = next[t]) {
    const realw w = jw[t];
    ax = ax + w * nrm[3 * t] * pr;
    ay = ay + w * nrm[3 * t + 1] * pr;
    az = az + w * nrm[3 * t + 2] * pr;
  }
  accel[3 * g] = ax;
  accel[3 * g + 1] = ay;
  accel[3 * g + 2] = az;
}

__global__ void k_free_surface(int n, const int* __restrict__ ig, realw* pot, realw* potd, realw* potdd) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int g = ig[t];
  pot[g] = 0.f;
  potd[g] = 0.f;
  potdd[g] = 0.f;
}

void launch_stacey_elastic(hipStream_t s, const FacePoints& f, const realw* veloc, realw* accel, realw* b_absorb,
                           int mode) {
  const int n0 = f.points();
  if (n0 <= 0) return;
  hipLaunchKernelGGL(k_stacey_el, sf_grid(n0, 128), dim3(128), 0, s, n0, f.iglob, f.normal, f.jacw, f.imp_p, f.imp_s,
                     f.slot, f.next, veloc, accel, mode ? b_absorb : (realw*)nullptr);
  SF_LAUNCH_CHECK("k_stacey_el");
}

void launch_stacey_elastic_replay(hipStream_t s, const FacePoints& f, const realw* rec, realw* b_accel) {
  const int n0 = f.points();
  if (n0 <= 0) return;
  hipLaunchKernelGGL(k_stacey_el_replay, sf_grid(n0, 128), dim3(128), 0, s, n0, f.iglob, f.slot, f.next, rec, b_accel);
  SF_LAUNCH_CHECK("k_stacey_el_replay");
}

void launch_stacey_acoustic(hipStream_t s, const FacePoints& f, const realw* potd, realw* potdd, realw* b_absorb,
                            int mode) {
  const int n0 = f.points();
  if (n0 <= 0) return;
  hipLaunchKernelGGL(k_stacey_ac, sf_grid(n0, 128), dim3(128), 0, s, n0, f.iglob, f.jacw, f.imp_p, f.imp_s, f.slot,
                     f.next, potd, potdd, mode ? b_absorb : (realw*)nullptr);
  SF_LAUNCH_CHECK("k_stacey_ac");
}

void launch_stacey_acoustic_replay(hipStream_t s, const FacePoints& f, const realw* rec, realw* b_potdd) {
  const int n0 = f.points();
  if (n0 <= 0) return;
  hipLaunchKernelGGL(k_stacey_ac_replay, sf_grid(n0, 128), dim3(128), 0, s, n0, f.iglob, f.slot, f.next, rec, b_potdd);
  SF_LAUNCH_CHECK("k_stacey_ac_replay");
}

void launch_coupling_ac_el(hipStream_t s, const FacePoints& f, const realw* displ, realw* potdd, int flip) {
  const int n0 = f.points();
  if (n0 <= 0) return;
  hipLaunchKernelGGL(k_coupling_ac_el, sf_grid(n0, 128), dim3(128), 0, s, n0, f.iglob, f.normal, f.jacw, f.next, displ,
                     potdd, flip);
  SF_LAUNCH_CHECK("k_coupling_ac_el");
}

void launch_coupling_el_ac(hipStream_t s, const FacePoints& f, const realw* potdd, realw* accel, int flip) {
  const int n0 = f.points();
  if (n0 <= 0) return;
  hipLaunchKernelGGL(k_coupling_el_ac, sf_grid(n0, 128), dim3(128), 0, s, n0, f.iglob, f.normal, f.jacw, f.next, potdd,
                     accel, flip);
  SF_LAUNCH_CHECK("k_coupling_el_ac");
}

void launch_free_surface(hipStream_t s, const FacePoints& f, realw* pot, realw* potd, realw* potdd) {
  if (f.n <= 0) return;
  hipLaunchKernelGGL(k_free_surface, sf_grid(f.n, 128), dim3(128), 0, s, f.n, f.iglob, pot, potd, potdd);
  SF_LAUNCH_CHECK("k_free_surface");
}

}  // namespace sf
