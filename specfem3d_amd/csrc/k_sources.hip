// k_sources.hip -- point sources, adjoint sources and receiver interpolation.
//
// Sources and adjoint sources are flattened to (owner, point) pairs sorted into rounds like
// the face points (FacePoints.ispec holds the owner: source or adjoint-receiver index); a lane per
// point of round 0 follows the point's other pairs (FacePoints::next), so points shared by several
// sources are summed in the reference's source order by one launch without atomics.
// The step's source time functions or adjoint samples come as a launch argument (SrcVals): a copy
// from pinned memory to the device before the launch took 4 us of a 38 us step on 20x20x20 elements.
// Built with -ffp-contract=off (reference rounding).
#include "kernels.h"

namespace sf {

__device__ __forceinline__ realw src_val(const SrcVals& a, int i) { return a.p ? a.p[i] : a.v[i]; }

// compute_add_sources_viscoelastic.F90:145-152: a(:,iglob) += sourcearray(isrc,:,i,j,k) * stf(isrc)
__global__ void k_add_sources_el(int n0, const int* __restrict__ ig, const int* __restrict__ owner,
                                 const int* __restrict__ ploc, const int* __restrict__ next,
                                 const realw* __restrict__ arr, SrcVals stf, realw* accel) {
  const int t0 = blockIdx.x * blockDim.x + threadIdx.x;
  if (t0 >= n0) return;
  const int64_t g = ig[t0];
  realw ax = accel[3 * g], ay = accel[3 * g + 1], az = accel[3 * g + 2];
  for (int t = t0; t >= 0; t = next[t]) {
    const int s = owner[t];
    const realw* sa = arr + ((int64_t)s * 125 + ploc[t]) * 3;
    const realw st = src_val(stf, s);
    ax = ax + sa[0] * st;
    ay = ay + sa[1] * st;
    az = az + sa[2] * st;
  }
  accel[3 * g] = ax;
  accel[3 * g + 1] = ay;
  accel[3 * g + 2] = az;
}

// compute_add_sources_acoustic.f90: chi'' -= sourcearray * stf / kappa (pressure source)
__global__ void k_add_sources_ac(int n0, const int* __restrict__ ig, const int* __restrict__ owner,
                                 const int* __restrict__ ploc, const int* __restrict__ next,
                                 const realw* __restrict__ arr, const realw* __restrict__ kap,
                                 SrcVals stf, realw* potdd) {
  const int t0 = blockIdx.x * blockDim.x + threadIdx.x;
  if (t0 >= n0) return;
  const int g = ig[t0];
  realw a = potdd[g];
  for (int t = t0; t >= 0; t = next[t]) {
    const int s = owner[t];
    const int64_t q = (int64_t)s * 125 + ploc[t];
    a = a - arr[3 * q] * src_val(stf, s) / kap[q];
  }
  potdd[g] = a;
}

// compute_add_sources_viscoelastic.F90:226-245: a += adj(:,irec) * hxi heta hgamma (CUSTOM_REAL)
__global__ void k_adjoint_sources_el(int n0, const int* __restrict__ ig, const int* __restrict__ owner,
                                     const int* __restrict__ ploc, const int* __restrict__ next,
                                     const realw* __restrict__ h, SrcVals adj, realw* accel) {
  const int t0 = blockIdx.x * blockDim.x + threadIdx.x;
  if (t0 >= n0) return;
  const int64_t g = ig[t0];
  realw ax = accel[3 * g], ay = accel[3 * g + 1], az = accel[3 * g + 2];
  for (int t = t0; t >= 0; t = next[t]) {
    const int r = owner[t];
    const realw hl = h[(int64_t)r * 125 + ploc[t]];
    ax = ax + src_val(adj, 3 * r) * hl;
    ay = ay + src_val(adj, 3 * r + 1) * hl;
    az = az + src_val(adj, 3 * r + 2) * hl;
  }
  accel[3 * g] = ax;
  accel[3 * g + 1] = ay;
  accel[3 * g + 2] = az;
}

// compute_add_sources_acoustic.f90:205-235 (adjoint sources in fluid elements):
// chi'' += adj(1, irec) * hxi heta hgamma, the product of the CUSTOM_REAL interpolants, added as is
// (no 1/kappa, positive sign)
__global__ void k_adjoint_sources_ac(int n0, const int* __restrict__ ig, const int* __restrict__ owner,
                                     const int* __restrict__ ploc, const int* __restrict__ next,
                                     const realw* __restrict__ h, SrcVals adj, realw* potdd) {
  const int t0 = blockIdx.x * blockDim.x + threadIdx.x;
  if (t0 >= n0) return;
  const int g = ig[t0];
  realw a = potdd[g];
  for (int t = t0; t >= 0; t = next[t]) {
    const int r = owner[t];
    a = a + src_val(adj, 3 * r) * h[(int64_t)r * 125 + ploc[t]];
  }
  potdd[g] = a;
}

// receiver interpolation (compute_interpolated_dva.f90:84-100): double-precision sum of
// h_i h_j h_k u over the 125 element points, rotated by nu_rec; one wave64 per listed receiver.
// WAIT: the field waits to be summed (waiting_value).
template <bool WAIT, typename T>
__global__ void __launch_bounds__(64) k_seismo_el(int n, const int* __restrict__ list, const int* __restrict__ ig,
                                                  const double* __restrict__ h, const double* __restrict__ nu,
                                                  const realw* __restrict__ field, GatherArgs A,
                                                  const int* __restrict__ first, int what, realw* __restrict__ out) {
  if ((int)blockIdx.x >= n) return;
  const int r = list ? list[blockIdx.x] : (int)blockIdx.x;
  const int lane = threadIdx.x;
  double sx = 0.0, sy = 0.0, sz = 0.0;
  for (int p = lane; p < 125; p += 64) {
    const int64_t q = (int64_t)r * 125 + p, g = ig[q];
    const double hl = h[q];
    realw f[3];
    if (WAIT) {
      waiting_value<3, T>(A, what, g, first[q], f);
    } else {
#pragma unroll
      for (int c = 0; c < 3; c++) f[c] = field[3 * g + c];
    }
    sx += (double)f[0] * hl;
    sy += (double)f[1] * hl;
    sz += (double)f[2] * hl;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    sx += __shfl_xor(sx, off, 64);
    sy += __shfl_xor(sy, off, 64);
    sz += __shfl_xor(sz, off, 64);
  }
  if (lane == 0) {
    const double* n = nu + (int64_t)r * 9;
    out[3 * r] = (realw)(n[0] * sx + n[1] * sy + n[2] * sz);
    out[3 * r + 1] = (realw)(n[3] * sx + n[4] * sy + n[5] * sz);
    out[3 * r + 2] = (realw)(n[6] * sx + n[7] * sy + n[8] * sz);
  }
}

void launch_add_sources_el(hipStream_t s, const FacePoints& f, const realw* arr, const SrcVals& stf, realw* accel) {
  const int n0 = f.points();
  if (n0 <= 0) return;
  hipLaunchKernelGGL(k_add_sources_el, sf_grid(n0, 128), dim3(128), 0, s, n0, f.iglob, f.ispec, f.ploc, f.next,
                     arr, stf, accel);
  SF_LAUNCH_CHECK("k_add_sources_el");
}

void launch_add_sources_ac(hipStream_t s, const FacePoints& f, const realw* arr, const realw* kappa,
                           const SrcVals& stf, realw* potdd) {
  const int n0 = f.points();
  if (n0 <= 0) return;
  hipLaunchKernelGGL(k_add_sources_ac, sf_grid(n0, 128), dim3(128), 0, s, n0, f.iglob, f.ispec, f.ploc, f.next,
                     arr, kappa, stf, potdd);
  SF_LAUNCH_CHECK("k_add_sources_ac");
}

void launch_adjoint_sources_el(hipStream_t s, const FacePoints& f, const realw* h, const SrcVals& adj, realw* accel) {
  const int n0 = f.points();
  if (n0 <= 0) return;
  hipLaunchKernelGGL(k_adjoint_sources_el, sf_grid(n0, 128), dim3(128), 0, s, n0, f.iglob, f.ispec, f.ploc, f.next,
                     h, adj, accel);
  SF_LAUNCH_CHECK("k_adjoint_sources_el");
}

void launch_adjoint_sources_ac(hipStream_t s, const FacePoints& f, const realw* h, const SrcVals& adj, realw* potdd) {
  const int n0 = f.points();
  if (n0 <= 0) return;
  hipLaunchKernelGGL(k_adjoint_sources_ac, sf_grid(n0, 128), dim3(128), 0, s, n0, f.iglob, f.ispec, f.ploc, f.next,
                     h, adj, potdd);
  SF_LAUNCH_CHECK("k_adjoint_sources_ac");
}

void launch_seismo_el(hipStream_t s, int n, const int* list, const int* iglob, const double* h, const double* nu,
                      const realw* field, realw* out) {
  if (n <= 0) return;
  hipLaunchKernelGGL((k_seismo_el<false, float>), dim3(n), dim3(64), 0, s, n, list, iglob, h, nu, field, GatherArgs{},
                     nullptr, 0, out);
  SF_LAUNCH_CHECK("k_seismo_el");
}

void launch_seismo_el_waiting(hipStream_t s, int n, const int* list, const int* iglob, const double* h,
                              const double* nu, const GatherArgs& a, const int* first, int what, bool exact,
                              realw* out) {
  if (n <= 0) return;
  auto* kernel = exact ? &k_seismo_el<true, float> : &k_seismo_el<true, double>;
  hipLaunchKernelGGL(kernel, dim3(n), dim3(64), 0, s, n, list, iglob, h, nu, nullptr, a, first, what, out);
  SF_LAUNCH_CHECK("k_seismo_el");
}

}  // namespace sf
