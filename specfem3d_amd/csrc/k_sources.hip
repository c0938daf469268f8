// k_sources.hip -- receiver interpolation.
// Built with -ffp-contract=off (reference rounding).
#include "kernels.h"

namespace sf {

// receiver interpolation (compute_interpolated_dva.f90:84-100): double-precision sum of
// h_i h_j h_k u over the 125 element points, rotated by nu_rec; one wave64 per listed receiver.
// WAIT: the field waits to be summed (waiting_value).
template <bool WAIT>
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
      waiting_value<3>(A, what, g, first[q], f);
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

void launch_seismo_el(hipStream_t s, int n, const int* list, const int* iglob, const double* h, const double* nu,
                      const realw* field, realw* out) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_seismo_el<false>, dim3(n), dim3(64), 0, s, n, list, iglob, h, nu, field, GatherArgs{},
                     nullptr, 0, out);
  SF_LAUNCH_CHECK("k_seismo_el");
}

void launch_seismo_el_waiting(hipStream_t s, int n, const int* list, const int* iglob, const double* h,
                              const double* nu, const GatherArgs& a, const int* first, int what, realw* out) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_seismo_el<true>, dim3(n), dim3(64), 0, s, n, list, iglob, h, nu, nullptr, a, first, what, out);
  SF_LAUNCH_CHECK("k_seismo_el");
}

}  // namespace sf
