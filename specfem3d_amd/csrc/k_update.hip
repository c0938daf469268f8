// k_update.hip -- Newmark time-marching streams (pure HBM-bound, float4 vectorised).
//
// predictor   (update_displacement_scheme.f90:359-410, :206-227):
//     u += dt v + dt^2/2 a ; v += dt/2 a ; a = 0
// corrector   (compute_forces_viscoelastic_calling_routine.F90:368-374 + update_veloc_elastic):
//     a *= rmass^-1 ; v += dt/2 a
// corrector+predictor fused: the corrector of step n followed by the predictor of step n+1
// in one pass (same arithmetic, one read and one write of u, v, a instead of two).
// All arrays are flat (3*nglob for vector fields, nglob for potentials) and the inverse
// mass is stored with the same layout, so each thread handles 4 consecutive floats.
// Built with -ffp-contract=off: identical rounding to the CPU reference.
#include "kernels.h"

namespace sf {

__global__ void k_predictor(int64_t n4, int64_t n, realw* __restrict__ u, realw* __restrict__ v,
                            realw* __restrict__ a, realw dt, realw dt2, realw dtsq2) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n4) {
    float4 U = reinterpret_cast<float4*>(u)[t];
    float4 V = reinterpret_cast<float4*>(v)[t];
    const float4 A = reinterpret_cast<float4*>(a)[t];
    U.x = U.x + dt * V.x + dtsq2 * A.x; V.x = V.x + dt2 * A.x;
    U.y = U.y + dt * V.y + dtsq2 * A.y; V.y = V.y + dt2 * A.y;
    U.z = U.z + dt * V.z + dtsq2 * A.z; V.z = V.z + dt2 * A.z;
    U.w = U.w + dt * V.w + dtsq2 * A.w; V.w = V.w + dt2 * A.w;
    reinterpret_cast<float4*>(u)[t] = U;
    reinterpret_cast<float4*>(v)[t] = V;
    reinterpret_cast<float4*>(a)[t] = make_float4(0.f, 0.f, 0.f, 0.f);
  }
  // scalar tail
  const int64_t r = 4 * n4 + t;
  if (t < 4 && r < n) {
    u[r] = u[r] + dt * v[r] + dtsq2 * a[r];
    v[r] = v[r] + dt2 * a[r];
    a[r] = 0.f;
  }
}

__global__ void k_corrector(int64_t n4, int64_t n, realw* __restrict__ v, realw* __restrict__ a,
                            const realw* __restrict__ rm, realw dt2) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n4) {
    float4 V = reinterpret_cast<float4*>(v)[t];
    float4 A = reinterpret_cast<float4*>(a)[t];
    const float4 M = reinterpret_cast<const float4*>(rm)[t];
    A.x = A.x * M.x; A.y = A.y * M.y; A.z = A.z * M.z; A.w = A.w * M.w;
    V.x = V.x + dt2 * A.x; V.y = V.y + dt2 * A.y; V.z = V.z + dt2 * A.z; V.w = V.w + dt2 * A.w;
    reinterpret_cast<float4*>(v)[t] = V;
    reinterpret_cast<float4*>(a)[t] = A;
  }
  const int64_t r = 4 * n4 + t;
  if (t < 4 && r < n) {
    a[r] = a[r] * rm[r];
    v[r] = v[r] + dt2 * a[r];
  }
}

// OLD = 1 also stores PML_displ_old = u + t1 v + t2 a of the corrected field before the predictor
// (the arithmetic of k_pml_store_old), for every point of the range
template <int OLD>
__global__ void k_corrector_predictor(int64_t n4, int64_t n, realw* __restrict__ u, realw* __restrict__ v,
                                      realw* __restrict__ a, const realw* __restrict__ rm, realw dt2p, realw dt,
                                      realw dt2, realw dtsq2, realw* __restrict__ old, realw t1, realw t2) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n4) {
    float4 U = reinterpret_cast<float4*>(u)[t];
    float4 V = reinterpret_cast<float4*>(v)[t];
    float4 A = reinterpret_cast<float4*>(a)[t];
    const float4 M = reinterpret_cast<const float4*>(rm)[t];
    float4 O;
#define SF_CP(c)                               \
  A.c = A.c * M.c;                             \
  V.c = V.c + dt2p * A.c;                      \
  if (OLD) O.c = U.c + t1 * V.c + t2 * A.c;    \
  U.c = U.c + dt * V.c + dtsq2 * A.c;          \
  V.c = V.c + dt2 * A.c;
    SF_CP(x) SF_CP(y) SF_CP(z) SF_CP(w)
#undef SF_CP
    reinterpret_cast<float4*>(u)[t] = U;
    reinterpret_cast<float4*>(v)[t] = V;
    reinterpret_cast<float4*>(a)[t] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (OLD) reinterpret_cast<float4*>(old)[t] = O;
  }
  const int64_t r = 4 * n4 + t;
  if (t < 4 && r < n) {
    realw ar = a[r] * rm[r];
    realw vr = v[r] + dt2p * ar;
    if (OLD) old[r] = u[r] + t1 * vr + t2 * ar;
    u[r] = u[r] + dt * vr + dtsq2 * ar;
    v[r] = vr + dt2 * ar;
    a[r] = 0.f;
  }
}

// PML_displ_old (update_displ_elastic_PML, update_displacement_scheme.f90:417-455) at the global points
// of the C-PML elements, from the field before the predictor: u + t1 v + t2 a with
// t1 = deltatover2 (1 - 2 theta), t2 = deltatsqover2 (1 - theta). Where a corrector is pending, the pass
// that runs it with the predictor stores the same for every point (OLD).
__global__ void k_pml_store_old(int n, const int* __restrict__ pts, const realw* __restrict__ u,
                                const realw* __restrict__ v, const realw* __restrict__ a, realw t1, realw t2,
                                realw* __restrict__ old) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int64_t g = pts[t];
#pragma unroll
  for (int c = 0; c < 3; c++) old[3 * g + c] = u[3 * g + c] + t1 * v[3 * g + c] + t2 * a[3 * g + c];
}

// Dirichlet condition on the outer faces of the C-PML layers (pml_impose_boundary_condition_elastic)
__global__ void k_zero_points(int n, const int* __restrict__ pts, realw* __restrict__ u, realw* __restrict__ v,
                              realw* __restrict__ a) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int64_t g = pts[t];
#pragma unroll
  for (int c = 0; c < 3; c++) {
    u[3 * g + c] = 0.f;
    v[3 * g + c] = 0.f;
    a[3 * g + c] = 0.f;
  }
}

// Gather assembly fused with the Newmark update: one lane per global point sums the point's local
// forces in list order, a = a - local[slot], then (KIND) the corrector and the predictor of the next
// step, with the arithmetic of the stream kernels above.
//
// Why a gather: the alternatives put the sums into the stiffness launch, as float atomics or as one
// read-modify-write launch per element colour. A store of the local forces and this pass move 24 B
// per local point plus 4 B of slot index; a colour launch reads and writes 24 B of accel for each of
// the point's elements, and eight small launches leave most of the chip idle on small meshes.
// Stiffness and update per step, before (colours without attenuation, atomics with it) and after,
// with the point-per-lane stiffness: 20x20x20 elastic 50 -> 25 us, 43x37x29 irregular 193 -> 152,
// 64x64x32 fluid over viscoelastic 958 -> 817.
//
// The pass is bound by HBM: 0.72 GB and 150 us on 64x64x32 elements. It took 194 us with three
// masses per point and a pointer array (0.81 GB) and 185 us without; the rest of the way came from
// the slots' order. Consecutive points run through consecutive elements (a structured numbering) or
// through one element (points numbered element by element): with one element's forces after the
// other's, a wave over a structured mesh takes 48 B out of each of 16 lines. build_slot_lists counts
// the lines of both orders and takes blocks of 20 elements (gather_slot) where those are fewer: 150
// us, and 99 -> 104 us for the stiffness launch that writes them (621 -> 643 with attenuation, one
// element per workgroup); blocks of 5, 10 and 40 elements: 156, 152, 149 us.
// `clean`: accel is known to be zero away from AF_TERM points (the previous pass left it so), and is
// neither read nor cleared there.
// The number of slots comes with the flags, 2 B per point, and the position of a point's first slot
// from a scan over the wave's 64 points. The three inverse masses of a point are equal away from the
// absorbing faces and read as one value there. Each XCD takes its blocks backwards: the element
// launches before and after go forwards, so both ends of this pass meet what the other pass left in
// the caches (188 -> 185 us forwards to backwards on 64x64x32).

// inclusive prefix sum over a wave64 (row shifts by 1, 2, 4, 8, then the last lanes of rows 0 / 0..1
// broadcast into the rows behind)
__device__ __forceinline__ int wave_prefix(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);
  return x;
}

template <int NC, int KIND, bool OLD>
__global__ void __launch_bounds__(256) k_gather_update(GatherArgs A) {
  const int nb = (int)gridDim.x, b = (int)blockIdx.x;
  const int q = nb >> 3, r = nb & 7, x = b & 7;  // contiguous blocks per XCD, last one first
  const int last = x < r ? q : q - 1;
  const int64_t t = (int64_t)(x * q + (x < r ? x : r) + last - (b >> 3)) * 256 + threadIdx.x;
  const int64_t g = A.g0 + t;
  const int fl = t < A.n ? A.info[g] : 0;
  const int cnt = fl >> AF_COUNT;
  const int p1w = wave_prefix(cnt);               // every lane of the wave takes part
  if (t >= A.n) return;
  int p1 = A.base[t >> 6] + p1w;
  const int p0 = p1 - cnt;
  const bool full = !A.clean || (fl & AF_TERM);
  realw a[NC], u[NC], v[NC], m[NC];
#pragma unroll
  for (int c = 0; c < NC; c++) {
    a[c] = 0;
    if (KIND != GATHER_ONLY) m[c] = A.rm1[g];
  }
#pragma unroll
  for (int c = 0; c < NC; c++) {
    if (KIND != GATHER_ONLY) v[c] = A.v[NC * g + c];
    if (KIND == GATHER_STEP) u[c] = A.u[NC * g + c];
  }
  const bool zero = fl & A.skip;
  if (full && !zero) {
#pragma unroll
    for (int c = 0; c < NC; c++) a[c] = A.a[NC * g + c];
  }
  if (NC == 3 && KIND != GATHER_ONLY && (fl & AF_MASS3)) {
#pragma unroll
    for (int c = 1; c < NC; c++) m[c] = A.rm[NC * g + c];
  }
  if (zero) p1 = p0;
  for (int s = p0; s < p1; s += 4) {  // four slots in flight (an interior face point has two)
    int k[4];
    realw l[4][NC];
#pragma unroll
    for (int w = 0; w < 4; w++) k[w] = s + w < p1 ? A.idx[s + w] : -1;
#pragma unroll
    for (int w = 0; w < 4; w++) {
      if (k[w] < 0) continue;
      const realw* o = A.local + NC * (int64_t)k[w];
#pragma unroll
      for (int c = 0; c < NC; c++) l[w][c] = o[c];
    }
#pragma unroll
    for (int w = 0; w < 4; w++) {
      if (k[w] < 0) continue;
#pragma unroll
      for (int c = 0; c < NC; c++) a[c] = a[c] + (-l[w][c]);
    }
  }
  if (KIND == GATHER_ONLY) {
    if (p1 > p0 || zero) {
#pragma unroll
      for (int c = 0; c < NC; c++) A.a[NC * g + c] = a[c];
    }
    return;
  }
#pragma unroll
  for (int c = 0; c < NC; c++) {
    a[c] = a[c] * m[c];
    v[c] = v[c] + A.dt2p * a[c];
    if (KIND == GATHER_STEP) {
      if (OLD) A.old[NC * g + c] = u[c] + A.t1 * v[c] + A.t2 * a[c];
      A.u[NC * g + c] = u[c] + A.dt * v[c] + A.dtsq2 * a[c];
      v[c] = v[c] + A.dt2 * a[c];
      if (full) A.a[NC * g + c] = 0.f;
    } else {
      A.a[NC * g + c] = a[c];
    }
    A.v[NC * g + c] = v[c];
  }
}

template <int NC, int KIND, bool OLD>
static void launch_gather(hipStream_t s, const GatherArgs& a) {
  hipLaunchKernelGGL((k_gather_update<NC, KIND, OLD>), sf_grid(a.n, 256), dim3(256), 0, s, a);
}

void launch_gather_update(hipStream_t s, const GatherArgs& a, int ncomp, int kind) {
  if (a.n <= 0) return;
  if (ncomp == 1) {
    if (kind == GATHER_ONLY) launch_gather<1, GATHER_ONLY, false>(s, a);
    else if (kind == GATHER_CORRECT) launch_gather<1, GATHER_CORRECT, false>(s, a);
    else launch_gather<1, GATHER_STEP, false>(s, a);
  } else {
    if (kind == GATHER_ONLY) launch_gather<3, GATHER_ONLY, false>(s, a);
    else if (kind == GATHER_CORRECT) launch_gather<3, GATHER_CORRECT, false>(s, a);
    else if (a.old) launch_gather<3, GATHER_STEP, true>(s, a);
    else launch_gather<3, GATHER_STEP, false>(s, a);
  }
  SF_LAUNCH_CHECK("k_gather_update");
}

static dim3 grid_for(int64_t n4, int block) {
  int64_t b = (n4 + block - 1) / block;
  if (b < 1) b = 1;
  return dim3((unsigned)b);
}

void launch_predictor(hipStream_t s, int64_t n, realw* u, realw* v, realw* a, realw dt, realw dt2, realw dtsq2) {
  if (n <= 0) return;
  const int64_t n4 = n / 4;
  hipLaunchKernelGGL(k_predictor, grid_for(n4, 256), dim3(256), 0, s, n4, n, u, v, a, dt, dt2, dtsq2);
  SF_LAUNCH_CHECK("k_predictor");
}

void launch_corrector(hipStream_t s, int64_t n, realw* v, realw* a, const realw* rmass, realw dt2) {
  if (n <= 0) return;
  const int64_t n4 = n / 4;
  hipLaunchKernelGGL(k_corrector, grid_for(n4, 256), dim3(256), 0, s, n4, n, v, a, rmass, dt2);
  SF_LAUNCH_CHECK("k_corrector");
}

void launch_corrector_predictor(hipStream_t s, int64_t n, realw* u, realw* v, realw* a, const realw* rmass,
                                realw dt2_prev, realw dt, realw dt2, realw dtsq2, realw* old, realw t1, realw t2) {
  if (n <= 0) return;
  const int64_t n4 = n / 4;
  if (old)
    hipLaunchKernelGGL(k_corrector_predictor<1>, grid_for(n4, 256), dim3(256), 0, s, n4, n, u, v, a, rmass,
                       dt2_prev, dt, dt2, dtsq2, old, t1, t2);
  else
    hipLaunchKernelGGL(k_corrector_predictor<0>, grid_for(n4, 256), dim3(256), 0, s, n4, n, u, v, a, rmass,
                       dt2_prev, dt, dt2, dtsq2, nullptr, 0.f, 0.f);
  SF_LAUNCH_CHECK("k_corrector_predictor");
}

void launch_pml_store_old(hipStream_t s, int n, const int* pts, const realw* u, const realw* v, const realw* a,
                          realw t1, realw t2, realw* old) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_pml_store_old, grid_for(n, 256), dim3(256), 0, s, n, pts, u, v, a, t1, t2, old);
  SF_LAUNCH_CHECK("k_pml_store_old");
}

void launch_zero_points(hipStream_t s, int n, const int* pts, realw* u, realw* v, realw* a) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_zero_points, grid_for(n, 256), dim3(256), 0, s, n, pts, u, v, a);
  SF_LAUNCH_CHECK("k_zero_points");
}

}  // namespace sf
