// batch.hip -- batched many-shot forward engine: many independent shots (own sources, receivers
// and record lengths) on one mesh prepared through the reference C-ABI.
//
// The reference runs one shot per process (one Mesh_pointer, one source set, iterate_time.F90).
// Here a Batch borrows a prepared elastic Mesh (ibool, moduli, Jacobians, inverse mass, Stacey
// face points, element colours) and steps S interleaved wavefields together:
//   * layout: groups of eight shots, each a field of its own with rows of eight (batch_idx);
//   * shots are placed in decreasing order of record length, so the live shots at any step are
//     a prefix and a finished group costs no memory traffic;
//   * a mesh with fluid elements also steps S potentials over its acoustic range of global points
//     in the same layout: per step the potential predictor, fluid Stacey, fluid side of the coupling,
//     acoustic stiffness, its sum with the corrector and the free surface come first, then the solid
//     side of the coupling with the elastic boundary terms (the single-shot call order of
//     iterate_time.F90);
//   * one step = sum of the local forces with the corrector and predictor (k_batch_gather), Stacey,
//     with the receivers, source rounds, stiffness (one launch that stores local forces), and a kernel
//     that advances the device step counter after a step or a captured group. Every kernel reads the
//     counter, so a group of steps is captured once into a hipGraph and replayed;
//   * the per-point arithmetic and the order of every sum equal the single-shot path (same
//     kernels' expressions, same colour order, same order of faces), so each shot of a batch is
//     bit-identical to its single-shot run under assembly = 2 (FMA builds: under assembly 2 without
//     attenuation; 3 rounds the update another way, see newmark, and k_visco_batch fuses other products
//     than k_elastic_pt).
// Shots-per-workgroup are chosen by an autotuner that times each candidate for a few steps from rest
// and then resets the batch.
#include <algorithm>
#include <cstring>
#include <numeric>
#include <vector>

#include "kernels.h"

namespace sf {
void ensure_element_colors(Mesh* m);
void release_gather_assembly(Mesh* m);
int* regular_first(Mesh* m, const int* list, int n, int* nreg);
void ensure_acoustic_colors(Mesh* m);
bool element_is_elastic(Mesh* m, int e);

struct Batch {
  Mesh* m = nullptr;
  int nshots = 0, S = 0;
  int sc = 4, mode = 2;          // shots per workgroup; assembly (3: see newmark)
  int overlay = 0;               // "lds_overlay", kept for callers that set it (no effect)
  int max_nstep = 0;
  realw dt = 0.f, dt2 = 0.f, dtsq2 = 0.f;  // deltat, deltatover2, deltatsqover2
  std::vector<int> nstep_user;   // per user shot
  std::vector<int> slot_of;      // user shot -> slot
  int* d_nstep = nullptr;        // per slot (S entries, decreasing, padding 0)
  int* d_it = nullptr;           // step counter, plus 0, 1 .. IT_AHEAD - 1
  int at = 0;                    // entry that the launches of a step read
  int h_it = 1;                  // host mirror of the step counter
  realw *u = nullptr, *v = nullptr, *a = nullptr;
  bool att = false;              // 3-SLS attenuation: per-shot memory variables and strain
  bool ac = false;               // fluid elements: per-shot potentials over the acoustic range
  int64_t ac_g0 = 0, ac_n = 0;   // acoustic range [ac_g0, ac_g0 + ac_n) of global points
  realw *pot = nullptr, *potd = nullptr, *potdd = nullptr;
  realw *R = nullptr, *eps = nullptr;
  // gather assembly: slots of each global point in colour order, AF_TERM per global point, local forces
  // of `loc_groups` groups of eight shots (all of them unless the card has no room)
  int *asm_ptr = nullptr, *asm_idx = nullptr, *ac_ptr = nullptr, *ac_idx = nullptr;
  int* elems = nullptr;          // launch order where the solid has regular and irregular elements (regular_first)
  int nreg = 0;
  uint16_t* info = nullptr;
  realw *local = nullptr, *ac_local = nullptr;  // ac_local: behind the solid's, in the same allocation
  int loc_groups = 0;
  int max_groups = 1 << 20;      // "local_groups"
  // sources: (source, point) entries sorted into rounds (the k-th source of each shot)
  struct Src { int shot, ispec; std::vector<realw> arr, stf; };
  std::vector<Src> srcs;
  int src_n = 0, src_nrounds = 0;
  std::vector<int> src_round_off;
  int *src_ig = nullptr, *src_slot = nullptr, *src_id = nullptr, *src_ploc = nullptr;
  realw *src_arr = nullptr, *src_stf = nullptr;
  // receivers
  struct Rec { int shot, ispec; double h[125]; double nu[9]; };
  std::vector<Rec> recs;
  int nrec = 0;
  std::vector<int> rec_order;    // device receiver index -> position in recs
  int *rec_slot = nullptr, *rec_ig = nullptr;
  double *rec_h = nullptr, *rec_nu = nullptr;
  realw* seis = nullptr;         // [max_nstep][nrec][3]
  bool ready = false;
  // captured step groups
  hipGraphExec_t gexec = nullptr;
  int graph_steps = 0;
  // timing of the stiffness launches (sf_batch_time)
  bool timing = false;
  std::vector<hipEvent_t> ev;
  int ev_used = 0;
};

static Batch* batch_of(long h) {
  if (!h) fatal("sf_batch", "null batch handle");
  return reinterpret_cast<Batch*>(h);
}

// ------------------------------------------------------------------------------ kernels
// The step counter is kept with the next steps' values beside it: the steps of a captured group read one
// each, and one launch advances them all (a launch per step took 4.5 us of it).
constexpr int IT_AHEAD = 32;

static __device__ __forceinline__ int load_it(const int* it) {
  return __hip_atomic_load(it, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Corrector of the finished step and predictor of the next one for one value. FMA: FMA builds under assembly =
// 3 form the corrected velocity and the displacement with fused multiply-adds (the second half step adds
// the rounded product), else the operations are those of k_update.hip.
template <bool FMA>
__device__ __forceinline__ void newmark(realw& u, realw& v, realw a, realw M, realw dt2p, realw dt, realw dt2,
                                        realw dtsq2) {
  a = a * M;
  if (FMA) {
    v = fmaf(dt2p, a, v);
    u = fmaf(dtsq2, a, fmaf(dt, v, u));
  } else {
    v = v + dt2p * a;
    u = u + dt * v + dtsq2 * a;
  }
  v = v + dt2 * a;
}

// Newmark update of every live (row, shot) from an assembled accel: the corrector of the previous step
// fused with the predictor (k_update.hip arithmetic), where the local forces have no room for all
// groups (see enqueue_stiffness).
// A lane takes four consecutive shots of one row (a float4), blockIdx.y is the group of eight.
// Finished shots keep their values (their lanes store what they loaded).
template <bool FMA>
__global__ void __launch_bounds__(256) k_batch_update(int64_t nrow, const int* __restrict__ nstep,
                                                      const int* __restrict__ itp, realw* __restrict__ u,
                                                      realw* __restrict__ v, realw* __restrict__ a,
                                                      const realw* __restrict__ rm, realw dt2p, realw dt, realw dt2,
                                                      realw dtsq2) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = t >> 1;
  if (row >= nrow) return;
  const int it = load_it(itp);
  const int s = 8 * (int)blockIdx.y + 4 * (int)(t & 1);
  if (nstep[s] < it) return;                       // shots are sorted: the whole quad has finished
  const bool l1 = nstep[s + 1] >= it, l2 = nstep[s + 2] >= it, l3 = nstep[s + 3] >= it;
  const int64_t o = batch_idx(nrow, row, s);
  const float4 U0 = *reinterpret_cast<const float4*>(u + o);
  const float4 V0 = *reinterpret_cast<const float4*>(v + o);
  const float4 A0 = *reinterpret_cast<const float4*>(a + o);
  const realw M = rm[row];
  float4 U = U0, V = V0, A = A0;
  newmark<FMA>(U.x, V.x, A.x, M, dt2p, dt, dt2, dtsq2);
  newmark<FMA>(U.y, V.y, A.y, M, dt2p, dt, dt2, dtsq2);
  newmark<FMA>(U.z, V.z, A.z, M, dt2p, dt, dt2, dtsq2);
  newmark<FMA>(U.w, V.w, A.w, M, dt2p, dt, dt2, dtsq2);
  A = make_float4(0.f, 0.f, 0.f, 0.f);
  if (!l1) { U.y = U0.y; V.y = V0.y; A.y = A0.y; }
  if (!l2) { U.z = U0.z; V.z = V0.z; A.z = A0.z; }
  if (!l3) { U.w = U0.w; V.w = V0.w; A.w = A0.w; }
  *reinterpret_cast<float4*>(u + o) = U;
  *reinterpret_cast<float4*>(v + o) = V;
  *reinterpret_cast<float4*>(a + o) = A;
}

// Sum of the local forces of every live (row, quad of shots) in list order, a = a - local, and with STEP
// the corrector of the finished step and the predictor of the next one (the arithmetic of
// k_batch_update; a: read and cleared at AF_TERM points, zero elsewhere).
//
// The element colours with the Newmark update folded in, which this replaced, moved fewer bytes but
// scattered their accel, u and v stores over parts of cache lines: on 64x64x32 elements x 32 shots
// the element pass without its arithmetic took 7.3 of 7.4 ms, of which the stores 4.4 ms (9.5 GB, 2.2
// TB/s), and the shared points' u was read once per colour (6.3 instead of 3.3 GB). Here both passes
// store whole lines, the element pass is bound by its arithmetic (3.45 ms there: VALU 2.4 ms, HBM 2.1,
// LDS 1.6) and this one by HBM (3.97 ms, 20.7 GB, 5.2 TB/s). Steps before and after: 32x32x16 x 16
// shots 598 -> 473 us, 64x64x32 x 32 8.53 -> 7.28 ms, viscoelastic 18x18x12 x 8 319 -> 233 us and
// 40x40x20 x 16 4.02 -> 3.41 ms.
struct BatchGatherArgs {
  int64_t g0, n, nrow;           // global points [g0, g0 + n), rows of a group
  const int *ptr, *idx;
  const realw* local;
  int64_t loc_group;
  int first_group;               // group of blockIdx.y = 0 (and of the buffer's first block)
  const uint16_t* info;
  const int *nstep, *it;
  realw *u, *v, *a;
  const realw* rm;
  realw dt2p, dt, dt2, dtsq2;
};

// a -= the local forces of slots ptr[g] .. ptr[g + 1], `unit` floats per slot, four slots in flight
__device__ __forceinline__ void gather4(realw a[4], const int* ptr, const int* idx, int64_t g, const realw* local,
                                        int unit) {
  const int p0 = ptr[g], p1 = ptr[g + 1];
  for (int p = p0; p < p1; p += 4) {
    int k[4];
    float4 l[4];
#pragma unroll
    for (int w = 0; w < 4; w++) k[w] = p + w < p1 ? idx[p + w] : -1;
#pragma unroll
    for (int w = 0; w < 4; w++)
      if (k[w] >= 0) l[w] = *reinterpret_cast<const float4*>(local + (int64_t)k[w] * unit);
#pragma unroll
    for (int w = 0; w < 4; w++) {
      if (k[w] < 0) continue;
      a[0] = a[0] + (-l[w].x);
      a[1] = a[1] + (-l[w].y);
      a[2] = a[2] + (-l[w].z);
      a[3] = a[3] + (-l[w].w);
    }
  }
}

// contiguous blocks of points per XCD
__device__ __forceinline__ int64_t xcd_block() {
  const int nb = (int)gridDim.x, b = (int)blockIdx.x;
  const int q = nb >> 3, r = nb & 7, x = b & 7;
  return (int64_t)x * q + (x < r ? x : r) + (b >> 3);
}

template <bool STEP, bool FMA>
__global__ void __launch_bounds__(256) k_batch_gather(BatchGatherArgs A) {
  const int64_t t = xcd_block() * 256 + threadIdx.x;
  const int64_t pt = t / 6;
  if (pt >= A.n) return;
  const int cq = (int)(t - 6 * pt), c = cq >> 1;
  const int it = load_it(A.it);
  const int s = 8 * (A.first_group + (int)blockIdx.y) + 4 * (cq & 1);
  if (A.nstep[s] < it) return;                       // shots are sorted: the whole quad has finished
  const int64_t g = A.g0 + pt;
  const int64_t o = batch_idx(A.nrow, 3 * g + c, s);
  const bool term = (A.info[g] & AF_TERM) != 0;
  float4 U, V;
  realw a[4] = {0, 0, 0, 0};
  realw M = 0.f;
  if (STEP) {
    U = *reinterpret_cast<const float4*>(A.u + o);
    V = *reinterpret_cast<const float4*>(A.v + o);
    M = A.rm[3 * g + c];
  }
  if (term) {
    const float4 a0 = *reinterpret_cast<const float4*>(A.a + o);
    a[0] = a0.x; a[1] = a0.y; a[2] = a0.z; a[3] = a0.w;
  }
  gather4(a, A.ptr, A.idx, g, A.local + (int64_t)blockIdx.y * A.loc_group + 8 * c + 4 * (cq & 1), 24);
  if (!STEP) {
    *reinterpret_cast<float4*>(A.a + o) = make_float4(a[0], a[1], a[2], a[3]);
    return;
  }
  newmark<FMA>(U.x, V.x, a[0], M, A.dt2p, A.dt, A.dt2, A.dtsq2);
  if (A.nstep[s + 1] >= it) newmark<FMA>(U.y, V.y, a[1], M, A.dt2p, A.dt, A.dt2, A.dtsq2);
  if (A.nstep[s + 2] >= it) newmark<FMA>(U.z, V.z, a[2], M, A.dt2p, A.dt, A.dt2, A.dtsq2);
  if (A.nstep[s + 3] >= it) newmark<FMA>(U.w, V.w, a[3], M, A.dt2p, A.dt, A.dt2, A.dtsq2);
  *reinterpret_cast<float4*>(A.u + o) = U;
  *reinterpret_cast<float4*>(A.v + o) = V;
  if (term) *reinterpret_cast<float4*>(A.a + o) = make_float4(0.f, 0.f, 0.f, 0.f);
}

// the same for the potentials: chi'' -= local forces, then the corrector chi'' *= rmass, chi' += dt/2 chi''
// (rows g - g0; the boundary terms are in chi'' already). Points on the free surface (AF_EDGE) take no
// forces and no terms: their potentials start at zero and stay there.
__global__ void __launch_bounds__(256) k_batch_ac_gather(int64_t nrow, int64_t g0, const int* __restrict__ ptr,
                                                         const int* __restrict__ idx, const realw* __restrict__ local,
                                                         int64_t loc_group, int first_group,
                                                         const uint16_t* __restrict__ info,
                                                         const int* __restrict__ nstep, const int* __restrict__ itp,
                                                         realw* __restrict__ potd, realw* __restrict__ potdd,
                                                         const realw* __restrict__ rm, realw dt2) {
  const int64_t t = xcd_block() * 256 + threadIdx.x;
  const int64_t row = t >> 1;
  if (row >= nrow) return;
  const int it = load_it(itp);
  const int s = 8 * (first_group + (int)blockIdx.y) + 4 * (int)(t & 1);
  if (nstep[s] < it) return;
  const int64_t o = batch_idx(nrow, row, s);
  float4 V = *reinterpret_cast<const float4*>(potd + o);
  const float4 a0 = *reinterpret_cast<const float4*>(potdd + o);
  const realw M = rm[row];
  realw a[4] = {0, 0, 0, 0};
  if (!(info[g0 + row] & AF_EDGE)) {
    a[0] = a0.x; a[1] = a0.y; a[2] = a0.z; a[3] = a0.w;
    gather4(a, ptr, idx, g0 + row, local + (int64_t)blockIdx.y * loc_group + 4 * (int)(t & 1), 8);
  }
  float4 Ac = a0;
#define SF_AG(c, r)                          \
  if (r == 0 || nstep[s + r] >= it) {        \
    Ac.c = a[r] * M;                         \
    V.c = V.c + dt2 * Ac.c;                  \
  }
  SF_AG(x, 0) SF_AG(y, 1) SF_AG(z, 2) SF_AG(w, 3)
#undef SF_AG
  *reinterpret_cast<float4*>(potd + o) = V;
  *reinterpret_cast<float4*>(potdd + o) = Ac;
}

// Face terms: a lane takes one global point (a face point of round 0) of one live shot and follows the
// point's other face points (FacePoints::next), with the sums of k_boundary.hip. Eight consecutive lanes
// are the shots of a group, blockIdx.y is the group. A launch takes about 5 us of a captured step at any
// of these sizes: with one per term instead of one per round, and the free surface in the fluid's sum,
// a step of 18x18x12 elements x 8 shots under a sea has 12 launches instead of 26 and takes 233 -> 203 us.
struct FaceLane {
  int t0, s;
  bool live;
};
__device__ __forceinline__ FaceLane face_lane(int n0, const int* nstep, const int* itp) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  FaceLane f;
  f.t0 = t >> 3;
  f.s = 8 * (int)blockIdx.y + (t & 7);
  f.live = f.t0 < n0 && nstep[f.s] >= load_it(itp);
  return f;
}

// source entries of one round: accel += sourcearray * stf(it) (k_add_sources_el arithmetic)
__global__ void k_batch_sources(int n, int64_t nrow, int max_nstep, const int* __restrict__ ig, const int* __restrict__ slot,
                                const int* __restrict__ sid, const int* __restrict__ ploc,
                                const realw* __restrict__ arr, const realw* __restrict__ stf,
                                const int* __restrict__ nstep, const int* __restrict__ itp, realw* accel) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int s = slot[t];
  const int it = load_it(itp);
  if (nstep[s] < it) return;
  const realw* sa = arr + ((int64_t)sid[t] * 125 + ploc[t]) * 3;
  const realw st = stf[(int64_t)sid[t] * max_nstep + it - 1];
  const int64_t b = batch_idx(nrow, 3 * (int64_t)ig[t], s);
  accel[b] = accel[b] + sa[0] * st;
  accel[b + 8] = accel[b + 8] + sa[1] * st;
  accel[b + 16] = accel[b + 16] + sa[2] * st;
}

// receivers (k_seismo_el arithmetic): one wave64 per receiver, FP64 sums, rotation by nu
__device__ __forceinline__ void record(int r, int nrec, int64_t nrow, const int* __restrict__ slot,
                                       const int* __restrict__ ig, const double* __restrict__ h,
                                       const double* __restrict__ nu, const int* __restrict__ nstep,
                                       const int* __restrict__ itp, const realw* __restrict__ u,
                                       realw* __restrict__ seis) {
  if (r >= nrec) return;
  const int s = slot[r];
  const int it = load_it(itp);
  if (nstep[s] < it) return;
  const int lane = threadIdx.x & 63;
  double sx = 0.0, sy = 0.0, sz = 0.0;
  for (int p = lane; p < 125; p += 64) {
    const int64_t b = batch_idx(nrow, 3 * (int64_t)ig[(int64_t)r * 125 + p], s);
    const double hl = h[(int64_t)r * 125 + p];
    sx += (double)u[b] * hl;
    sy += (double)u[b + 8] * hl;
    sz += (double)u[b + 16] * hl;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    sx += __shfl_xor(sx, off, 64);
    sy += __shfl_xor(sy, off, 64);
    sz += __shfl_xor(sz, off, 64);
  }
  if (lane == 0) {
    const double* n = nu + (int64_t)r * 9;
    realw* o = seis + ((int64_t)(it - 1) * nrec + r) * 3;
    o[0] = (realw)(n[0] * sx + n[1] * sy + n[2] * sz);
    o[1] = (realw)(n[3] * sx + n[4] * sy + n[5] * sz);
    o[2] = (realw)(n[6] * sx + n[7] * sy + n[8] * sz);
  }
}

// Stacey (k_stacey_el arithmetic)
// and, in the blocks behind the first `fb`, the receivers: both need only the updated u and v, and a
// launch of its own for the receivers took 5 us of a captured step
__global__ void __launch_bounds__(256) k_batch_stacey_seismo(
    int fb, int n0, int64_t nrow, const int* __restrict__ ig, const realw* __restrict__ nrm,
    const realw* __restrict__ jw, const realw* __restrict__ rvp, const realw* __restrict__ rvs,
    const int* __restrict__ next, const int* __restrict__ nstep, const int* __restrict__ itp,
    const realw* __restrict__ veloc, realw* accel, int nrec, const int* __restrict__ slot,
    const int* __restrict__ rec_ig, const double* __restrict__ h, const double* __restrict__ nu,
    const realw* __restrict__ u, realw* __restrict__ seis) {
  if ((int)blockIdx.x >= fb) {
    // a wave per receiver
    record(((((int)blockIdx.x - fb) * (int)gridDim.y + (int)blockIdx.y) << 2) + (int)(threadIdx.x >> 6), nrec, nrow, slot,
           rec_ig, h, nu, nstep, itp, u, seis);
    return;
  }
  const FaceLane f = face_lane(n0, nstep, itp);
  if (!f.live) return;
  const int64_t b = batch_idx(nrow, 3 * (int64_t)ig[f.t0], f.s);
  const realw vx = veloc[b], vy = veloc[b + 8], vz = veloc[b + 16];
  realw ax = accel[b], ay = accel[b + 8], az = accel[b + 16];
  for (int q = f.t0; q >= 0; q = next[q]) {
    const realw nx = nrm[3 * q], ny = nrm[3 * q + 1], nz = nrm[3 * q + 2];
    const realw vn = vx * nx + vy * ny + vz * nz;
    const realw p = rvp[q], sv = rvs[q];
    const realw tx = p * vn * nx + sv * (vx - vn * nx);
    const realw ty = p * vn * ny + sv * (vy - vn * ny);
    const realw tz = p * vn * nz + sv * (vz - vn * nz);
    const realw w = jw[q];
    const realw fx = tx * w, fy = ty * w, fz = tz * w;
    ax = ax - fx;
    ay = ay - fy;
    az = az - fz;
  }
  accel[b] = ax;
  accel[b + 8] = ay;
  accel[b + 16] = az;
}

// ---- fluid domain: potentials over the acoustic range, rows g - g0
// Predictor on the potential rows of live shots (k_update.hip arithmetic): chi += dt chi' + dt^2/2 chi'',
// chi' += dt/2 chi'', chi'' = 0. A lane takes four consecutive shots of one row.
__global__ void __launch_bounds__(256) k_batch_ac_predictor(int64_t nrow, const int* __restrict__ nstep,
                                                            const int* __restrict__ itp, realw* __restrict__ pot,
                                                            realw* __restrict__ potd, realw* __restrict__ potdd,
                                                            realw dt, realw dt2, realw dtsq2) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = t >> 1;
  if (row >= nrow) return;
  const int it = load_it(itp);
  const int s = 8 * (int)blockIdx.y + 4 * (int)(t & 1);
  if (nstep[s] < it) return;
  const bool l1 = nstep[s + 1] >= it, l2 = nstep[s + 2] >= it, l3 = nstep[s + 3] >= it;
  const int64_t o = batch_idx(nrow, row, s);
  const float4 V0 = *reinterpret_cast<const float4*>(potd + o);
  const float4 A0 = *reinterpret_cast<const float4*>(potdd + o);
  const float4 U0 = *reinterpret_cast<const float4*>(pot + o);
  float4 U = U0, V = V0, A = A0;
#define SF_AP(c) U.c = U.c + dt * V.c + dtsq2 * A.c; V.c = V.c + dt2 * A.c; A.c = 0.f;
  SF_AP(x) SF_AP(y) SF_AP(z) SF_AP(w)
#undef SF_AP
  if (!l1) { U.y = U0.y; V.y = V0.y; A.y = A0.y; }
  if (!l2) { U.z = U0.z; V.z = V0.z; A.z = A0.z; }
  if (!l3) { U.w = U0.w; V.w = V0.w; A.w = A0.w; }
  *reinterpret_cast<float4*>(pot + o) = U;
  *reinterpret_cast<float4*>(potd + o) = V;
  *reinterpret_cast<float4*>(potdd + o) = A;
}

// fluid Stacey (k_stacey_ac arithmetic)
__global__ void k_batch_stacey_ac(int n0, int64_t nrow, int64_t g0, const int* __restrict__ ig,
                                  const realw* __restrict__ jw, const realw* __restrict__ rho,
                                  const realw* __restrict__ cp, const int* __restrict__ next,
                                  const int* __restrict__ nstep, const int* __restrict__ itp,
                                  const realw* __restrict__ potd, realw* potdd) {
  const FaceLane f = face_lane(n0, nstep, itp);
  if (!f.live) return;
  const int64_t b = batch_idx(nrow, (int64_t)ig[f.t0] - g0, f.s);
  const realw v = potd[b];
  realw a = potdd[b];
  for (int q = f.t0; q >= 0; q = next[q]) {
    const realw absorbl = v * jw[q] / cp[q] / rho[q];
    a = a - absorbl;
  }
  potdd[b] = a;
}

// fluid side of the coupling (k_coupling_ac_el arithmetic, forward field): chi'' += w (u . n)
__global__ void k_batch_coupling_ac_el(int n0, int64_t nrow, int64_t nrow_ac, int64_t g0, const int* __restrict__ ig,
                                       const realw* __restrict__ nrm, const realw* __restrict__ jw,
                                       const int* __restrict__ next, const int* __restrict__ nstep,
                                       const int* __restrict__ itp, const realw* __restrict__ u, realw* potdd) {
  const FaceLane f = face_lane(n0, nstep, itp);
  if (!f.live) return;
  const int64_t g = ig[f.t0];
  const int64_t e = batch_idx(nrow, 3 * g, f.s);
  const realw ux = u[e], uy = u[e + 8], uz = u[e + 16];
  const int64_t b = batch_idx(nrow_ac, g - g0, f.s);
  realw a = potdd[b];
  for (int q = f.t0; q >= 0; q = next[q]) {
    const realw un = ux * nrm[3 * q] + uy * nrm[3 * q + 1] + uz * nrm[3 * q + 2];
    a = a + jw[q] * un;
  }
  potdd[b] = a;
}

// solid side of the coupling (k_coupling_el_ac arithmetic, forward field): a += w n (-chi'')
__global__ void k_batch_coupling_el_ac(int n0, int64_t nrow, int64_t nrow_ac, int64_t g0, const int* __restrict__ ig,
                                       const realw* __restrict__ nrm, const realw* __restrict__ jw,
                                       const int* __restrict__ next, const int* __restrict__ nstep,
                                       const int* __restrict__ itp, const realw* __restrict__ potdd, realw* accel) {
  const FaceLane f = face_lane(n0, nstep, itp);
  if (!f.live) return;
  const int64_t g = ig[f.t0];
  const realw pr = -potdd[batch_idx(nrow_ac, g - g0, f.s)];
  const int64_t e = batch_idx(nrow, 3 * g, f.s);
  realw ax = accel[e], ay = accel[e + 8], az = accel[e + 16];
  for (int q = f.t0; q >= 0; q = next[q]) {
    const realw w = jw[q];
    ax = ax + w * nrm[3 * q] * pr;
    ay = ay + w * nrm[3 * q + 1] * pr;
    az = az + w * nrm[3 * q + 2] * pr;
  }
  accel[e] = ax;
  accel[e + 8] = ay;
  accel[e + 16] = az;
}

__global__ void k_batch_tick(int* itp, int n) { itp[threadIdx.x] = itp[threadIdx.x] + n; }

__global__ void k_batch_fill(int64_t n, realw* p) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = 0.f;
}

// ------------------------------------------------------------------------------ host side
template <typename T>
static T* balloc(int64_t n) {
  void* p = nullptr;
  if (hipMalloc(&p, sizeof(T) * (size_t)(n > 0 ? n : 1)) != hipSuccess)
    fatal("sf_batch", "out of device memory for the batched wavefields");
  return reinterpret_cast<T*>(p);
}
template <typename T>
static void bfree(T*& p) {
  if (p) (void)hipFree(p);
  p = nullptr;
}
template <typename T>
static T* bupload(const T* h, int64_t n) {
  T* d = balloc<T>(n);
  if (n > 0) SF_CHECK(hipMemcpy(d, h, sizeof(T) * (size_t)n, hipMemcpyHostToDevice));
  return d;
}

static void drop_graph(Batch* b) {
  // a replay of the executable graph may still run on the stream: wait for it before destroying
  if (b->gexec) {
    SF_CHECK(hipStreamSynchronize(b->m->stream));
    (void)hipGraphExecDestroy(b->gexec);
  }
  b->gexec = nullptr;
  b->graph_steps = 0;
}

static void zero_state(Batch* b) {
  Mesh* m = b->m;
  const int64_t n = 3 * (int64_t)m->nglob * b->S;
  for (realw* p : {b->u, b->v, b->a})
    hipLaunchKernelGGL(k_batch_fill, sf_grid(n, 256), dim3(256), 0, m->stream, n, p);
  if (b->ac) {
    const int64_t na = b->ac_n * b->S;
    for (realw* p : {b->pot, b->potd, b->potdd})
      hipLaunchKernelGGL(k_batch_fill, sf_grid(na, 256), dim3(256), 0, m->stream, na, p);
  }
  if (b->att) {
    const int64_t nr = 18 * (int64_t)m->nspec * 125 * b->S, ne = 6 * (int64_t)m->nspec * 125 * b->S;
    hipLaunchKernelGGL(k_batch_fill, sf_grid(nr, 256), dim3(256), 0, m->stream, nr, b->R);
    hipLaunchKernelGGL(k_batch_fill, sf_grid(ne, 256), dim3(256), 0, m->stream, ne, b->eps);
  }
  if (b->seis) {
    const int64_t ns = (int64_t)b->max_nstep * b->nrec * 3;
    hipLaunchKernelGGL(k_batch_fill, sf_grid(ns, 256), dim3(256), 0, m->stream, ns, b->seis);
  }
  SF_LAUNCH_CHECK("k_batch_fill");
  b->h_it = 1;
  int it[IT_AHEAD];
  for (int k = 0; k < IT_AHEAD; k++) it[k] = b->h_it + k;
  SF_CHECK(hipMemcpyAsync(b->d_it, it, sizeof(it), hipMemcpyHostToDevice, m->stream));
  SF_CHECK(hipStreamSynchronize(m->stream));
}

// First and last writers of each point when the colours run one after the other, for callers of
// sf_batch_point_flags: the element of a point's lowest colour writes first (unless Stacey or a source adds
// to the point before the colours), the element of its highest colour last. The engine sums per point and
// does not use them.
static int point_flags(int nglob, int nelem, const int* ibool0, const int* elems, const int* color,
                       const unsigned char* forced, unsigned char* flags) {
  std::vector<int> cmin((size_t)nglob, 1 << 30), cmax((size_t)nglob, -1), nlast((size_t)nglob, 0);
  for (int q = 0; q < nelem; q++)
    for (int p = 0; p < 125; p++) {
      const int g = ibool0[(size_t)elems[q] * 125 + p];
      cmin[g] = std::min(cmin[g], color[q]);
      cmax[g] = std::max(cmax[g], color[q]);
    }
  for (int q = 0; q < nelem; q++) {
    const int e = elems[q], c = color[q];
    for (int p = 0; p < 125; p++) {
      const int g = ibool0[(size_t)e * 125 + p];
      unsigned char f = forced[g] ? BF_ZERO : 0;
      if (c == cmin[g] && !forced[g]) f |= BF_FIRST;
      if (c == cmax[g]) {
        f |= BF_LAST;
        nlast[g]++;
      }
      flags[(size_t)e * 125 + p] = f;
    }
  }
  for (int g = 0; g < nglob; g++)
    if (cmax[g] >= 0 && nlast[g] != 1) return -1;  // two elements of one colour share the point
  return 0;
}

// room for the local forces of as many groups as the card takes, at least one
static realw* local_room(int64_t per_group, int groups, int* got) {
  for (int n = groups; n > 0; n /= 2) {
    void* p = nullptr;
    if (hipMalloc(&p, sizeof(realw) * (size_t)(per_group * n)) == hipSuccess) {
      *got = n;
      return reinterpret_cast<realw*>(p);
    }
    (void)hipGetLastError();
  }
  fatal("sf_batch", "out of device memory for the batched wavefields");
}

// slot lists in the colour order of the single-shot run, points that take boundary or source terms,
// buffers of the local forces
static void build_gather(Batch* b) {
  Mesh* m = b->m;
  if (!b->asm_ptr) b->elems = regular_first(m, m->elastic_elems, m->nspec_elastic, &b->nreg);
  if (!b->asm_ptr)
    (void)build_slot_lists(m->stream, m->nglob, m->nspec, m->nspec_elastic, m->el_color_elems, b->elems ? b->elems : m->elastic_elems,
                           m->nspec_elastic, 0, 3, 1, m->ibool, b->asm_ptr, b->asm_idx);
  if (b->ac && !b->ac_ptr)
    (void)build_slot_lists(m->stream, m->nglob, m->nspec, m->nspec_acoustic, m->ac_color_elems, m->acoustic_elems,
                           m->nspec_acoustic, 0, 1, 1, m->ibool, b->ac_ptr, b->ac_idx);
  if (!b->info) b->info = balloc<uint16_t>(m->nglob);
  if (!b->local) {
    // last, and the solid's and the fluid's together: the one must not take the room of the other
    const int64_t el = (int64_t)m->nspec_elastic * 3000, ac = b->ac ? (int64_t)m->nspec_acoustic * 1000 : 0;
    b->local = local_room(el + ac, std::min(b->S / 8, b->max_groups), &b->loc_groups);
    b->ac_local = b->local + el * b->loc_groups;
  }
  SF_CHECK(hipMemsetAsync(b->info, 0, sizeof(uint16_t) * (size_t)m->nglob, m->stream));
  if (m->stacey) launch_mark_points(m->stream, m->abs_el.n, m->abs_el.iglob, AF_TERM, b->info);
  if (b->ac) launch_mark_points(m->stream, m->coupling.n, m->coupling.iglob, AF_TERM, b->info);
  launch_mark_points(m->stream, b->src_n, b->src_ig, AF_TERM, b->info);
  if (b->ac) launch_mark_points(m->stream, m->free_ac.n, m->free_ac.iglob, AF_EDGE, b->info);
}

static BatchGatherArgs gather_args(Batch* b) {
  Mesh* m = b->m;
  BatchGatherArgs A;
  A.g0 = m->el_g0;
  A.n = m->el_n;
  A.nrow = 3 * (int64_t)m->nglob;
  A.ptr = b->asm_ptr;
  A.idx = b->asm_idx;
  A.local = b->local;
  A.loc_group = (int64_t)m->nspec_elastic * 3000;
  A.first_group = 0;
  A.info = b->info;
  A.nstep = b->d_nstep;
  A.it = b->d_it + b->at;
  A.u = b->u;
  A.v = b->v;
  A.a = b->a;
  A.rm = m->rmass;
  A.dt2p = b->dt2;
  A.dt = b->dt;
  A.dt2 = b->dt2;
  A.dtsq2 = b->dtsq2;
  return A;
}

static void enqueue_stiffness(Batch* b, hipStream_t st) {
  Mesh* m = b->m;
  BatchArgs A;
  std::memset(&A, 0, sizeof(A));
  A.elems = b->elems ? b->elems : m->elastic_elems;
  A.nelem = m->nspec_elastic;
  A.nreg = b->nreg;
  A.S = b->S;
  A.nrow = 3 * (int64_t)m->nglob;
  A.ibool = m->ibool;
  A.irregular = m->irregular;
  A.xix_regular = m->xix_regular;
  A.jacobian_regular = m->jacobian_regular;
  A.jac = m->jac;
  A.jac_plane = (int64_t)m->nspec_irregular * 125;
  A.kappamu = m->kappamu;
  A.u = b->u;
  A.v = b->v;
  A.dt = b->dt;
  A.loc_group = (int64_t)m->nspec_elastic * 3000;
  A.nstep = b->d_nstep;
  A.it = b->d_it + b->at;
  if (b->att) {
    A.R = b->R;
    A.eps = b->eps;
    A.fc_index = m->fc_index;
    A.fc_table = m->fc_table;
    A.fc_rows = m->fc_rows;
    A.fc = m->factor_common;
    A.fck = m->factor_common_kappa;
    A.nloc = (int64_t)m->nspec * 125;
    for (int s = 0; s < 3; s++) {
      A.alpha[s] = m->alphaval[s];
      A.beta[s] = m->betaval[s];
      A.gamma[s] = m->gammaval[s];
    }
  }
  const int groups = b->S / 8;
  for (int g = 0; g < groups; g += b->loc_groups) {
    const int n = std::min(b->loc_groups, groups - g);
    A.s_first = 8 * g;
    A.ngroups = 8 * n / b->sc;
    A.local = b->local - g * A.loc_group;            // indexed by the shot's own group
    if (b->att) launch_visco_batch(st, A, b->sc, m->exact != 0);
    else launch_elastic_batch(st, A, b->sc, m->exact != 0);
    if (b->loc_groups < groups) {
      // no room for the local forces of all groups: sum them into accel before the next ones
      BatchGatherArgs ga = gather_args(b);
      ga.first_group = g;
      const dim3 grid(sf_grid(6 * ga.n, 256).x, (unsigned)n);
      hipLaunchKernelGGL((k_batch_gather<false, false>), grid, dim3(256), 0, st, ga);
      SF_LAUNCH_CHECK("k_batch_gather");
    }
  }
}

// launches over (global point of the faces, shot)
static dim3 face_grid(const FacePoints& f, int S) { return dim3(sf_grid(8 * (int64_t)f.points(), 256).x, (unsigned)(S / 8)); }

// the fluid part of a step (the acoustic calls of iterate_time.F90 before the elastic ones):
// predictor, Stacey, coupling (fluid side), stiffness (all elements are inner at NPROC = 1, so the
// stiffness runs in phase 2, after the boundary terms of phase 1), corrector and free surface (the free
// surface before the forces finds its points at zero)
static void enqueue_fluid(Batch* b, hipStream_t st) {
  Mesh* m = b->m;
  const int S = b->S;
  const int64_t na = b->ac_n, nrow = 3 * (int64_t)m->nglob;
  const dim3 rows(sf_grid(2 * na, 256).x, (unsigned)(S / 8));
  hipLaunchKernelGGL(k_batch_ac_predictor, rows, dim3(256), 0, st, na, b->d_nstep, b->d_it + b->at, b->pot, b->potd,
                     b->potdd, b->dt, b->dt2, b->dtsq2);
  SF_LAUNCH_CHECK("k_batch_ac_predictor");
  const FacePoints& f = m->abs_ac;
  if (m->stacey && f.points() > 0) {
    hipLaunchKernelGGL(k_batch_stacey_ac, face_grid(f, S), dim3(256), 0, st, f.points(), na, b->ac_g0, f.iglob, f.jacw,
                       f.imp_p, f.imp_s, f.next, b->d_nstep, b->d_it + b->at, b->potd, b->potdd);
    SF_LAUNCH_CHECK("k_batch_stacey_ac");
  }
  const FacePoints& cf = m->coupling;
  if (cf.points() > 0) {
    hipLaunchKernelGGL(k_batch_coupling_ac_el, face_grid(cf, S), dim3(256), 0, st, cf.points(), nrow, na, b->ac_g0,
                       cf.iglob, cf.normal, cf.jacw, cf.next, b->d_nstep, b->d_it + b->at, b->u, b->potdd);
    SF_LAUNCH_CHECK("k_batch_coupling_ac_el");
  }
  BatchAcArgs A;
  std::memset(&A, 0, sizeof(A));
  A.elems = m->acoustic_elems;
  A.nelem = m->nspec_acoustic;
  A.nrow = na;
  A.g0 = b->ac_g0;
  A.ibool = m->ibool;
  A.irregular = m->irregular;
  A.xix_regular = m->xix_regular;
  A.jacobian_regular = m->jacobian_regular;
  A.jac = m->jac;
  A.jac_plane = (int64_t)m->nspec_irregular * 125;
  A.rho = m->rho;
  A.pot = b->pot;
  A.loc_group = (int64_t)m->nspec_acoustic * 1000;
  A.nstep = b->d_nstep;
  A.it = b->d_it + b->at;
  for (int g = 0; g < S / 8; g += b->loc_groups) {
    const int n = std::min(b->loc_groups, S / 8 - g);
    A.s_first = 8 * g;
    A.ngroups = 8 * n / b->sc;
    A.local = b->ac_local - g * A.loc_group;
    launch_acoustic_batch(st, A, b->sc, m->exact != 0);
    hipLaunchKernelGGL(k_batch_ac_gather, dim3(rows.x, (unsigned)n), dim3(256), 0, st, na, b->ac_g0, b->ac_ptr, b->ac_idx,
                       b->ac_local, A.loc_group, g, b->info, b->d_nstep, b->d_it + b->at, b->potd, b->potdd, m->rmass_ac + b->ac_g0,
                       b->dt2);
    SF_LAUNCH_CHECK("k_batch_ac_gather");
  }
}

// one time step; `first`: the wavefields are zero
static void enqueue_step(Batch* b, hipStream_t st, bool first) {
  Mesh* m = b->m;
  if (!first) {
    const bool fma = !m->exact && b->mode == 3;
    // sums, corrector and predictor (at rest before the first step: nothing to do)
    if (b->loc_groups == b->S / 8) {
      const BatchGatherArgs ga = gather_args(b);
      const dim3 grid(sf_grid(6 * ga.n, 256).x, (unsigned)(b->S / 8));
      if (fma) hipLaunchKernelGGL((k_batch_gather<true, true>), grid, dim3(256), 0, st, ga);
      else hipLaunchKernelGGL((k_batch_gather<true, false>), grid, dim3(256), 0, st, ga);
      SF_LAUNCH_CHECK("k_batch_gather");
    } else {
      const int64_t nrow = 3 * (int64_t)m->nglob;
      auto* update = fma ? &k_batch_update<true> : &k_batch_update<false>;
      hipLaunchKernelGGL(update, dim3(sf_grid(2 * nrow, 256).x, (unsigned)(b->S / 8)), dim3(256), 0, st, nrow,
                         b->d_nstep, b->d_it + b->at, b->u, b->v, b->a, m->rmass, b->dt2, b->dt, b->dt2, b->dtsq2);
      SF_LAUNCH_CHECK("k_batch_update");
    }
  }
  if (b->ac) enqueue_fluid(b, st);
  const FacePoints& f = m->abs_el;
  const int groups = b->S / 8, n0 = m->stacey ? f.points() : 0;
  const int fb = n0 > 0 ? (int)sf_grid(8 * (int64_t)n0, 256).x : 0, rb = (b->nrec + 4 * groups - 1) / (4 * groups);
  if (fb + rb > 0) {
    hipLaunchKernelGGL(k_batch_stacey_seismo, dim3((unsigned)(fb + rb), (unsigned)groups), dim3(256), 0, st, fb, n0,
                       3 * (int64_t)m->nglob, f.iglob, f.normal, f.jacw, f.imp_p, f.imp_s, f.next, b->d_nstep,
                       b->d_it + b->at, b->v, b->a, b->nrec, b->rec_slot, b->rec_ig, b->rec_h, b->rec_nu, b->u, b->seis);
    SF_LAUNCH_CHECK("k_batch_stacey_seismo");
  }
  const FacePoints& cf = m->coupling;
  if (b->ac && cf.points() > 0) {
    hipLaunchKernelGGL(k_batch_coupling_el_ac, face_grid(cf, b->S), dim3(256), 0, st, cf.points(), 3 * (int64_t)m->nglob,
                       b->ac_n, b->ac_g0, cf.iglob, cf.normal, cf.jacw, cf.next, b->d_nstep, b->d_it + b->at, b->potdd, b->a);
    SF_LAUNCH_CHECK("k_batch_coupling_el_ac");
  }
  for (int r = 0; r < b->src_nrounds; r++) {
    const int o = b->src_round_off[r], cnt = b->src_round_off[r + 1] - o;
    if (cnt <= 0) continue;
    hipLaunchKernelGGL(k_batch_sources, sf_grid(cnt, 128), dim3(128), 0, st, cnt, 3 * (int64_t)m->nglob, b->max_nstep, b->src_ig + o,
                       b->src_slot + o, b->src_id + o, b->src_ploc + o, b->src_arr, b->src_stf, b->d_nstep, b->d_it + b->at,
                       b->a);
    SF_LAUNCH_CHECK("k_batch_sources");
  }
  const bool timed = b->timing && b->ev_used + 2 <= (int)b->ev.size();
  if (timed) SF_CHECK(hipEventRecord(b->ev[b->ev_used], st));
  enqueue_stiffness(b, st);
  if (timed) {
    SF_CHECK(hipEventRecord(b->ev[b->ev_used + 1], st));
    b->ev_used += 2;
  }
}

// after n steps
static void enqueue_tick(Batch* b, hipStream_t st, int n) {
  hipLaunchKernelGGL(k_batch_tick, dim3(1), dim3(IT_AHEAD), 0, st, b->d_it, n);
  SF_LAUNCH_CHECK("k_batch_tick");
}

// advance n steps (eagerly for the first step and for a tail shorter than the captured group)
static void run_steps(Batch* b, int n, int graph_steps) {
  Mesh* m = b->m;
  n = std::min(n, b->max_nstep - b->h_it + 1);
  while (n > 0) {
    if (b->h_it == 1 || graph_steps <= 1 || n < graph_steps) {
      enqueue_step(b, m->stream, b->h_it == 1);
      enqueue_tick(b, m->stream, 1);
      b->h_it++;
      n--;
      continue;
    }
    if (!b->gexec || b->graph_steps != graph_steps) {
      drop_graph(b);
      hipGraph_t g;
      SF_CHECK(hipStreamBeginCapture(m->stream, hipStreamCaptureModeThreadLocal));
      for (int k = 0; k < graph_steps; k++) {
        b->at = k % IT_AHEAD;
        enqueue_step(b, m->stream, false);
        if (b->at == IT_AHEAD - 1 || k == graph_steps - 1) enqueue_tick(b, m->stream, b->at + 1);
      }
      b->at = 0;
      SF_CHECK(hipStreamEndCapture(m->stream, &g));
      SF_CHECK(hipGraphInstantiate(&b->gexec, g, nullptr, nullptr, 0));
      SF_CHECK(hipGraphDestroy(g));
      b->graph_steps = graph_steps;
    }
    SF_CHECK(hipGraphLaunch(b->gexec, m->stream));
    b->h_it += graph_steps;
    n -= graph_steps;
  }
}

}  // namespace sf

using namespace sf;

// Create a batch of `nshots` shots with record lengths nstep[i] on a prepared elastic mesh (after
// prepare_constants_device_ and prepare_fields_elastic_device_; sources/receivers of the mesh
// itself are not used), time step constants as the host computes them (prepare_timerun.F90:
// deltat, deltatover2 = deltat/2, deltatsqover2 = deltat^2/2). Returns the handle; shots are
// numbered 0..nshots-1 by the caller.
extern "C" long sf_batch_create(long* Mesh_pointer, int nshots, const int* nstep, realw deltat, realw deltatover2,
                                realw deltatsqover2) {
  Mesh* m = from_handle(Mesh_pointer);
  if (nshots <= 0) fatal("sf_batch_create", "need at least one shot");
  if (!m->rmass || !m->kappamu || m->nspec_elastic <= 0) fatal("sf_batch_create", "mesh has no prepared elastic domain");
  if (m->pml_n > 0) fatal("sf_batch_create", "C-PML meshes are not supported by the batched engine");
  if (m->nspec_acoustic > 0 && (!m->ac[0].pot || !m->rmass_ac))
    fatal("sf_batch_create", "mesh has fluid elements but prepare_fields_acoustic_device was not called");
  if (m->attenuation && !m->fc_index && !m->factor_common)
    fatal("sf_batch_create", "attenuation factors not prepared");
  Batch* b = new Batch();
  b->m = m;
  b->dt = deltat;
  b->dt2 = deltatover2;
  b->dtsq2 = deltatsqover2;
  b->nshots = nshots;
  release_gather_assembly(m);
  ensure_element_colors(m);
  if (m->nspec_acoustic > 0) {
    ensure_acoustic_colors(m);
    b->ac = true;
    b->ac_g0 = m->ac_g0;
    b->ac_n = m->ac_n;
  }
  b->S = (nshots + 7) / 8 * 8;
  if (b->S > 1024) fatal("sf_batch_create", "at most 1024 shots per batch");
  b->nstep_user.assign(nstep, nstep + nshots);
  for (int i = 0; i < nshots; i++)
    if (nstep[i] <= 0) fatal("sf_batch_create", "record lengths must be positive");
  b->max_nstep = *std::max_element(nstep, nstep + nshots);
  std::vector<int> order(nshots);
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return nstep[x] > nstep[y]; });
  b->slot_of.assign(nshots, 0);
  std::vector<int> ns(b->S, 0);
  for (int k = 0; k < nshots; k++) {
    b->slot_of[order[k]] = k;
    ns[k] = nstep[order[k]];
  }
  b->d_nstep = bupload(ns.data(), b->S);
  b->d_it = balloc<int>(IT_AHEAD);
  const int64_t n = 3 * (int64_t)m->nglob * b->S;
  b->u = balloc<realw>(n);
  b->v = balloc<realw>(n);
  b->a = balloc<realw>(n);
  if (b->ac) {
    b->pot = balloc<realw>(b->ac_n * b->S);
    b->potd = balloc<realw>(b->ac_n * b->S);
    b->potdd = balloc<realw>(b->ac_n * b->S);
  }
  if (m->attenuation) {
    b->att = true;
    b->mode = 3;
    b->R = balloc<realw>(18 * (int64_t)m->nspec * 125 * b->S);
    b->eps = balloc<realw>(6 * (int64_t)m->nspec * 125 * b->S);
  }
  return reinterpret_cast<long>(b);
}

// Add a moment-tensor or force source to a shot: element ispec (0-based), sourcearray in the
// reference's (NDIM,NGLLX,NGLLY,NGLLZ) order (component fastest), and the source-time-function
// value used at every step of the shot (stf[it-1] = real(stf_pre_compute) of step it).
extern "C" void sf_batch_add_source(long h, int shot, int ispec, const realw* sourcearray, const realw* stf) {
  Batch* b = batch_of(h);
  if (shot < 0 || shot >= b->nshots) fatal("sf_batch_add_source", "shot index out of range");
  if (ispec < 0 || ispec >= b->m->nspec) fatal("sf_batch_add_source", "element index out of range");
  if (!element_is_elastic(b->m, ispec))
    fatal("sf_batch_add_source", "batched sources must lie in elastic elements (single-shot runs take fluid ones)");
  Batch::Src s;
  s.shot = shot;
  s.ispec = ispec;
  s.arr.assign(sourcearray, sourcearray + 375);
  s.stf.assign(stf, stf + b->nstep_user[shot]);
  b->srcs.push_back(std::move(s));
  b->ready = false;
}

// Add a receiver to a shot: element ispec (0-based), Lagrange interpolants hxi/heta/hgamma (5 each,
// double) and the rotation nu (3x3, nu_rec(3,3) column-major as the reference passes it).
extern "C" void sf_batch_add_receiver(long h, int shot, int ispec, const double* hxi, const double* heta,
                                      const double* hgamma, const double* nu) {
  Batch* b = batch_of(h);
  if (shot < 0 || shot >= b->nshots) fatal("sf_batch_add_receiver", "shot index out of range");
  if (ispec < 0 || ispec >= b->m->nspec) fatal("sf_batch_add_receiver", "element index out of range");
  if (!element_is_elastic(b->m, ispec))
    fatal("sf_batch_add_receiver",
          "batched receivers must lie in elastic elements (single-shot runs record fluid ones)");
  Batch::Rec r;
  r.shot = shot;
  r.ispec = ispec;
  for (int p = 0; p < 125; p++) r.h[p] = hxi[p % 5] * heta[(p / 5) % 5] * hgamma[p / 25];
  // rotated component a = sum_b nu(a, b) u_b; nu_rec(3,3) column-major: nu(a,b) at a + 3 b
  for (int x = 0; x < 3; x++)
    for (int y = 0; y < 3; y++) r.nu[3 * x + y] = nu[x + 3 * y];
  b->recs.push_back(r);
  b->ready = false;
}

// Upload sources and receivers, zero the wavefields and seismograms, set the step counter to 1.
extern "C" void sf_batch_finalize(long h) {
  Batch* b = batch_of(h);
  Mesh* m = b->m;
  SF_CHECK(hipStreamSynchronize(m->stream));
  drop_graph(b);
  std::vector<int> hib((size_t)m->nspec * 125);
  SF_CHECK(hipMemcpy(hib.data(), m->ibool, sizeof(int) * hib.size(), hipMemcpyDeviceToHost));
  // sources: round of an entry = index of its source within its shot
  {
    std::vector<int> k_in_shot(b->srcs.size()), count(b->nshots, 0);
    for (size_t q = 0; q < b->srcs.size(); q++) k_in_shot[q] = count[b->srcs[q].shot]++;
    const int nr = b->srcs.empty() ? 0 : *std::max_element(count.begin(), count.end());
    std::vector<int> ig, slot, sid, ploc;
    b->src_round_off.assign(nr + 1, 0);
    for (int r = 0; r < nr; r++) {
      b->src_round_off[r] = (int)ig.size();
      for (size_t q = 0; q < b->srcs.size(); q++) {
        if (k_in_shot[q] != r) continue;
        for (int p = 0; p < 125; p++) {
          ig.push_back(hib[(size_t)b->srcs[q].ispec * 125 + p]);
          slot.push_back(b->slot_of[b->srcs[q].shot]);
          sid.push_back((int)q);
          ploc.push_back(p);
        }
      }
    }
    b->src_round_off[nr] = (int)ig.size();
    b->src_nrounds = nr;
    b->src_n = (int)ig.size();
    std::vector<realw> arr(b->srcs.size() * 375), stf(b->srcs.size() * (size_t)b->max_nstep, 0.f);
    for (size_t q = 0; q < b->srcs.size(); q++) {
      // (c, i, j, k) with c fastest -> [p][c]
      for (int p = 0; p < 125; p++)
        for (int c = 0; c < 3; c++) arr[q * 375 + p * 3 + c] = b->srcs[q].arr[c + 3 * p];
      std::copy(b->srcs[q].stf.begin(), b->srcs[q].stf.end(), stf.begin() + q * b->max_nstep);
    }
    bfree(b->src_ig); bfree(b->src_slot); bfree(b->src_id); bfree(b->src_ploc); bfree(b->src_arr); bfree(b->src_stf);
    b->src_ig = bupload(ig.data(), (int64_t)ig.size());
    b->src_slot = bupload(slot.data(), (int64_t)slot.size());
    b->src_id = bupload(sid.data(), (int64_t)sid.size());
    b->src_ploc = bupload(ploc.data(), (int64_t)ploc.size());
    b->src_arr = bupload(arr.data(), (int64_t)arr.size());
    b->src_stf = bupload(stf.data(), (int64_t)stf.size());
  }
  // receivers, device order = order of addition
  {
    b->nrec = (int)b->recs.size();
    std::vector<int> slot(b->nrec), ig((size_t)b->nrec * 125);
    std::vector<double> hh((size_t)b->nrec * 125), nu((size_t)b->nrec * 9);
    for (int r = 0; r < b->nrec; r++) {
      const Batch::Rec& R = b->recs[r];
      slot[r] = b->slot_of[R.shot];
      for (int p = 0; p < 125; p++) {
        ig[(size_t)r * 125 + p] = hib[(size_t)R.ispec * 125 + p];
        hh[(size_t)r * 125 + p] = R.h[p];
      }
      for (int q = 0; q < 9; q++) nu[(size_t)r * 9 + q] = R.nu[q];
    }
    bfree(b->rec_slot); bfree(b->rec_ig); bfree(b->rec_h); bfree(b->rec_nu); bfree(b->seis);
    b->rec_slot = bupload(slot.data(), (int64_t)slot.size());
    b->rec_ig = bupload(ig.data(), (int64_t)ig.size());
    b->rec_h = bupload(hh.data(), (int64_t)hh.size());
    b->rec_nu = bupload(nu.data(), (int64_t)nu.size());
    b->seis = balloc<realw>((int64_t)b->max_nstep * std::max(1, b->nrec) * 3);
  }
  build_gather(b);
  b->ready = true;
  zero_state(b);
}

// shots per workgroup (4 or 8; divides the padded shot count) and assembly (0, 2 or 3: every value sums in
// the colour order, and FMA builds round the update of 3 as newmark<true> does). The batch must be at step 1
// (new, or after sf_batch_reset).
extern "C" void sf_batch_set_options(long h, int shots_per_group, int assembly) {
  Batch* b = batch_of(h);
  if (shots_per_group != 4 && shots_per_group != 8)
    fatal("sf_batch_set_options", "shots per workgroup must be 4 or 8");
  if (assembly != 0 && assembly != 2 && assembly != 3)
    fatal("sf_batch_set_options", "assembly must be 0, 2 or 3");
  if (b->h_it != 1) fatal("sf_batch_set_options", "options change only at step 1 (call sf_batch_reset first)");
  if (b->att && assembly == 0) fatal("sf_batch_set_options", "viscoelastic batches take assembly 2 or 3");
  SF_CHECK(hipStreamSynchronize(b->m->stream));
  drop_graph(b);
  b->sc = shots_per_group;
  b->mode = assembly;
}

// "local_groups": groups of eight shots whose local forces are held at a time (at most all of them, the
// default where the card has the room; fewer save 24 B per local point and shot, 8 B in the fluid, and take
// an extra pass over accel; same bits). "lds_overlay" 0/1 is accepted and read back without effect: the elastic
// kernel's rows always share their LDS with the stress products. Unknown names are fatal.
extern "C" void sf_batch_set_tuning(long h, const char* name, int value) {
  Batch* b = batch_of(h);
  if (std::strcmp(name, "lds_overlay") == 0) {
    if (value < 0 || value > 1) fatal("sf_batch_set_tuning", "lds_overlay must be 0 or 1");
    SF_CHECK(hipStreamSynchronize(b->m->stream));
    drop_graph(b);
    b->overlay = value;
  } else if (std::strcmp(name, "local_groups") == 0) {
    if (value < 1) fatal("sf_batch_set_tuning", "local_groups must be positive");
    if (b->h_it != 1) fatal("sf_batch_set_tuning", "local_groups changes only at step 1 (call sf_batch_reset first)");
    SF_CHECK(hipStreamSynchronize(b->m->stream));
    drop_graph(b);
    bfree(b->local);
    b->max_groups = value;
    if (b->ready) build_gather(b);
  } else {
    fatal("sf_batch_set_tuning", "unknown tuning switch");
  }
}

extern "C" int sf_batch_get_tuning(long h, const char* name) {
  Batch* b = batch_of(h);
  if (std::strcmp(name, "lds_overlay") == 0) return b->overlay;
  if (std::strcmp(name, "local_groups") == 0) return b->loc_groups;
  fatal("sf_batch_get_tuning", "unknown tuning switch");
  return 0;
}

extern "C" void sf_batch_get_options(long h, int* shots_per_group, int* assembly) {
  Batch* b = batch_of(h);
  *shots_per_group = b->sc;
  *assembly = b->mode;
}

// advance `nsteps` steps (at most to the longest record); `graph_steps` > 1 captures that many
// steps into one hipGraph and replays it
extern "C" void sf_batch_run(long h, int nsteps, int graph_steps) {
  Batch* b = batch_of(h);
  if (!b->ready) fatal("sf_batch_run", "sf_batch_finalize not called after adding sources/receivers");
  run_steps(b, nsteps, graph_steps);
}

extern "C" int sf_batch_current_step(long h) { return batch_of(h)->h_it; }

// Seismograms of one shot: out[(it-1) * nrec_shot * 3 + r * 3 + c] for its receivers in the order
// they were added, for it = 1..nstep of the shot. Synchronises the stream.
extern "C" void sf_batch_seismograms(long h, int shot, realw* out) {
  Batch* b = batch_of(h);
  if (shot < 0 || shot >= b->nshots) fatal("sf_batch_seismograms", "shot index out of range");
  SF_CHECK(hipStreamSynchronize(b->m->stream));
  std::vector<int> mine;
  for (int r = 0; r < b->nrec; r++)
    if (b->recs[r].shot == shot) mine.push_back(r);
  if (mine.empty()) return;
  const int ns = b->nstep_user[shot];
  std::vector<realw> all((size_t)ns * b->nrec * 3);
  SF_CHECK(hipMemcpy(all.data(), b->seis, sizeof(realw) * all.size(), hipMemcpyDeviceToHost));
  const size_t nr = mine.size();
  for (int t = 0; t < ns; t++)
    for (size_t q = 0; q < nr; q++)
      for (int c = 0; c < 3; c++) out[((size_t)t * nr + q) * 3 + c] = all[((size_t)t * b->nrec + mine[q]) * 3 + c];
}

// Displacement of one shot (3*NGLOB, xyz interleaved) copied to the host; synchronises.
extern "C" void sf_batch_displ(long h, int shot, realw* out) {
  Batch* b = batch_of(h);
  if (shot < 0 || shot >= b->nshots) fatal("sf_batch_displ", "shot index out of range");
  SF_CHECK(hipStreamSynchronize(b->m->stream));
  const int64_t n = 3 * (int64_t)b->m->nglob;
  const int s = b->slot_of[shot];
  std::vector<realw> all((size_t)n * 8);           // the shot's group
  SF_CHECK(hipMemcpy(all.data(), b->u + batch_idx(n, 0, s & ~7), sizeof(realw) * all.size(), hipMemcpyDeviceToHost));
  for (int64_t q = 0; q < n; q++) out[q] = all[(size_t)q * 8 + (s & 7)];
}

// Potential of one shot over all global points (zero outside the acoustic range; all zero on a mesh
// without fluid elements). Synchronises the stream.
extern "C" void sf_batch_potential(long h, int shot, realw* out) {
  Batch* b = batch_of(h);
  if (shot < 0 || shot >= b->nshots) fatal("sf_batch_potential", "shot index out of range");
  SF_CHECK(hipStreamSynchronize(b->m->stream));
  const int64_t n = b->m->nglob;
  for (int64_t q = 0; q < n; q++) out[q] = 0.f;
  if (!b->ac) return;
  const int s = b->slot_of[shot];
  std::vector<realw> all((size_t)b->ac_n * 8);
  SF_CHECK(hipMemcpy(all.data(), b->pot + batch_idx(b->ac_n, 0, s & ~7), sizeof(realw) * all.size(),
                     hipMemcpyDeviceToHost));
  for (int64_t q = 0; q < b->ac_n; q++) out[b->ac_g0 + q] = all[(size_t)q * 8 + (s & 7)];
}

// Rewind to step 1 with zero wavefields and seismograms (keeps sources, receivers and options).
extern "C" void sf_batch_reset(long h) {
  Batch* b = batch_of(h);
  SF_CHECK(hipStreamSynchronize(b->m->stream));
  zero_state(b);
}

// Time `nsteps` eager steps from the current state: average milliseconds of the stiffness launches
// per step (HIP events around them on the mesh stream) and of the whole step.
extern "C" void sf_batch_time(long h, int nsteps, double* stiffness_ms, double* step_ms) {
  Batch* b = batch_of(h);
  Mesh* m = b->m;
  nsteps = std::min(nsteps, b->max_nstep - b->h_it + 1);
  if (nsteps <= 0) fatal("sf_batch_time", "no steps left to time");
  b->ev.resize(2 * (size_t)nsteps + 2);
  for (auto& e : b->ev) SF_CHECK(hipEventCreate(&e));
  b->ev_used = 0;
  b->timing = true;
  hipEvent_t t0 = b->ev[2 * nsteps], t1 = b->ev[2 * nsteps + 1];
  b->ev.resize(2 * (size_t)nsteps);
  SF_CHECK(hipEventRecord(t0, m->stream));
  run_steps(b, nsteps, 1);
  SF_CHECK(hipEventRecord(t1, m->stream));
  SF_CHECK(hipStreamSynchronize(m->stream));
  b->timing = false;
  double tot = 0.0;
  for (int k = 0; k + 1 < b->ev_used; k += 2) {
    float ms = 0.f;
    SF_CHECK(hipEventElapsedTime(&ms, b->ev[k], b->ev[k + 1]));
    tot += ms;
  }
  float all = 0.f;
  SF_CHECK(hipEventElapsedTime(&all, t0, t1));
  *stiffness_ms = tot / std::max(1, b->ev_used / 2);
  *step_ms = (double)all / nsteps;
  for (auto& e : b->ev) (void)hipEventDestroy(e);
  (void)hipEventDestroy(t0);
  (void)hipEventDestroy(t1);
  b->ev.clear();
  b->ev_used = 0;
}

// Autotuner: times every shots-per-workgroup candidate for `trial_steps` eager steps from rest (after a
// warm-up; a candidate whose first step takes over twice the best so far is dropped), keeps the
// fastest and rewinds the batch. Returns the chosen step time in ms.
// The assembly becomes 3 from 25000 elements x shots on, with attenuation from 160000, and 2 below. Both are
// the same launches here and differ in the rounding of FMA builds alone (see newmark); the lines are
// where trials found 3 faster while it folded the update into the element launches, so that records of weak
// arrivals, which show that rounding, stay what they were. 14 batches without attenuation of 7900 to 262000
// elements x shots: 2 up to 20600, 3 from 33000 on (three took now one, now the other); 19 with attenuation of
// 8400 to 1.05 million: 2 up to 138000, 3 from 197000 on, between them either.
extern "C" double sf_batch_autotune(long h, int trial_steps) {
  Batch* b = batch_of(h);
  if (!b->ready) fatal("sf_batch_autotune", "sf_batch_finalize first");
  double best = 1e300;
  int best_sc = b->sc;
  for (int sc : {4, 8}) {
    if (b->S % sc) continue;
    b->sc = sc;
    drop_graph(b);
    zero_state(b);
    run_steps(b, 2, 1);  // warm-up (the first step has no update)
    double ks = 0.0, st = 0.0;
    sf_batch_time(h, 1, &ks, &st);
    if (st > 2.0 * best) continue;  // far behind the best so far: not worth the full trial
    sf_batch_time(h, trial_steps, &ks, &st);
    if (st < best) {
      best = st;
      best_sc = sc;
    }
  }
  b->sc = best_sc;
  b->mode = (int64_t)b->m->nspec_elastic * b->S >= (b->att ? 160000 : 25000) ? 3 : 2;
  drop_graph(b);
  zero_state(b);
  return best;
}

extern "C" void sf_batch_destroy(long h) {
  Batch* b = batch_of(h);
  SF_CHECK(hipStreamSynchronize(b->m->stream));
  drop_graph(b);
  bfree(b->d_nstep); bfree(b->d_it); bfree(b->u); bfree(b->v); bfree(b->a); bfree(b->R); bfree(b->eps);
  bfree(b->pot); bfree(b->potd); bfree(b->potdd);
  bfree(b->asm_ptr); bfree(b->asm_idx); bfree(b->ac_ptr); bfree(b->ac_idx); bfree(b->info);
  bfree(b->local); bfree(b->elems);
  bfree(b->src_ig); bfree(b->src_slot); bfree(b->src_id); bfree(b->src_ploc); bfree(b->src_arr); bfree(b->src_stf);
  bfree(b->rec_slot); bfree(b->rec_ig); bfree(b->rec_h); bfree(b->rec_nu); bfree(b->seis);
  delete b;
}

// Host-only (no device needed): per-local-point flags of a scatter colour by colour for elements elems[q] of
// colour color[q] (colours run in increasing order) and the points that Stacey or sources add to
// before the colours (forced[g] != 0): bit 1 first writer, bit 2 last writer, bit 4 a point that is
// added to before the colours. flags has 125 entries per element of ibool0. Returns 0, or -1 if two
// elements of one colour share a point.
extern "C" int sf_batch_point_flags(int nglob, int nelem, const int* ibool0, const int* elems, const int* color,
                                    const unsigned char* forced, unsigned char* flags) {
  return point_flags(nglob, nelem, ibool0, elems, color, forced, flags);
}
