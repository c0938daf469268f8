// k_assembly.hip -- structures of the gather assembly, built on the device.
//
// The element stiffness stores its local forces, three floats per local point (one in the fluid), and
// the pass that needs the assembled acceleration sums them (k_gather_update in k_update.hip). The sums need, per
// global point, the list of its local points in a fixed element order: a CSR, each point's entries
// sorted by the position of their element in a list. It is built here (count, scan, fill, sort each
// point's few entries) instead of on the host: 131072 elements take about a millisecond, a host
// loop over their 16.4 M local points about 0.2 s.
#include "kernels.h"

namespace sf {

constexpr int SCAN_BLOCK = 256, SCAN_PER = 8, SCAN_TILE = SCAN_BLOCK * SCAN_PER;

__global__ void k_fill_int(int64_t n, int v, int* __restrict__ p) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = v;
}

__global__ void k_list_position(int n, const int* __restrict__ list, int* __restrict__ pos, int first) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) pos[list[t]] = first + t;
}

__global__ void k_csr_count(int64_t n, const int* __restrict__ list, const int* __restrict__ ibool, int* cnt) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  atomicAdd(cnt + ibool[(int64_t)list[t / 125] * 125 + t % 125], 1);
}

// exclusive scan in three launches: tile sums, scan of the tile sums by one block, tiles
__global__ void __launch_bounds__(SCAN_BLOCK) k_scan_sums(int64_t n, const int* __restrict__ a, int* __restrict__ sums) {
  __shared__ int sm[SCAN_BLOCK];
  const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + threadIdx.x * SCAN_PER;
  int s = 0;
  for (int r = 0; r < SCAN_PER; r++) s += base + r < n ? a[base + r] : 0;
  sm[threadIdx.x] = s;
  __syncthreads();
  for (int w = SCAN_BLOCK / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sm[threadIdx.x] += sm[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) sums[blockIdx.x] = sm[0];
}

// exclusive prefix of one value per thread over the block; total returned in *tot
__device__ __forceinline__ int block_prefix(int v, int* sm, int* tot) {
  const int t = threadIdx.x;
  sm[t] = v;
  __syncthreads();
  for (int w = 1; w < SCAN_BLOCK; w <<= 1) {
    const int x = t >= w ? sm[t - w] : 0;
    __syncthreads();
    sm[t] += x;
    __syncthreads();
  }
  *tot = sm[SCAN_BLOCK - 1];
  const int r = sm[t] - v;
  __syncthreads();
  return r;
}

__global__ void __launch_bounds__(SCAN_BLOCK) k_scan_tops(int n, int* sums) {
  __shared__ int sm[SCAN_BLOCK];
  int carry = 0;
  for (int b = 0; b < n; b += SCAN_BLOCK) {
    const int t = b + threadIdx.x;
    int tot;
    const int v = t < n ? sums[t] : 0;
    const int x = block_prefix(v, sm, &tot);
    if (t < n) sums[t] = carry + x;
    carry += tot;
  }
}

__global__ void __launch_bounds__(SCAN_BLOCK) k_scan_tiles(int64_t n, int* a, const int* __restrict__ sums,
                                                           int* __restrict__ copy) {
  __shared__ int sm[SCAN_BLOCK];
  const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + threadIdx.x * SCAN_PER;
  int v[SCAN_PER], s = 0, tot;
  for (int r = 0; r < SCAN_PER; r++) {
    v[r] = base + r < n ? a[base + r] : 0;
    s += v[r];
  }
  int x = block_prefix(s, sm, &tot) + sums[blockIdx.x];
  for (int r = 0; r < SCAN_PER; r++) {
    if (base + r < n) {
      a[base + r] = x;
      copy[base + r] = x;
    }
    x += v[r];
  }
}

__global__ void k_csr_fill(int64_t n, const int* __restrict__ list, const int* __restrict__ ibool, int* cursor,
                           int* __restrict__ idx) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int slot = list[t / 125] * 125 + (int)(t % 125);
  idx[atomicAdd(cursor + ibool[slot], 1)] = slot;
}

// each point's slots by (position of the element in the list, slot): insertion sort, the lists are short
__global__ void k_csr_sort(int nglob, const int* __restrict__ ptr, const int* __restrict__ pos, int* idx) {
  const int g = blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= nglob) return;
  const int b = ptr[g], e = ptr[g + 1];
  for (int i = b + 1; i < e; i++) {
    const int s = idx[i], ps = pos[s / 125];
    int j = i;
    for (; j > b; j--) {
      const int o = idx[j - 1], po = pos[o / 125];
      if (po < ps || (po == ps && o < s)) break;
      idx[j] = o;
    }
    idx[j] = s;
  }
}

// 128-byte lines of the local forces that a wave over 64 consecutive points reads (one wave in 16 is
// counted): lanes whose w-th slot lies in another line than that of the lane before
__global__ void k_count_lines(int nglob, const int* __restrict__ ptr, const int* __restrict__ idx,
                              const int* __restrict__ pos, int ncomp, int eb, unsigned long long* lines) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int g = (t >> 6) * 1024 + (t & 63);
  const int b = g < nglob ? ptr[g] : 0, e = g < nglob ? ptr[g + 1] : 0;
  int n1 = 0, n2 = 0;
  for (int w = 0; w < 4; w++) {
    int l1 = -1, l2 = -1;
    if (b + w < e) {
      const int p = idx[b + w] % 125, q = pos[idx[b + w] / 125];
      l1 = (int)((int64_t)gather_slot(q, p / 5, p % 5, 1) * ncomp / 32);
      l2 = (int)((int64_t)gather_slot(q, p / 5, p % 5, eb) * ncomp / 32);
    }
    const int o1 = __shfl_up(l1, 1), o2 = __shfl_up(l2, 1);
    const bool head = (threadIdx.x & 63) == 0;
    n1 += l1 >= 0 && (head || l1 != o1);
    n2 += l2 >= 0 && (head || l2 != o2);
  }
  for (int off = 32; off > 0; off >>= 1) {
    n1 += __shfl_xor(n1, off);
    n2 += __shfl_xor(n2, off);
  }
  if ((threadIdx.x & 63) == 0) {
    atomicAdd(lines, (unsigned long long)n1);
    atomicAdd(lines + 1, (unsigned long long)n2);
  }
}

// e*125+p -> slot
__global__ void k_to_slots(int64_t n, const int* __restrict__ pos, int eb, int* idx) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int p = idx[t] % 125;
  idx[t] = gather_slot(pos[idx[t] / 125], p / 5, p % 5, eb);
}

__global__ void k_mark_points(int n, const int* __restrict__ ig, uint16_t bit, uint16_t* info) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  // several entries may name one point: they all write the same value (the kinds are marked one
  // launch after the other)
  if (t < n) info[ig[t]] |= bit;
}

__global__ void k_gather_info(int64_t g0, int64_t n, const int* __restrict__ ptr, const realw* __restrict__ rm,
                              uint16_t* __restrict__ info, int* __restrict__ base, realw* __restrict__ rm1) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int64_t g = g0 + t;
  bool same = true;
  if (rm) {
    const realw x = rm[3 * g], y = rm[3 * g + 1], z = rm[3 * g + 2];
    same = x == y && x == z;
    rm1[g] = x;
  }
  info[g] = (uint16_t)(((ptr[g + 1] - ptr[g]) << AF_COUNT) | (same ? 0 : AF_MASS3));
  if (t % 64 == 0) base[t / 64] = ptr[g];
}

__global__ void k_pick(int64_t n, const int* __restrict__ ig, const int* __restrict__ ptr, int* __restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) out[t] = ptr[ig[t]];
}

template <typename T>
static T* alloc_dev(int64_t n) {
  void* p = nullptr;
  SF_CHECK(hipMalloc(&p, sizeof(T) * (size_t)(n > 0 ? n : 1)));
  return reinterpret_cast<T*>(p);
}

int build_slot_lists(hipStream_t s, int nglob, int nspec, int nelem, const int* order, const int* launch, int nlaunch,
                     int pos0, int ncomp, int eb, const int* ibool, int*& ptr, int*& idx) {
  const int64_t nl = (int64_t)nelem * 125, np = (int64_t)nglob + 1;
  const int64_t ntile = (np + SCAN_TILE - 1) / SCAN_TILE;
  ptr = alloc_dev<int>(np);
  idx = alloc_dev<int>(nl);
  int* pos = alloc_dev<int>(nspec);
  int* cursor = alloc_dev<int>(np);
  int* sums = alloc_dev<int>(ntile);
  unsigned long long* lines = alloc_dev<unsigned long long>(2);
  hipLaunchKernelGGL(k_fill_int, sf_grid(np, 256), dim3(256), 0, s, np, 0, ptr);
  hipLaunchKernelGGL(k_fill_int, dim3(1), dim3(4), 0, s, (int64_t)4, 0, reinterpret_cast<int*>(lines));
  if (nelem > 0) {
    hipLaunchKernelGGL(k_list_position, sf_grid(nelem, 256), dim3(256), 0, s, nelem, order, pos, 0);
    hipLaunchKernelGGL(k_csr_count, sf_grid(nl, 256), dim3(256), 0, s, nl, order, ibool, ptr);
  }
  hipLaunchKernelGGL(k_scan_sums, dim3((unsigned)ntile), dim3(SCAN_BLOCK), 0, s, np, ptr, sums);
  hipLaunchKernelGGL(k_scan_tops, dim3(1), dim3(SCAN_BLOCK), 0, s, (int)ntile, sums);
  hipLaunchKernelGGL(k_scan_tiles, dim3((unsigned)ntile), dim3(SCAN_BLOCK), 0, s, np, ptr, sums, cursor);
  unsigned long long h[2] = {0, 0};
  if (nelem > 0) {
    hipLaunchKernelGGL(k_csr_fill, sf_grid(nl, 256), dim3(256), 0, s, nl, order, ibool, cursor, idx);
    hipLaunchKernelGGL(k_csr_sort, sf_grid(nglob, 256), dim3(256), 0, s, nglob, ptr, pos, idx);
    // launch positions: `launch` from 0, the elements of `order` behind its first nlaunch from pos0
    if (nlaunch > 0)
      hipLaunchKernelGGL(k_list_position, sf_grid(nlaunch, 256), dim3(256), 0, s, nlaunch, launch, pos, 0);
    if (nelem > nlaunch)
      hipLaunchKernelGGL(k_list_position, sf_grid(nelem - nlaunch, 256), dim3(256), 0, s, nelem - nlaunch,
                         order + nlaunch, pos, pos0);
    hipLaunchKernelGGL(k_count_lines, sf_grid((nglob + 1023) / 1024 * 64, 256), dim3(256), 0, s, nglob, ptr, idx, pos, ncomp,
                       eb, lines);
    SF_CHECK(hipMemcpyAsync(h, lines, sizeof(h), hipMemcpyDeviceToHost, s));
    SF_CHECK(hipStreamSynchronize(s));
    if (h[0] <= h[1]) eb = 1;
    hipLaunchKernelGGL(k_to_slots, sf_grid(nl, 256), dim3(256), 0, s, nl, pos, eb, idx);
  }
  SF_LAUNCH_CHECK("build_slot_lists");
  SF_CHECK(hipStreamSynchronize(s));
  for (void* p : {(void*)pos, (void*)cursor, (void*)sums, (void*)lines}) (void)hipFree(p);
  return eb;
}

void launch_mark_points(hipStream_t s, int n, const int* ig, uint16_t bit, uint16_t* info) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_mark_points, sf_grid(n, 256), dim3(256), 0, s, n, ig, bit, info);
  SF_LAUNCH_CHECK("k_mark_points");
}

void launch_pick(hipStream_t s, int64_t n, const int* ig, const int* ptr, int* out) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_pick, sf_grid(n, 256), dim3(256), 0, s, n, ig, ptr, out);
  SF_LAUNCH_CHECK("k_pick");
}

void launch_gather_info(hipStream_t s, int64_t g0, int64_t n, const int* ptr, const realw* rm, uint16_t* info,
                        int* base, realw* rm1) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_gather_info, sf_grid(n, 256), dim3(256), 0, s, g0, n, ptr, rm, info, base, rm1);
  SF_LAUNCH_CHECK("k_gather_info");
}

}  // namespace sf
