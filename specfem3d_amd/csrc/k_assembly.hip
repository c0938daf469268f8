// k_assembly.hip -- structures of the gather assembly, built on the device.
//
// The element stiffness stores its local forces, three floats per local point, and the pass that
// needs the assembled acceleration sums them (k_gather_update in k_update.hip). The sums need, per
// global point, the list of its local points in a fixed element order: a CSR of slots e*125+p, each
// point's slots sorted by the position of their element in a list. It is built here (count, scan,
// fill, sort each point's few slots) instead of on the host: 131072 elements take about a
// millisecond, a host loop over their 16.4 M local points about 0.2 s.
#include "kernels.h"

namespace sf {

constexpr int SCAN_BLOCK = 256, SCAN_PER = 8, SCAN_TILE = SCAN_BLOCK * SCAN_PER;

__global__ void k_fill_int(int64_t n, int v, int* __restrict__ p) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = v;
}

__global__ void k_list_position(int n, const int* __restrict__ list, int* __restrict__ pos) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) pos[list[t]] = t;
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

__global__ void k_mark_points(int n, const int* __restrict__ ig, unsigned char bit, unsigned char* flags) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  // several entries may name one point: they all write the same byte (the kinds are marked one
  // launch after the other)
  if (t < n) flags[ig[t]] |= bit;
}

template <typename T>
static T* alloc_dev(int64_t n) {
  void* p = nullptr;
  SF_CHECK(hipMalloc(&p, sizeof(T) * (size_t)(n > 0 ? n : 1)));
  return reinterpret_cast<T*>(p);
}

void build_slot_lists(hipStream_t s, int nglob, int nspec, int nelem, const int* list, const int* ibool, int*& ptr,
                      int*& idx) {
  const int64_t nl = (int64_t)nelem * 125, np = (int64_t)nglob + 1;
  const int64_t ntile = (np + SCAN_TILE - 1) / SCAN_TILE;
  ptr = alloc_dev<int>(np);
  idx = alloc_dev<int>(nl);
  int* pos = alloc_dev<int>(nspec);
  int* cursor = alloc_dev<int>(np);
  int* sums = alloc_dev<int>(ntile);
  hipLaunchKernelGGL(k_fill_int, sf_grid(np, 256), dim3(256), 0, s, np, 0, ptr);
  if (nelem > 0) {
    hipLaunchKernelGGL(k_list_position, sf_grid(nelem, 256), dim3(256), 0, s, nelem, list, pos);
    hipLaunchKernelGGL(k_csr_count, sf_grid(nl, 256), dim3(256), 0, s, nl, list, ibool, ptr);
  }
  hipLaunchKernelGGL(k_scan_sums, dim3((unsigned)ntile), dim3(SCAN_BLOCK), 0, s, np, ptr, sums);
  hipLaunchKernelGGL(k_scan_tops, dim3(1), dim3(SCAN_BLOCK), 0, s, (int)ntile, sums);
  hipLaunchKernelGGL(k_scan_tiles, dim3((unsigned)ntile), dim3(SCAN_BLOCK), 0, s, np, ptr, sums, cursor);
  if (nelem > 0) {
    hipLaunchKernelGGL(k_csr_fill, sf_grid(nl, 256), dim3(256), 0, s, nl, list, ibool, cursor, idx);
    hipLaunchKernelGGL(k_csr_sort, sf_grid(nglob, 256), dim3(256), 0, s, nglob, ptr, pos, idx);
  }
  SF_LAUNCH_CHECK("build_slot_lists");
  SF_CHECK(hipStreamSynchronize(s));
  (void)hipFree(pos);
  (void)hipFree(cursor);
  (void)hipFree(sums);
}

void launch_mark_points(hipStream_t s, int n, const int* ig, unsigned char bit, unsigned char* flags) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_mark_points, sf_grid(n, 256), dim3(256), 0, s, n, ig, bit, flags);
  SF_LAUNCH_CHECK("k_mark_points");
}

}  // namespace sf
