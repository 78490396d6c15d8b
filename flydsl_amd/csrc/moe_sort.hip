// Routing metadata of the MoE GEMMs on the device: top-k expert ids -> rows sorted by expert, each
// expert's rows padded to whole routing blocks (the buffers that moe.h describes; reference
// tests/kernels/test_moe_gemm.py:97-160).  C-ABI: flygemm_moe_sort (include/flygemm.h).
//
// The work is a counting sort of tokens * topk small keys, bound by launches and latency rather
// than by bytes (65536 routes are 0.5 MB), so it is one launch up to kOneLaunchRoutes routes and
// two above.  Every workgroup places one chunk of consecutive routes.  It needs the routes per
// expert in all, for the experts' first rows, and those in front of its chunk.  In one launch it
// counts all routes itself, again in every workgroup; in two, a first kernel counts each chunk into
// a scratch array and the second sums that array's rows.  Inside a workgroup each of the 16 waves
// takes a contiguous sixteenth of the chunk, 64 routes at a time: the lanes holding the same
// expert find each other by one ballot per key bit, their lowest lane takes that many rows from the
// wave's own counter, and a lane's row is its rank among them, so equal keys keep their order
// (a stable sort without a comparison) and no two lanes ever add to one counter at once, however
// skewed the routing is.  Padding rows, block experts and totals are spread over all workgroups.
//
// Measured on MI355X, top-8, graph-timed / in back-to-back calls of moe_sorting from Python: 8 tokens,
// 256 experts 6.9 / 16.5 us against 400 for the calls of the operators it stands in for (about 40 launches and
// two waits for the device); 8192 tokens, 128 experts 17.0 / 21 against 440-460; 65536 tokens, 256 experts
// 25.1 / 25.1 against 578.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/flygemm.h"
#include "abi_error.h"

using namespace flygemm;

namespace {

constexpr int kThreads = 1024, kWaves = kThreads / 64;
constexpr int kMaxExperts = FLYGEMM_MOE_SORT_MAX_EXPERTS;
static_assert(kMaxExperts <= kThreads && kMaxExperts % 64 == 0, "one thread per expert in the scans");
// routes per workgroup, one launch / two
constexpr int kChunkOne = 1024, kChunkTwo = 4096;
// Routes up to which every workgroup counts all of them (one launch).  Graph-timed on MI355X: one
// launch 6.9 us at 64 routes, 8.4 at 4096, 11.5 at 8192 and 16.9 at 16384, as much as two launches take
// from 8200 routes (16.7) to 65536 (17.0, 18.5 with 256 experts); the extra launch also costs the
// host 2.5 us.
constexpr int kOneLaunchRoutes = 8192;

struct SortArgs {
  const void* ids;        // [routes] int32 or int64
  const float* weights;   // [routes]
  const uint8_t* mask;    // [experts], 0 = the expert's routes are dropped; may be null
  int32_t* scratch;       // [chunks][experts] counts (two launches) or null
  int32_t* out_ids;
  float* out_weights;
  int32_t* out_eids;
  int32_t* out_post;
  long routes, max_pad;
  int tokens, topk, experts, block, max_blocks, chunk, ids64;
};

// the expert of route r, or E where the route is dropped or r is past the end
__device__ __forceinline__ int route_key(const SortArgs& p, long r, long end) {
  if (r >= end) return p.experts;
  const int64_t v = p.ids64 ? ((const int64_t*)p.ids)[r] : (int64_t)((const int32_t*)p.ids)[r];
  if (v < 0 || v >= p.experts) return p.experts;
  return p.mask && !p.mask[v] ? p.experts : (int)v;
}

// lanes of this wave that hold the same key (every lane is active)
__device__ __forceinline__ uint64_t same_key(int key, int nbits) {
  uint64_t m = ~0ull;
  for (int b = 0; b < nbits; ++b) {
    const bool one = (key >> b) & 1;
    const uint64_t bal = __builtin_amdgcn_ballot_w64(one);
    m &= one ? bal : ~bal;
  }
  return m;
}

__device__ __forceinline__ uint64_t lanes_below(int lane) { return (1ull << lane) - 1; }

// Inclusive sum over the workgroup's threads; `part` holds one value per wave.
__device__ __forceinline__ int block_scan(int v, int* part) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int off = 1; off < 64; off <<= 1) {
    const int u = __shfl_up(v, off, 64);
    if (lane >= off) v += u;
  }
  __syncthreads();
  if (lane == 63) part[wave] = v;
  __syncthreads();
  for (int w = 0; w < wave; ++w) v += part[w];
  return v;
}

// two launches, the first: routes per expert of each chunk
__global__ void __launch_bounds__(kThreads) moe_sort_count_kernel(SortArgs p) {
  __shared__ int cnt[kMaxExperts];
  const int tid = threadIdx.x, lane = tid & 63, E = p.experts, nbits = 32 - __builtin_clz(E);
  if (tid < E) cnt[tid] = 0;
  __syncthreads();
  const long c0 = (long)blockIdx.x * p.chunk, c1 = min(c0 + p.chunk, p.routes);
  for (long r0 = c0; r0 < c1; r0 += kThreads) {
    const int key = route_key(p, r0 + tid, c1);
    const uint64_t m = same_key(key, nbits);
    if (key < E && (m & lanes_below(lane)) == 0) atomicAdd(&cnt[key], __builtin_popcountll(m));
  }
  __syncthreads();
  if (tid < E) p.scratch[(long)blockIdx.x * E + tid] = cnt[tid];
}

__global__ void __launch_bounds__(kThreads) moe_sort_place_kernel(SortArgs p) {
  __shared__ int tot[kMaxExperts], before[kMaxExperts];   // routes in all / in front of this chunk
  __shared__ int start[kMaxExperts], end[kMaxExperts];    // first row, and first row past the padding
  __shared__ int local[kMaxExperts];                      // expert id after the mask's renumbering
  __shared__ int next[kWaves][kMaxExperts];               // next row of each (wave, expert)
  __shared__ int part[kWaves];
  const int tid = threadIdx.x, lane = tid & 63, E = p.experts, nbits = 32 - __builtin_clz(E);
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long c0 = (long)blockIdx.x * p.chunk, c1 = min(c0 + p.chunk, p.routes);
  const long per = p.chunk / kWaves;                      // consecutive routes of one wave
  if (tid < E) tot[tid] = before[tid] = 0;
  for (int i = tid; i < kWaves * E; i += kThreads) next[i / E][i % E] = 0;
  __syncthreads();
  if (p.scratch) {
    const int chunks = (int)((p.routes + p.chunk - 1) / p.chunk);
    if (tid < E) {
      int t = 0, b = 0;
#pragma unroll 8
      for (int c = 0; c < chunks; ++c) {
        const int v = p.scratch[(long)c * E + tid];
        t += v;
        b += c < (int)blockIdx.x ? v : 0;
      }
      tot[tid] = t;
      before[tid] = b;
    }
  } else {
#pragma unroll 4
    for (long r0 = 0; r0 < p.routes; r0 += kThreads) {
      const int key = route_key(p, r0 + tid, p.routes);
      const uint64_t m = same_key(key, nbits);
      if (key < E && (m & lanes_below(lane)) == 0) {
        const int n = __builtin_popcountll(m);
        atomicAdd(&tot[key], n);
        if (r0 < c0) atomicAdd(&before[key], n);          // chunks are whole multiples of kThreads
      }
    }
  }
  // this chunk's routes per (wave, expert)
  const long w0 = c0 + wave * per, w1 = min(w0 + per, c1);
  for (long r0 = w0; r0 < w1; r0 += 64) {
    const int key = route_key(p, r0 + lane, w1);
    const uint64_t m = same_key(key, nbits);
    if (key < E && (m & lanes_below(lane)) == 0) atomicAdd(&next[wave][key], __builtin_popcountll(m));
  }
  __syncthreads();
  // the experts' first rows, and their ids among the experts kept
  const int cnt = tid < E ? tot[tid] : 0;
  const int padded = (cnt + p.block - 1) / p.block * p.block;
  const int stop = block_scan(padded, part);
  const int kept = p.mask ? block_scan(tid < E && p.mask[tid] ? 1 : 0, part) - 1 : tid;
  if (tid < E) {
    start[tid] = stop - padded;
    end[tid] = stop;
    local[tid] = kept;
    int row = stop - padded + before[tid];
    for (int w = 0; w < kWaves; ++w) {
      const int n = next[w][tid];
      next[w][tid] = row;
      row += n;
    }
  }
  __syncthreads();
  const int total = end[E - 1];
  for (long r0 = w0; r0 < w1; r0 += 64) {
    const long r = r0 + lane;
    const int key = route_key(p, r, w1);
    const uint64_t m = same_key(key, nbits);
    const int lead = __builtin_ctzll(m);
    int row = 0;
    if (key < E && lane == lead) row = atomicAdd(&next[wave][key], __builtin_popcountll(m));
    row = __shfl(row, lead, 64) + __builtin_popcountll(m & lanes_below(lane));
    if (key < E && row < p.max_pad) {
      const uint32_t t = (uint32_t)r / (uint32_t)p.topk, s = (uint32_t)r - t * (uint32_t)p.topk;   // routes < 2^31
      p.out_ids[row] = (int32_t)((s << 24) | t);
      p.out_weights[row] = p.weights[r];
    }
  }
  // what no route fills: each expert's last block, and the rows past the last expert
  const int32_t pad = (int32_t)(((uint32_t)p.topk << 24) | (uint32_t)p.tokens);
  const long g0 = (long)blockIdx.x * kThreads + tid, gn = (long)gridDim.x * kThreads;
  for (long i = g0; i < (long)E * p.block; i += gn) {
    const int e = (int)((uint32_t)i / (uint32_t)p.block);
    const long row = start[e] + tot[e] + (i - (long)e * p.block);
    if (row < end[e] && row < p.max_pad) {
      p.out_ids[row] = pad;
      p.out_weights[row] = 0.f;
    }
  }
  for (long row = total + g0; row < p.max_pad; row += gn) {
    p.out_ids[row] = pad;
    p.out_weights[row] = 0.f;
  }
  // the expert of each block: the first whose rows end past the block's first row
  for (long b = g0; b < p.max_blocks; b += gn) {
    const long row = b * p.block;
    int32_t e = -1;
    if (row < total) {
      int lo = 0, hi = E - 1;
      while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (end[mid] > row)
          hi = mid;
        else
          lo = mid + 1;
      }
      e = local[lo];
    }
    p.out_eids[b] = e;
  }
  if (blockIdx.x == 0 && tid == 0) {
    p.out_post[0] = total;
    p.out_post[1] = p.tokens;
  }
}

long sort_chunks(long routes) {
  const int chunk = routes <= kOneLaunchRoutes ? kChunkOne : kChunkTwo;
  return (routes + chunk - 1) / chunk;
}

}  // namespace

extern "C" {

int32_t flygemm_moe_sort_scratch(int32_t tokens, int32_t topk, int32_t experts) {
  const long routes = (long)tokens * topk;
  if (tokens <= 0 || topk <= 0 || experts <= 0 || routes <= kOneLaunchRoutes) return 0;
  const long n = sort_chunks(routes) * experts;
  return n < (1L << 31) ? (int32_t)n : -1;
}

int flygemm_moe_sort(int32_t* sorted_ids, float* sorted_weights, int32_t* sorted_expert_ids, int32_t* num_post_pad,
                     int32_t* scratch, const void* topk_ids, const float* topk_weights, const uint8_t* expert_mask,
                     int32_t tokens, int32_t topk, int32_t experts, int32_t block, int32_t ids_64bit, void* stream) {
  const char* what = "moe_sort";
  if (tokens < 1 || topk < 1 || experts < 1 || block < 1)
    return fail(hipErrorInvalidValue, "%s: invalid sizes tokens=%d topk=%d experts=%d block=%d", what, tokens, topk,
                experts, block);
  if (experts > kMaxExperts)
    return fail(hipErrorInvalidValue, "%s: experts=%d must be at most %d", what, experts, kMaxExperts);
  if (topk > experts) return fail(hipErrorInvalidValue, "%s: topk=%d above experts=%d", what, topk, experts);
  const long routes = (long)tokens * topk;
  const long max_pad = routes + (long)experts * block - topk;
  if (max_pad >= (1L << 31) - (1 << 16))
    return fail(hipErrorInvalidValue, "%s: %ld sorted rows do not fit 32 bits", what, max_pad);
  if (!sorted_ids || !sorted_weights || !sorted_expert_ids || !num_post_pad || !topk_ids || !topk_weights)
    return fail(hipErrorInvalidValue, "%s: null tensor pointer", what);
  const bool two = routes > kOneLaunchRoutes;
  if (two && !scratch) return fail(hipErrorInvalidValue, "%s: null scratch", what);
  SortArgs a{topk_ids, topk_weights, expert_mask, two ? scratch : nullptr, sorted_ids, sorted_weights,
             sorted_expert_ids, num_post_pad, routes, max_pad, tokens, topk, experts, block,
             (int)((max_pad + block - 1) / block), two ? kChunkTwo : kChunkOne, ids_64bit ? 1 : 0};
  const long chunks = sort_chunks(routes);
  // few routes over many experts: more workgroups than chunks, for the padding rows
  const long fill = ((long)experts * block + 4 * kThreads - 1) / (4 * kThreads);
  long grid = chunks > fill ? chunks : fill;
  if (grid > 65535 && chunks <= 65535) grid = 65535;
  hipStream_t s = (hipStream_t)stream;
  if (two) {
    hipLaunchKernelGGL(moe_sort_count_kernel, dim3((unsigned)chunks), dim3(kThreads), 0, s, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(e, "launch of %s (count) failed: %s", what, hipGetErrorString(e));
  }
  hipLaunchKernelGGL(moe_sort_place_kernel, dim3((unsigned)grid), dim3(kThreads), 0, s, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(e, "launch of %s failed: %s", what, hipGetErrorString(e));
  return 0;
}

}  // extern "C"
