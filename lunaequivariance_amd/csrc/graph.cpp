// Graph tables of the convolution on the GPU (the work of the reference's
// one-pass topology kernel, src/lunatp/utils/graph.py:142-846, and of
// make_graph / make_source_segments, src/lunatp/graph.py:49-141 and
// src/lunatp/uvu_conv/graph.py:38-99), as a short pipeline of integer
// kernels:
//   * one pass over the edges: validation (min, max, dst sorted), int32 copies,
//     edge ids;
//   * edge ids by source: stable LSD radix sort of (src, edge id), 8-bit digits
//     (count per 2048-element tile, scan per digit, stable scatter);
//   * CSR row pointers by binary search in dst and in the sorted src (counting
//     the sources with atomics took 45 us more: 1M scattered 4-byte atomics);
//   * segment counts and largest degrees;
//   * node orders: the same sort on keys (largest degree - degree), ties by node
//     id; both orders and the segments' first sort share their launches;
//   * node tiers: scan of the ordered degrees and a search for E/4, 2E/4, 3E/4;
//   * source segments: max(1, ceil(degree/32)) chunks per node, ordered by
//     descending length, then descending node degree, then segment index.
// The caller may read the validation, the segment count and the largest
// degrees back after the first half (luna_graph_scan), which sizes the sorts of
// the second (luna_graph_finish): degrees below 256 take one digit instead of
// the three that E needs.
//
// Bound: launches, each a few microseconds of latency on tables of a few MB.
// 20,000 nodes and 1.05M edges: 702 us with 4-bit digits (22 sort passes,
// about 110 launches, 190 us of them 64-bit atomics of the validation pass on
// three addresses), 178 us with 24 launches, none above 20 us.
// Every buffer is the caller's; scratch comes from one caller-sized
// workspace.  Kernels are compiled with hipRTC once (code-object cache).
#include <algorithm>
#include <cstdint>
#include <initializer_list>
#include <memory>
#include <string>
#include <vector>

#include "../../include/lunaeq_amd.h"
#include "common.h"

namespace luna {
namespace {

constexpr int kTile = 2048;    // scan: elements per workgroup (256 threads x 8)
constexpr int kSortTile = 2048;  // sort: elements per workgroup (4 waves x 8 x 64)
constexpr int kDigits = 256;   // 8-bit digits
constexpr int kFewTiles = 64;   // scan: up to this many tile sums are added up by every workgroup itself
constexpr int kSegment = 32;   // edges per source segment

const char* kGraphSource = R"(
typedef long long i64;
typedef unsigned int u32;

extern "C" __global__ void luna_graph_bounds_init(i64* status) {
  if (threadIdx.x == 0) {
    status[0] = 0x7fffffffffffffffLL;     // min index
    status[1] = -0x7fffffffffffffffLL - 1;  // max index
    status[2] = 0;                        // dst not sorted
    status[3] = 0;
  }
}

// min / max and the flag of a workgroup of 256, then one set of atomics each
// (per wave they were 24,576 on three addresses for a million edges, 190 us).
__device__ void publish(i64 lo, i64 hi, int unsorted, i64* status) {
  __shared__ i64 los[4], his[4];
  __shared__ int flags[4];
  for (int m = 32; m >= 1; m >>= 1) {
    lo = min(lo, (i64)__shfl_xor(lo, m, 64));
    hi = max(hi, (i64)__shfl_xor(hi, m, 64));
    unsorted |= __shfl_xor(unsorted, m, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    los[threadIdx.x >> 6] = lo;
    his[threadIdx.x >> 6] = hi;
    flags[threadIdx.x >> 6] = unsorted;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    // Most workgroups find the bounds already there.
    lo = min(min(los[0], los[1]), min(los[2], los[3]));
    hi = max(max(his[0], his[1]), max(his[2], his[3]));
    if (lo < __hip_atomic_load(&status[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMin((long long*)&status[0], (long long)lo);
    if (hi > __hip_atomic_load(&status[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMax((long long*)&status[1], (long long)hi);
    if (flags[0] | flags[1] | flags[2] | flags[3]) atomicOr((unsigned long long*)&status[2], 1ULL);
  }
}

// min / max over src and dst, and whether dst descends anywhere.
template <typename T>
__device__ void bounds(const T* src, const T* dst, i64 E, i64* status) {
  i64 lo = 0x7fffffffffffffffLL, hi = -0x7fffffffffffffffLL - 1;
  int unsorted = 0;
  for (i64 i = (i64)blockIdx.x * blockDim.x + threadIdx.x; i < E; i += (i64)gridDim.x * blockDim.x) {
    const i64 s = (i64)src[i], d = (i64)dst[i];
    lo = min(lo, min(s, d));
    hi = max(hi, max(s, d));
    if (i + 1 < E && (i64)dst[i + 1] < d) unsorted = 1;
  }
  publish(lo, hi, unsorted, status);
}
extern "C" __global__ void __launch_bounds__(256) luna_graph_bounds32(const int* src, const int* dst, i64 E,
                                                                      i64* status) {
  bounds(src, dst, E, status);
}
extern "C" __global__ void __launch_bounds__(256) luna_graph_bounds64(const i64* src, const i64* dst, i64 E,
                                                                      i64* status) {
  bounds(src, dst, E, status);
}

// status: min, max, unsorted, segments, largest in- and out-degree, 0, 0.
extern "C" __global__ void luna_graph_scan_init(i64* status) {
  const int i = threadIdx.x;
  if (i < 8) status[i] = i == 0 ? 0x7fffffffffffffffLL : i == 1 ? -0x7fffffffffffffffLL - 1 : 0;
}

// One pass over the edges: bounds, int32 copies, edge ids.
template <typename T>
__device__ void edges(const T* src, const T* dst, i64 E, int* src32, int* dst32, int* ids, i64* status) {
  i64 lo = 0x7fffffffffffffffLL, hi = -0x7fffffffffffffffLL - 1;
  int unsorted = 0;
  #pragma unroll 4
  for (i64 i = (i64)blockIdx.x * 256 + threadIdx.x; i < E; i += (i64)gridDim.x * 256) {
    const i64 s = (i64)src[i], d = (i64)dst[i];
    lo = min(lo, min(s, d));
    hi = max(hi, max(s, d));
    if (i + 1 < E && (i64)dst[i + 1] < d) unsorted = 1;
    src32[i] = (int)s;
    dst32[i] = (int)d;
    ids[i] = (int)i;
  }
  publish(lo, hi, unsorted, status);
}
extern "C" __global__ void __launch_bounds__(256) luna_graph_edges(const void* src, const void* dst, int is64, i64 E,
                                                                   int* src32, int* dst32, int* ids, i64* status) {
  if (is64)
    edges((const i64*)src, (const i64*)dst, E, src32, dst32, ids, status);
  else
    edges((const int*)src, (const int*)dst, E, src32, dst32, ids, status);
}

// rowptr[n] = first index i with keys[i] >= n, for n = 0..N (keys ascending), of
// two lists at once.
extern "C" __global__ void __launch_bounds__(256) luna_graph_rowptr(const int* keys0, const int* keys1, i64 E, int N,
                                                                    int* rowptr0, int* rowptr1) {
  const i64 n = (i64)blockIdx.x * 256 + threadIdx.x;
  if (n > N) return;
  const int* const keys = blockIdx.y ? keys1 : keys0;
  int* const rowptr = blockIdx.y ? rowptr1 : rowptr0;
  i64 lo = 0, hi = E;
  while (lo < hi) {
    const i64 mid = (lo + hi) >> 1;
    if (keys[mid] < n) lo = mid + 1; else hi = mid;
  }
  rowptr[n] = (int)lo;
}

// ---- exclusive scan of int32 (tiles of 2048, block sums scanned recursively)
__device__ int block_exclusive_scan(int v, int* wsum, int* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int inc = v;
  for (int m = 1; m < 64; m <<= 1) {
    const int o = __shfl_up(inc, m, 64);
    if (lane >= m) inc += o;
  }
  if (lane == 63) wsum[wave] = inc;
  __syncthreads();
  int before = 0, all = 0;
  for (int w = 0; w < 4; ++w) {
    before += w < wave ? wsum[w] : 0;
    all += wsum[w];
  }
  __syncthreads();
  *total = all;
  return before + inc - v;
}

// out[i] = exclusive prefix of in within its tile (in[i] = 0 past n_in), for
// i < n_out; sums[tile] = tile total.
extern "C" __global__ void __launch_bounds__(256) luna_graph_scan_tiles(const int* in, i64 n_in, int* out,
                                                                        i64 n_out, int* sums) {
  __shared__ int wsum[4];
  const i64 base = (i64)blockIdx.x * 2048 + threadIdx.x * 8;
  int v[8], s = 0;
  for (int j = 0; j < 8; ++j) {
    v[j] = base + j < n_in ? in[base + j] : 0;
    s += v[j];
  }
  int total;
  int run = block_exclusive_scan(s, wsum, &total);
  for (int j = 0; j < 8; ++j) {
    if (base + j < n_out) out[base + j] = run;
    run += v[j];
  }
  if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// Adds each tile's offset, or the sum of the sums before it (at most 64 of
// them); the last value also goes to *last, if given.
extern "C" __global__ void __launch_bounds__(256) luna_graph_scan_add(int* out, i64 n_out, const int* offsets,
                                                                      const int* sums, i64* last) {
  const i64 i = (i64)blockIdx.x * 256 + threadIdx.x;
  const i64 tile = (i64)blockIdx.x * 256 / 2048;
  int before;
  if (offsets) {
    before = offsets[tile];
  } else {
    const int lane = threadIdx.x & 63;
    before = lane < tile ? sums[lane] : 0;
    for (int m = 32; m >= 1; m >>= 1) before += __shfl_xor(before, m, 64);
  }
  if (i >= n_out) return;
  const int v = out[i] + before;
  out[i] = v;
  if (last && i == n_out - 1) *last = v;
}

// ---- stable LSD radix sort, 8-bit digits, up to three sorts per launch
struct Job {
  const u32* keys;
  const int* vals;  // null: the element index
  u32* keys_out;    // null: not wanted
  int* vals_out;
  int* hist;        // [tiles + 1][256]: counts, then offsets within a digit; last row: totals
  i64 n;
  int tiles;
};
struct Jobs {
  Job job[3];
};

extern "C" __global__ void __launch_bounds__(256) luna_graph_radix_count(Jobs jobs, int shift) {
  const Job& j = jobs.job[blockIdx.y];
  __shared__ int count[256];
  const int t = threadIdx.x;
  if (blockIdx.x >= j.tiles) return;
  count[t] = 0;
  __syncthreads();
  const i64 base = (i64)blockIdx.x * 2048 + t;
  #pragma unroll
  for (int k = 0; k < 8; ++k)
    if (base + k * 256 < j.n) atomicAdd(&count[(j.keys[base + k * 256] >> shift) & 255], 1);
  __syncthreads();
  j.hist[(i64)blockIdx.x * 256 + t] = count[t];
}

// Exclusive scan of one digit's counts over the tiles.
extern "C" __global__ void __launch_bounds__(256) luna_graph_radix_columns(Jobs jobs) {
  const Job& j = jobs.job[blockIdx.y];
  __shared__ int wsum[4];
  int run = 0;
  for (int base = 0; base < j.tiles; base += 256) {
    const int tile = base + threadIdx.x;
    int* const at = j.hist + (i64)tile * 256 + blockIdx.x;
    const int v = tile < j.tiles ? *at : 0;
    int total;
    const int before = block_exclusive_scan(v, wsum, &total);
    if (tile < j.tiles) *at = run + before;
    run += total;
  }
  if (threadIdx.x == 0) j.hist[(i64)j.tiles * 256 + blockIdx.x] = run;
}

// Scatter of one tile, in order: a wave owns 512 consecutive elements, 64 at a
// time; equal digits of the 64 find each other by eight ballots.
extern "C" __global__ void __launch_bounds__(256) luna_graph_radix_scatter(Jobs jobs, int shift) {
  const Job& j = jobs.job[blockIdx.y];
  __shared__ int at[4][256];
  __shared__ int wsum[4];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  if (blockIdx.x >= j.tiles) return;
  for (int w = 0; w < 4; ++w) at[w][t] = 0;
  __syncthreads();
  const i64 base = (i64)blockIdx.x * 2048 + wave * 512 + lane;
  u32 key[8];
  #pragma unroll
  for (int k = 0; k < 8; ++k) {
    key[k] = base + k * 64 < j.n ? j.keys[base + k * 64] : 0u;
    if (base + k * 64 < j.n) atomicAdd(&at[wave][(key[k] >> shift) & 255], 1);
  }
  int unused;
  const int first = block_exclusive_scan(j.hist[(i64)j.tiles * 256 + t], wsum, &unused);
  __syncthreads();
  int run = first + j.hist[(i64)blockIdx.x * 256 + t];
  for (int w = 0; w < 4; ++w) {
    const int c = at[w][t];
    at[w][t] = run;
    run += c;
  }
  __syncthreads();
  volatile int* const mine = at[wave];
  #pragma unroll
  for (int k = 0; k < 8; ++k) {
    const i64 i = base + k * 64;
    const bool real = i < j.n;
    const int d = (key[k] >> shift) & 255;
    unsigned long long same = __ballot(real);
    #pragma unroll
    for (int b = 0; b < 8; ++b) {
      const unsigned long long set = __ballot((d >> b) & 1);
      same &= (d >> b) & 1 ? set : ~set;
    }
    const int rank = __popcll(same & ((1ULL << lane) - 1));
    const int pos = mine[d] + rank;
    __builtin_amdgcn_wave_barrier();
    if (real && (same >> lane) == 1ULL) mine[d] = pos + 1;
    __builtin_amdgcn_wave_barrier();
    if (real) {
      if (j.keys_out) j.keys_out[pos] = key[k];
      j.vals_out[pos] = j.vals ? j.vals[i] : (int)i;
    }
  }
}

// Keys of the two node orders, and the nodes' segments with their degree keys.
extern "C" __global__ void __launch_bounds__(256) luna_graph_node_keys(const int* dst_rowptr, const int* src_rowptr,
                                                                       const int* seg_rowptr, int N, int most,
                                                                       u32* in_key, u32* out_key, int* nodes,
                                                                       int* begin, int* end, u32* seg_key) {
  const int n = blockIdx.x * 256 + threadIdx.x;
  if (n >= N) return;
  const int r0 = src_rowptr[n], r1 = src_rowptr[n + 1];
  in_key[n] = (u32)(most - (dst_rowptr[n + 1] - dst_rowptr[n]));
  out_key[n] = (u32)(most - (r1 - r0));
  for (int s = seg_rowptr[n], k = 0; s < seg_rowptr[n + 1]; ++s, ++k) {
    nodes[s] = n;
    // (what is left, not positions: past the last edge they wrap near 2^31 edges)
    const int b = r0 + 32 * k;
    begin[s] = b;
    end[s] = r1 - b > 32 ? b + 32 : r1;
    seg_key[s] = (u32)(most - (r1 - r0));
  }
}

// Past the real segments (seg_rowptr[N] of them): empty ranges whose keys sort
// after all others.
extern "C" __global__ void __launch_bounds__(256) luna_graph_segment_padding(const int* seg_rowptr, int N, i64 S,
                                                                            int most, int* begin, int* end,
                                                                            u32* seg_key) {
  const i64 s = (i64)blockIdx.x * 256 + threadIdx.x;
  if (s < S && s >= seg_rowptr[N]) {
    begin[s] = 1;
    end[s] = 0;
    seg_key[s] = (u32)most + 1u;
  }
}

// Length keys in the order of the degree sort (padding: 33, after every real one).
extern "C" __global__ void __launch_bounds__(256) luna_graph_length_keys(const int* order, const int* begin,
                                                                         const int* end, i64 S, u32* keys) {
  const i64 i = (i64)blockIdx.x * 256 + threadIdx.x;
  if (i < S) keys[i] = (u32)(32 - (end[order[i]] - begin[order[i]]));
}

// node_tiers[t-1] = (first i with cum[i] >= t*E/4) + 1, cum = inclusive scan of
// the degrees in node order (ex = its exclusive scan, ex[N] = E).
extern "C" __global__ void __launch_bounds__(256) luna_graph_tiers(const int* ex, int N, i64 E, int* tiers) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (E == 0 || N == 0) {
    if (i < 3) tiers[i] = N;
    return;
  }
  if (i >= N) return;
  const i64 lo = ex[i], hi = ex[i + 1];
  for (int q = 1; q <= 3; ++q) {
    const i64 thr = q * E / 4;
    if (thr <= hi && (i == 0 || lo < thr)) tiers[q - 1] = i + 1;
  }
}

extern "C" __global__ void __launch_bounds__(256) luna_graph_gather_degree(const int* order, const int* rowptr,
                                                                          int N, int* out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < N) {
    const int n = order[i];
    out[i] = rowptr[n + 1] - rowptr[n];
  }
}

// Segments per node, max(1, ceil(out-degree / 32)), and the largest degrees.
extern "C" __global__ void __launch_bounds__(256) luna_graph_segment_counts(const int* dst_rowptr, const int* src_rowptr,
                                                                            int N, int* count, i64* status) {
  const int n = blockIdx.x * 256 + threadIdx.x;
  int in = 0, out = 0;
  if (n < N) {
    in = dst_rowptr[n + 1] - dst_rowptr[n];
    out = src_rowptr[n + 1] - src_rowptr[n];
    count[n] = out > 0 ? (out - 1) / 32 + 1 : 1;
  }
  for (int m = 32; m >= 1; m >>= 1) {
    in = max(in, __shfl_xor(in, m, 64));
    out = max(out, __shfl_xor(out, m, 64));
  }
  if ((threadIdx.x & 63) == 0) {
    if (in > __hip_atomic_load(&status[4], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMax((long long*)&status[4], (long long)in);
    if (out > __hip_atomic_load(&status[5], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMax((long long*)&status[5], (long long)out);
  }
}
)";

struct GraphKernels {
  ModuleCache kernels;
  GraphKernels() { kernels.tag = "graph"; }
};

// Never destroyed: unloading modules after main would call a HIP runtime that is
// being taken down.
GraphKernels& graph_kernels() {
  static GraphKernels* const g = new GraphKernels;
  return *g;
}

hipModule_t graph_module(const char* cache_dir) {
  GraphKernels& g = graph_kernels();
  if (cache_dir && g.kernels.cache_dir.empty()) g.kernels.cache_dir = cache_dir;
  return g.kernels.module_for("graph", [] { return std::string(kGraphSource); });
}

unsigned blocks_of(int64_t n, int64_t per) { return (unsigned)std::max<int64_t>(1, (n + per - 1) / per); }
int64_t sort_tiles(int64_t n) { return (n + kSortTile - 1) / kSortTile; }
int64_t tiles_of(int64_t n) { return (n + kTile - 1) / kTile; }
size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

// Bump allocator over the caller's workspace.
// Scratch is taken and released in stack order; `peak` sizes the workspace.
struct Arena {
  char* base;
  size_t size, used = 0, peak = 0;
  template <typename T>
  T* take(int64_t count) {
    const size_t bytes = align256((size_t)std::max<int64_t>(count, 1) * sizeof(T));
    if (base && used + bytes > size) fail("luna_graph_build: workspace too small");
    T* p = base ? (T*)(base + used) : nullptr;
    used += bytes;
    peak = std::max(peak, used);
    return p;
  }
};

// The kernels' Job and Jobs.
struct GraphJob {
  const uint32_t* keys;
  const int* vals;
  uint32_t* keys_out;
  int* vals_out;
  int* hist;
  int64_t n;
  int tiles;
};
struct GraphJobs {
  GraphJob job[3];
};

struct Builder {
  hipModule_t module;
  hipStream_t stream;
  Arena& arena;

  void run(const char* name, dim3 grid, void** args) {
    launch(std::string("graph_") + name, function_for(module, std::string("luna_graph_") + name), grid, dim3(256),
           stream, args);
  }

  // out[0..n_out) = exclusive scan of in[0..n_in) (zero past n_in); out[n_out - 1] also in *last.
  void scan(const int* in, int64_t n_in, int* out, int64_t n_out, int64_t* last = nullptr) {
    if (n_out <= 0) return;
    const size_t mark = arena.used;
    const int64_t tiles = tiles_of(n_out);
    int* sums = arena.take<int>(tiles);
    int* offsets = tiles > kFewTiles ? arena.take<int>(tiles) : nullptr;
    if (module) {
      void* a[] = {&in, &n_in, &out, &n_out, &sums};
      run("scan_tiles", blocks_of(n_out, kTile), a);
    }
    if (tiles > kFewTiles) scan(sums, tiles, offsets, tiles);
    if (module && (tiles > 1 || last)) {
      void* b[] = {&out, &n_out, &offsets, &sums, &last};
      run("scan_add", blocks_of(n_out, 256), b);
    }
    arena.used = mark;
  }

  struct Sort {
    uint32_t* keys;      // consumed
    const int* vals;     // null: the element index
    int64_t n;
    int* vals_out;
    uint32_t* keys_out = nullptr;  // the sorted keys, if wanted
  };

  // Stable sorts (up to three in each launch) by the low `bits` of the keys, in
  // 8-bit digits; at least one digit, so that vals_out is always written.
  void sort(std::initializer_list<Sort> sorts, int bits) {
    const size_t mark = arena.used;
    const int passes = std::max(1, (bits + 7) / 8);
    struct Buffers {
      uint32_t* keys[2];
      int *vals, *hist;
    };
    std::vector<Buffers> bufs;
    unsigned most = 0;
    for (const Sort& q : sorts) {
      const int64_t tiles = sort_tiles(q.n);
      Buffers f;
      f.keys[0] = arena.take<uint32_t>(passes > 1 ? q.n : 0);
      f.keys[1] = arena.take<uint32_t>(passes > 2 ? q.n : 0);
      f.vals = arena.take<int>(passes > 1 ? q.n : 0);
      f.hist = arena.take<int>((tiles + 1) * kDigits);
      bufs.push_back(f);
      most = std::max(most, (unsigned)tiles);
    }
    if (module && most) {
      for (int p = 0; p < passes; ++p) {
        GraphJobs jobs{};
        int n = 0;
        for (const Sort& q : sorts) {
          const Buffers& f = bufs[n];
          GraphJob& j = jobs.job[n++];
          // The last pass writes vals_out, those before it alternate; the input
          // buffer of keys is free once pass 0 has read it.
          const int left = passes - 1 - p;
          j.keys = p == 0 ? q.keys : f.keys[(p - 1) % 2];
          j.keys_out = left ? f.keys[p % 2] : q.keys_out;
          j.vals_out = left % 2 ? f.vals : q.vals_out;
          j.vals = p == 0 ? q.vals : ((left + 1) % 2 ? f.vals : q.vals_out);
          j.hist = f.hist;
          j.n = q.n;
          j.tiles = (int)sort_tiles(q.n);
        }
        int shift = 8 * p;
        void* a[] = {&jobs, &shift};
        run("radix_count", dim3(most, (unsigned)n), a);
        void* c[] = {&jobs};
        run("radix_columns", dim3(kDigits, (unsigned)n), c);
        run("radix_scatter", dim3(most, (unsigned)n), a);
      }
    }
    arena.used = mark;
  }
};

int bits_for(int64_t max_key) {
  int b = 0;
  while (b < 32 && (max_key >> b) != 0) ++b;
  return b;
}

struct Outputs {
  int32_t *src32, *dst32, *dst_rowptr, *src_rowptr, *edge_ids_by_src, *edge_ids_by_dst, *node_order,
      *source_node_order, *node_tiers, *seg_rowptr, *seg_nodes, *seg_begin, *seg_end, *seg_order;
};

// A call with module == null sizes the workspace; with one it launches.

// Tables known before any sort, and status = min, max, unsorted, segments,
// largest in- and out-degree, 0, 0.
// Any indices sort and search without fault, so the caller may read the
// validation after all of it.
void scan_half(hipModule_t module, hipStream_t stream, Arena& arena, const void* src, const void* dst, int is64,
               int64_t N, int64_t E, Outputs o, int64_t* status) {
  Builder b{module, stream, arena};
  uint32_t* sorted = arena.take<uint32_t>(E);
  int* count = arena.take<int>(N);
  int Ni = (int)N;
  if (module) {
    void* a[] = {&status};
    b.run("scan_init", dim3(1), a);
    if (E > 0) {
      void* c[] = {(void*)&src, (void*)&dst, &is64, &E, &o.src32, &o.dst32, &o.edge_ids_by_dst, &status};
      b.run("edges", (unsigned)std::min<int64_t>(1024, (E + 255) / 256), c);
    }
  }
  if (E > 0)
    b.sort({{(uint32_t*)o.src32, nullptr, E, o.edge_ids_by_src, sorted}}, bits_for(N > 0 ? N - 1 : 0));
  if (module) {
    void* r[] = {&o.dst32, &sorted, &E, &Ni, &o.dst_rowptr, &o.src_rowptr};
    b.run("rowptr", dim3(blocks_of(N + 1, 256), 2), r);
  }
  if (module && N > 0) {
    void* a[] = {&o.dst_rowptr, &o.src_rowptr, &Ni, &count, &status};
    b.run("segment_counts", blocks_of(N, 256), a);
  }
  b.scan(count, N, o.seg_rowptr, N + 1, status ? status + 3 : nullptr);
}

// Node orders, tiers and segments.  `most`: a bound of every degree; segments:
// their number, or -1 to sort the upper bound N + E/32 + 1 with padding keys
// past the real ones (then the tables must have room for it).
void node_half(hipModule_t module, hipStream_t stream, Arena& arena, int64_t N, int64_t E, int64_t most64,
               int64_t segments, Outputs o) {
  Builder b{module, stream, arena};
  const int64_t S = N == 0 ? 0 : segments >= 0 ? segments : N + E / kSegment + 1;
  uint32_t* in_key = arena.take<uint32_t>(N);
  uint32_t* out_key = arena.take<uint32_t>(N);
  uint32_t* seg_key = arena.take<uint32_t>(S);
  int* perm = arena.take<int>(S);
  int* work = arena.take<int>(N + 1);
  int* degrees = arena.take<int>(N);
  int Ni = (int)N, most = (int)most64;
  if (module && N > 0) {
    void* a[] = {&o.dst_rowptr, &o.src_rowptr, &o.seg_rowptr, &Ni, &most, &in_key, &out_key,
                 &o.seg_nodes, &o.seg_begin, &o.seg_end, &seg_key};
    b.run("node_keys", blocks_of(N, 256), a);
    if (segments < 0) {
      void* p[] = {&o.seg_rowptr, &Ni, (void*)&S, &most, &o.seg_begin, &o.seg_end, &seg_key};
      b.run("segment_padding", blocks_of(S, 256), p);
    }
  }
  if (N > 0) {
    b.sort({{in_key, nullptr, N, o.node_order}, {out_key, nullptr, N, o.source_node_order}, {seg_key, nullptr, S, perm}},
           bits_for(most64 + (segments < 0)));
    if (module) {
      void* a[] = {&perm, &o.seg_begin, &o.seg_end, (void*)&S, &seg_key};
      b.run("length_keys", blocks_of(S, 256), a);
    }
    b.sort({{seg_key, perm, S, o.seg_order}}, 6);
  }
  if (module && N > 0) {
    void* a[] = {&o.node_order, &o.dst_rowptr, &Ni, &degrees};
    b.run("gather_degree", blocks_of(N, 256), a);
  }
  b.scan(degrees, N, work, N + 1);
  if (module) {
    void* a[] = {&work, &Ni, &E, &o.node_tiers};
    b.run("tiers", blocks_of(std::max<int64_t>(N, 3), 256), a);
  }
}

// The halves use the workspace one after the other (and nothing of an earlier
// one), behind the status words.
void build(hipModule_t module, hipStream_t stream, Arena& arena, const void* src, const void* dst, int is64,
           int64_t N, int64_t E, Outputs o) {
  int64_t* status = arena.take<int64_t>(8);
  const size_t mark = arena.used;
  scan_half(module, stream, arena, src, dst, is64, N, E, o, status);
  arena.used = mark;
  node_half(module, stream, arena, N, E, E, -1, o);
}

size_t workspace_bytes_of(int64_t N, int64_t E) {
  Arena arena{nullptr, 0};
  build(nullptr, nullptr, arena, nullptr, nullptr, 0, N, E, Outputs{});
  return arena.peak;
}

void check_graph(int64_t N, int64_t E, const char* what) {
  if (N < 0 || E < 0) fail(std::string(what) + ": negative size");
  if (N >= (1LL << 31) || E >= (1LL << 31) - 1) fail("graph exceeds int32 indexing");
}

}  // namespace
}  // namespace luna

using namespace luna;

extern "C" {

int luna_graph_bounds(const void* src, const void* dst, int index_bits, int64_t num_edges, int64_t* status,
                      LunaStream stream) {
  return guard_call([&] {
    if (index_bits != 32 && index_bits != 64) fail("luna_graph_bounds: index_bits must be 32 or 64");
    if (num_edges < 0) fail("luna_graph_bounds: negative edge count");
    if (!status || (num_edges > 0 && (!src || !dst))) fail("luna_graph_bounds: null argument");
    hipModule_t module = graph_module(nullptr);
    hipStream_t s = (hipStream_t)stream;
    void* a[] = {&status};
    launch("graph_bounds_init", function_for(module, "luna_graph_bounds_init"), dim3(1), dim3(64), s, a);
    if (num_edges > 0) {
      void* b[] = {(void*)&src, (void*)&dst, &num_edges, &status};
      const unsigned grid = (unsigned)std::min<int64_t>(512, (num_edges + 255) / 256);
      launch("graph_bounds", function_for(module, index_bits == 64 ? "luna_graph_bounds64" : "luna_graph_bounds32"),
             dim3(grid), dim3(256), s, b);
    }
  });
}

int luna_graph_workspace(int64_t num_nodes, int64_t num_edges, size_t* bytes) {
  return guard_call([&] {
    if (!bytes) fail("luna_graph_workspace: null argument");
    check_graph(num_nodes, num_edges, "luna_graph_workspace");
    *bytes = workspace_bytes_of(num_nodes, num_edges);
  });
}

int luna_graph_build(const void* src, const void* dst, int index_bits, int64_t num_nodes, int64_t num_edges,
                     int32_t* src32, int32_t* dst32, int32_t* dst_rowptr, int32_t* src_rowptr,
                     int32_t* edge_ids_by_src, int32_t* edge_ids_by_dst, int32_t* node_order,
                     int32_t* source_node_order, int32_t* node_tiers, int32_t* seg_rowptr, int32_t* seg_nodes,
                     int32_t* seg_begin, int32_t* seg_end, int32_t* seg_order, void* workspace,
                     size_t workspace_bytes, LunaStream stream) {
  return guard_call([&] {
    if (index_bits != 32 && index_bits != 64) fail("luna_graph_build: index_bits must be 32 or 64");
    check_graph(num_nodes, num_edges, "luna_graph_build");
    if (!dst_rowptr || !src_rowptr || !node_tiers || !seg_rowptr) fail("luna_graph_build: null table");
    if (num_edges > 0 && (!src || !dst || !src32 || !dst32 || !edge_ids_by_src || !edge_ids_by_dst))
      fail("luna_graph_build: null edge table");
    if (num_nodes > 0 && (!node_order || !source_node_order || !seg_nodes || !seg_begin || !seg_end || !seg_order))
      fail("luna_graph_build: null node table");
    if (!workspace || workspace_bytes < workspace_bytes_of(num_nodes, num_edges))
      fail("luna_graph_build: workspace too small");
    Arena arena{(char*)workspace, workspace_bytes};
    Outputs o{src32, dst32, dst_rowptr, src_rowptr, edge_ids_by_src, edge_ids_by_dst, node_order,
              source_node_order, node_tiers, seg_rowptr, seg_nodes, seg_begin, seg_end, seg_order};
    build(graph_module(nullptr), (hipStream_t)stream, arena, src, dst, index_bits == 64, num_nodes, num_edges, o);
  });
}

int luna_graph_scan(const void* src, const void* dst, int index_bits, int64_t num_nodes, int64_t num_edges,
                    int32_t* src32, int32_t* dst32, int32_t* dst_rowptr, int32_t* src_rowptr,
                    int32_t* edge_ids_by_src, int32_t* edge_ids_by_dst, int32_t* seg_rowptr, int64_t* status,
                    void* workspace, size_t workspace_bytes, LunaStream stream) {
  return guard_call([&] {
    if (index_bits != 32 && index_bits != 64) fail("luna_graph_scan: index_bits must be 32 or 64");
    check_graph(num_nodes, num_edges, "luna_graph_scan");
    if (!dst_rowptr || !src_rowptr || !seg_rowptr || !status) fail("luna_graph_scan: null table");
    if (num_edges > 0 && (!src || !dst || !src32 || !dst32 || !edge_ids_by_src || !edge_ids_by_dst))
      fail("luna_graph_scan: null edge table");
    if (!workspace || workspace_bytes < workspace_bytes_of(num_nodes, num_edges))
      fail("luna_graph_scan: workspace too small");
    Arena arena{(char*)workspace, workspace_bytes};
    Outputs o{};
    o.src32 = src32, o.dst32 = dst32, o.dst_rowptr = dst_rowptr, o.src_rowptr = src_rowptr;
    o.edge_ids_by_src = edge_ids_by_src, o.edge_ids_by_dst = edge_ids_by_dst, o.seg_rowptr = seg_rowptr;
    scan_half(graph_module(nullptr), (hipStream_t)stream, arena, src, dst, index_bits == 64, num_nodes, num_edges, o,
              status);
  });
}

int luna_graph_finish(const int32_t* dst_rowptr, const int32_t* src_rowptr, const int32_t* seg_rowptr,
                      int64_t num_nodes, int64_t num_edges, int64_t largest_degree, int64_t segments,
                      int32_t* node_order, int32_t* source_node_order, int32_t* node_tiers, int32_t* seg_nodes,
                      int32_t* seg_begin, int32_t* seg_end, int32_t* seg_order, void* workspace,
                      size_t workspace_bytes, LunaStream stream) {
  return guard_call([&] {
    check_graph(num_nodes, num_edges, "luna_graph_finish");
    if (largest_degree < 0 || largest_degree > num_edges || segments < 0 || segments > num_nodes + num_edges / kSegment + 1)
      fail("luna_graph_finish: degree or segment count out of range");
    if (!dst_rowptr || !src_rowptr || !seg_rowptr || !node_tiers) fail("luna_graph_finish: null table");
    if (num_nodes > 0 && (!node_order || !source_node_order || !seg_nodes || !seg_begin || !seg_end || !seg_order))
      fail("luna_graph_finish: null node table");
    if (!workspace || workspace_bytes < workspace_bytes_of(num_nodes, num_edges))
      fail("luna_graph_finish: workspace too small");
    Arena arena{(char*)workspace, workspace_bytes};
    Outputs o{};
    o.dst_rowptr = const_cast<int32_t*>(dst_rowptr), o.src_rowptr = const_cast<int32_t*>(src_rowptr);
    o.seg_rowptr = const_cast<int32_t*>(seg_rowptr), o.node_order = node_order;
    o.source_node_order = source_node_order, o.node_tiers = node_tiers, o.seg_nodes = seg_nodes;
    o.seg_begin = seg_begin, o.seg_end = seg_end, o.seg_order = seg_order;
    node_half(graph_module(nullptr), (hipStream_t)stream, arena, num_nodes, num_edges, largest_degree, segments, o);
  });
}

int luna_graph_precompile(const char* cache_dir) {
  return guard_call([&] {
    GraphKernels& g = graph_kernels();
    if (cache_dir && g.kernels.cache_dir.empty()) g.kernels.cache_dir = cache_dir;
    g.kernels.code_for("graph", [] { return std::string(kGraphSource); });
  });
}

}  // extern "C"
