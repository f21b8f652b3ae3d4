// Shared-weight contraction of aggregated uvw products on CDNA4 matrix cores
// (fp32 and fp64).
//
// The UVW convolution with shared weights is an aggregation A[n] of the
// Clebsch-Gordan products over edges (the UVU kernels) followed, per output
// block o, by a contraction over the block's channels c = (path, v, u):
//   out[n, oo + m*d3 + k] = sum_c A[n, ao + c*d3 + k] W[row(c) + m]
// with row(c) the start of weight row (u, v) of c's path in the e3nn layout
// (m contiguous).  Its two derivatives are contractions of the same operands:
//   gA[n, ao + c*d3 + k]  = sum_m g[n, oo + m*d3 + k] W[row(c) + m]
//   gW[row(c) + m]        = sum_{n,k} A[n, ao + c*d3 + k] g[n, oo + m*d3 + k]
// All three read and write the convolution's own layouts (component fastest):
// a tile's columns are the (n, k) pairs of a few rows, whose values are one
// contiguous run per row and channel chunk, so no transposed copy of A or g
// is made.  The three kernels run every output block in one launch.
//
// Bound and shape.  At 64 channels, lmax 3 and 2,083 rows the work is 1.7
// GFLOP on 53 MB of A: 11 us of either.  Measured there 32 us (forward), 42
// us (gA) and 33 + 7 us (gW and its reduction), against about 550 us for the
// library products, layout copies and concatenations they replaced (step 975
// -> 397 us); at 20,011 fp64 rows of 32 channels, lmax 2 (180 MB of A, 38 us)
// 51, 67 and 64 + 18 us (step 1,142 -> 290 us).  The launches are bound by
// latency in the first case (two workgroups per CU) and by the traffic of A
// in the second.  A workgroup of four waves owns a 64 x 64 or 32 x 128 tile
// (half as many columns in fp64, whose 64-bit tiles would halve the
// workgroups per CU), each wave 32 x 32 on v_mfma_f32_32x32x2f32 or 32 x 16 on
// v_mfma_f64_16x16x4f64; operands go through LDS, the next chunk is in
// registers while the current one is multiplied, and results leave through
// LDS as contiguous runs.  Wide products of many rows, where the matrix rate
// counts and these tiles reach about 55 % of it, stay with the library
// (LunaTPUVWConv.contracts_natively).
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <memory>
#include <sstream>

#include "../../include/lunaeq_amd.h"
#include "common.h"

namespace luna {
namespace {

struct CPath {
  int w_off, mul1, mul2;
};

struct CBlock {
  int out_off, a_off, d3, mul3, channels;
  std::vector<CPath> paths;  // in channel order: (path, v, u)
};

struct CPlan {
  int bits = 32, adim = 0, out = 0, wnum = 0;
  std::vector<CBlock> blocks;
  ModuleCache kernels;
};

// Values of a row whose offsets within a tile of up to 128 rows fit 32 bits.
constexpr int kMaxRow = 1 << 23;
// Degrees whose staged tiles fit 64 KB of LDS (4 rows x 160 channels x d3 doubles).
constexpr int kMaxD3 = 11;

int read_int(std::istringstream& in, const char* what) {
  long long value;
  if (!(in >> value)) fail(std::string("contraction spec: expected integer for ") + what);
  if (value < 0 || value > (1LL << 31) - 1) fail(std::string("contraction spec: value out of range for ") + what);
  return (int)value;
}

void parse(CPlan& p, const std::string& text) {
  std::istringstream in(text);
  std::string magic;
  in >> magic;
  if (magic != "LUNACON1") fail("contraction spec: missing LUNACON1 header");
  p.bits = read_int(in, "dtype");
  if (p.bits != 32 && p.bits != 64) fail("contraction spec: dtype must be 32 or 64");
  p.adim = read_int(in, "aggregate_dim");
  p.out = read_int(in, "out_dim");
  p.wnum = read_int(in, "weight_numel");
  if (p.adim > kMaxRow || p.out > kMaxRow) fail("contraction spec: rows of more than 2^23 values are not supported");
  const int nblocks = read_int(in, "blocks");
  for (int n = 0; n < nblocks; ++n) {
    CBlock b;
    b.out_off = read_int(in, "out_off");
    b.a_off = read_int(in, "a_off");
    b.d3 = read_int(in, "d3");
    b.mul3 = read_int(in, "mul3");
    b.channels = 0;
    const int npaths = read_int(in, "paths");
    for (int k = 0; k < npaths; ++k) {
      CPath q;
      q.w_off = read_int(in, "w_off");
      q.mul1 = read_int(in, "mul1");
      q.mul2 = read_int(in, "mul2");
      if (q.mul1 <= 0 || q.mul2 <= 0) fail("contraction spec: positive multiplicities required");
      if ((long)q.w_off + (long)q.mul1 * q.mul2 * b.mul3 > p.wnum)
        fail("contraction spec: weight block outside weight_numel");
      b.channels += q.mul1 * q.mul2;
      b.paths.push_back(q);
    }
    if (b.mul3 <= 0 || b.channels <= 0) fail("contraction spec: empty block");
    if (b.d3 < 1 || b.d3 > kMaxD3 || b.d3 % 2 == 0) fail("contraction spec: output degree above 5 is not supported");
    if ((long)b.out_off + (long)b.mul3 * b.d3 > p.out) fail("contraction spec: output block outside out_dim");
    if ((long)b.a_off + (long)b.channels * b.d3 > p.adim) fail("contraction spec: block outside aggregate_dim");
    p.blocks.push_back(std::move(b));
  }
  if (p.blocks.empty()) fail("contraction spec: no blocks");
}

// Tile shapes.  A 32-wide output side takes 32 x 128 tiles, so that layers of
// up to 32 channels do not multiply padding.
int tile_m(int m) { return m <= 32 ? 32 : 64; }
// Rows of a tile: four waves of 32 x 32 (fp32) or 32 x 16 (fp64) results.
int tile_nodes(int bits, const CBlock& b, int m) {
  return std::max(1, (bits == 64 ? 2048 : 4096) / tile_m(m) / b.d3);
}
// Weight gradient: TC channels x TW output channels.
int grad_tw(const CBlock& b) { return b.mul3 <= 32 ? 32 : 64; }
int grad_tc(const CBlock& b) { return 4096 / grad_tw(b); }
// Rows staged at once by the weight gradient: a multiple of the matrix
// instruction's K (2 or 4), about 32 (fp32) or 16 (fp64) (n, k) pairs.
int grad_stage(const CPlan& p, const CBlock& b) {
  const int ks = p.bits == 64 ? 4 : 2, want = p.bits == 64 ? 16 : 32;
  return std::max(ks, want / b.d3 / ks * ks);
}
int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

int64_t grad_tiles(const CBlock& b) {
  return ceil_div(b.channels, grad_tc(b)) * ceil_div(b.mul3, grad_tw(b));
}

// (n, k) pairs per workgroup of the weight gradient: enough workgroups for
// four per CU, but at least 256 pairs each, so that the partial tiles stay
// small beside the operands.
int64_t grad_span(const CPlan& p, int64_t rows) {
  int64_t pairs = 0;
  for (const CBlock& b : p.blocks) pairs += grad_tiles(b) * rows * b.d3;
  return std::max<int64_t>(256, ceil_div(pairs, 1024));
}
int64_t grad_rows(const CPlan& p, const CBlock& b, int64_t span) {
  return ceil_div(ceil_div(span, b.d3), grad_stage(p, b)) * grad_stage(p, b);
}
size_t grad_partials(const CPlan& p, int64_t rows) {
  const int64_t span = grad_span(p, rows);
  size_t total = 0;
  for (const CBlock& b : p.blocks) total += (size_t)ceil_div(rows, grad_rows(p, b, span)) * grad_tiles(b) * 4096;
  return total;
}

const char* kBody = R"(
// D += A B: lane l supplies A[l % T][l / T] and B[l / T][l % T]; value r of
// lane l is D[row_of(r, l / T)][l % T].
#if BITS == 64
typedef double real;
typedef double accv __attribute__((ext_vector_type(4)));
constexpr int T = 16, KS = 4, AV = 4;
__device__ __forceinline__ accv mma(real a, real b, accv c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ constexpr int row_of(int r, int hi) { return 4 * r + hi; }
#else
typedef float real;
typedef float accv __attribute__((ext_vector_type(16)));
constexpr int T = 32, KS = 2, AV = 16;
__device__ __forceinline__ accv mma(real a, real b, accv c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ constexpr int row_of(int r, int hi) { return 8 * (r >> 2) + 4 * hi + (r & 3); }
#endif
typedef long long i64;
constexpr int FR = 32 / T;  // fragments per 32 rows of a wave's tile

// Tiles [mt0, mt1) of TM values of m of out[n, oo + m*D + k] = sum_kk in[n, io + kk*D + k] Wm(kk, m)
// for NB rows (their NB*D columns).  Wm(kk, m) = wt[rows[kk] + m] (forward, KN
// channels to MN outputs), or wt[rows[m] + kk] (SWAP: KN outputs back to MN
// channels).  LDS rows are (KC + 1)*D and (TM + 1)*D apart, which puts
// consecutive columns in consecutive banks.  When the whole K fits one chunk
// the staged rows serve every tile of m.  With LIN the weight rows of a chunk
// (forward) or tile (SWAP) are consecutive, so their addresses need one scalar
// table entry; otherwise the entry of each weight row is a scalar load too, as
// RUN consecutive lanes share a row (read per lane, before every weight load, they
// took longer than the products: 20,000 rows, lmax 3, forward 80 channels 1,767 -> 702
// us, gA and gW 96 channels 3,895 -> 1,466 us).  Offsets are formed once, since fp32
// matrix and vector instructions of a SIMD do not overlap.  Rows past N and m past
// MN repeat the last one: they only reach results that are not stored.  K past KN is
// cleared; the last chunk's loads are skipped (forward, 66 against 107 us at 112
// channels, lmax 1) or repeat another value (SWAP).
template <int D, int KN, int MN, int TM, int KC, bool SWAP, bool LIN>
__device__ __forceinline__ void product_tiles(const real* __restrict__ in, int ldi, const real* __restrict__ wt,
                                              const int* __restrict__ rows, real* __restrict__ out, int ldo, i64 n0,
                                              int mt0, int mt1, i64 N, real* lds) {
  constexpr int COLT = 128 * T / TM, NB = COLT / D > 0 ? COLT / D : 1, COLS = NB * D;
  constexpr int LDI = (KC + 1) * D, LDW = TM + 1, LDO = (TM + 1) * D;
  constexpr int IN_PT = (NB * KC * D + 255) / 256, W_PT = KC * TM / 256;
  constexpr int CHUNKS = (KN + KC - 1) / KC;
  constexpr int RUN = SWAP ? KC : TM, ROWS = SWAP ? MN : KN;  // lanes in a row on one weight row; weight rows
  real* const ins = lds;
  real* const ws = lds + NB * LDI;  // and, after the products, the results
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wm = wave % (TM / 32), wn = wave / (TM / 32);
  const int hi = lane / T, lo = lane % T;
  const int left = N - n0 < NB ? (int)(N - n0) : NB;
  in += n0 * ldi;
  out += n0 * ldo;
  int oi[IN_PT];
  #pragma unroll
  for (int i = 0; i < IN_PT; ++i) {
    const int idx = i * 256 + t, n = idx / (KC * D), e = idx % (KC * D);
    oi[i] = (n < left ? n : left - 1) * ldi + e;
  }
  real rin[IN_PT], rw[W_PT];
  auto fetch_in = [&](int c) {
    #pragma unroll
    for (int i = 0; i < IN_PT; ++i) {
      const int e = (i * 256 + t) % (KC * D);
      const bool ok = KN % KC == 0 || c * KC * D + e < KN * D;
      rin[i] = 0;
      if (SWAP)
        rin[i] = in[oi[i] + (ok ? c * KC * D : -e)];
      else if (ok)
        rin[i] = in[oi[i] + c * KC * D];
    }
  };
  auto fetch_w = [&](int mt, int c) {
    const int m0 = mt * TM, c0 = c * KC;
    const real* const base = wt + (LIN ? (SWAP ? rows[m0] + c0 : rows[c0] + m0) : 0);
    #pragma unroll
    for (int i = 0; i < W_PT; ++i) {
      const int idx = i * 256 + t;
      const int kk = SWAP ? idx % KC : idx / TM, m = SWAP ? idx / KC : idx % TM;
      const int mc = MN % TM == 0 || m0 + m < MN ? m : MN - 1 - m0;
      const int kc = KN % KC == 0 || c0 + kk < KN ? kk : KN - 1 - c0;
      rw[i] = 0;
      if (!SWAP && kc != kk) continue;
      if (LIN) {
        rw[i] = SWAP ? base[mc * KN + kc] : base[kc * MN + mc];
      } else {
        const int first = (SWAP ? m0 : c0) + i * (256 / RUN) + wave * (64 / RUN);
        int row = rows[first < ROWS ? first : ROWS - 1];
        if (RUN < 64) {
          const int other = rows[first + 1 < ROWS ? first + 1 : ROWS - 1];
          row = lane < RUN ? row : other;
        }
        rw[i] = wt[row + (SWAP ? c0 + kc : m0 + mc)];
      }
    }
  };
  const int col = wn * T + lo;  // this lane's column of its wave's 32 x T tile
  const int cb = col < COLS ? (col / D) * LDI + col % D : 0, ca = wm * 32 + lo;
  fetch_in(0);
  fetch_w(mt0, 0);
  for (int mt = mt0; mt < mt1; ++mt) {
    accv acc[FR];
    #pragma unroll
    for (int x = 0; x < FR; ++x) acc[x] = (accv)(0);
    for (int c = 0; c < CHUNKS; ++c) {
      if (CHUNKS > 1 || mt == mt0) {
        #pragma unroll
        for (int i = 0; i < IN_PT; ++i) {
          const int idx = i * 256 + t, n = idx / (KC * D), e = idx % (KC * D);
          if (n < NB) ins[n * LDI + e] = !SWAP || KN % KC == 0 || c * KC * D + e < KN * D ? rin[i] : (real)0;
        }
      }
      #pragma unroll
      for (int i = 0; i < W_PT; ++i) {
        const int idx = i * 256 + t;
        const int kk = SWAP ? idx % KC : idx / TM, m = SWAP ? idx / KC : idx % TM;
        ws[kk * LDW + m] = !SWAP || KN % KC == 0 || c * KC + kk < KN ? rw[i] : (real)0;
      }
      __syncthreads();
      if (c + 1 < CHUNKS) {
        fetch_in(c + 1);
        fetch_w(mt, c + 1);
      } else if (mt + 1 < mt1) {
        if (CHUNKS > 1) fetch_in(0);
        fetch_w(mt + 1, 0);
      }
      #pragma unroll
      for (int s = 0; s < KC; s += KS) {
        const real b = ins[cb + (s + hi) * D];
        #pragma unroll
        for (int x = 0; x < FR; ++x) acc[x] = mma(ws[(s + hi) * LDW + ca + x * T], b, acc[x]);
      }
      __syncthreads();
    }
    if (col < COLS) {
      real* const o = ws + (col / D) * LDO + col % D;
      #pragma unroll
      for (int x = 0; x < FR; ++x)
        #pragma unroll
        for (int r = 0; r < AV; ++r) o[(wm * 32 + x * T + row_of(r, hi)) * D] = acc[x][r];
    }
    __syncthreads();
    const int m0 = mt * TM, width = (MN - m0 < TM ? MN - m0 : TM) * D;
    #pragma unroll 4
    for (int idx = t; idx < left * TM * D; idx += 256) {
      const int n = idx / (TM * D), e = idx % (TM * D);
      if (MN % TM == 0 || e < width) out[n * ldo + m0 * D + e] = ws[n * LDO + e];
    }
    if (mt + 1 < mt1) __syncthreads();
  }
}

// One TC x TW tile of gW over the rows [n0, n1): K = (n, k), taken k by k over
// NS staged rows; the partial tile is stored whole (zeros past the edges).
template <int D, int C, int MN, int TC, int TW, int NS>
__device__ __forceinline__ void grad_tile(const real* __restrict__ a, i64 lda, const real* __restrict__ g, i64 ldg,
                                          real* __restrict__ part, i64 n0, i64 n1, int c0, int w0, real* lds) {
  constexpr int RA = TC * D, RG = TW * D, A_PT = (NS * RA + 255) / 256, G_PT = (NS * RG + 255) / 256;
  real* const as = lds;
  real* const gs = lds + NS * RA;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wc = wave % (TC / 32), ww = wave / (TC / 32);
  const int hi = lane / T, lo = lane % T;
  const int wide_a = (C - c0 < TC ? C - c0 : TC) * D, wide_g = (MN - w0 < TW ? MN - w0 : TW) * D;
  // Whole fp32 tiles test each value's bounds.  Where channels remain, and in fp64,
  // that cost up to a fifth (20,000 rows, lmax 3, gA and gW: 80 channels 1,222 -> 1,082
  // us, 160 channels 3,506 -> 3,013 us; 64 channels 428 us, 461 without the tests): there
  // offsets within a step are formed once, channels past the last repeat it (their
  // results are not stored), rows past the last repeat it and are cleared.
  constexpr bool TESTED = BITS == 32 && C % TC == 0 && MN % TW == 0;
  int oa[A_PT], og[G_PT];
  #pragma unroll
  for (int i = 0; i < A_PT; ++i) {
    const int r = (i * 256 + t) / RA, e = (i * 256 + t) % RA;
    oa[i] = (r < NS ? r : NS - 1) * (int)lda + c0 * D + (e < wide_a ? e : wide_a - 1);
  }
  #pragma unroll
  for (int i = 0; i < G_PT; ++i) {
    const int r = (i * 256 + t) / RG, e = (i * 256 + t) % RG;
    og[i] = (r < NS ? r : NS - 1) * (int)ldg + w0 * D + (e < wide_g ? e : wide_g - 1);
  }
  real ra[A_PT], rg[G_PT];
  auto fetch = [&](i64 n) {
    const real* const an = a + n * lda;
    const real* const gn = g + n * ldg;
    if (TESTED) {
      #pragma unroll
      for (int i = 0; i < A_PT; ++i) {
        const int idx = i * 256 + t, r = idx / RA, e = idx % RA;
        ra[i] = 0;
        if (r < NS && n + r < n1 && e < wide_a) ra[i] = a[(n + r) * lda + c0 * D + e];
      }
      #pragma unroll
      for (int i = 0; i < G_PT; ++i) {
        const int idx = i * 256 + t, r = idx / RG, e = idx % RG;
        rg[i] = 0;
        if (r < NS && n + r < n1 && e < wide_g) rg[i] = g[(n + r) * ldg + w0 * D + e];
      }
    } else if (n + NS <= n1) {
      #pragma unroll
      for (int i = 0; i < A_PT; ++i) ra[i] = an[oa[i]];
      #pragma unroll
      for (int i = 0; i < G_PT; ++i) rg[i] = gn[og[i]];
    } else {
      const int last = (int)(n1 - n) - 1;
      #pragma unroll
      for (int i = 0; i < A_PT; ++i) {
        const int r = (i * 256 + t) / RA, back = r > last ? (r < NS ? r : NS - 1) - last : 0;
        ra[i] = an[oa[i] - back * (int)lda];
        if (back) ra[i] = 0;
      }
      #pragma unroll
      for (int i = 0; i < G_PT; ++i) {
        const int r = (i * 256 + t) / RG, back = r > last ? (r < NS ? r : NS - 1) - last : 0;
        rg[i] = gn[og[i] - back * (int)ldg];
        if (back) rg[i] = 0;
      }
    }
  };
  accv acc[FR][FR];
  #pragma unroll
  for (int x = 0; x < FR; ++x)
    #pragma unroll
    for (int y = 0; y < FR; ++y) acc[x][y] = (accv)(0);
  fetch(n0);
  for (i64 n = n0; n < n1; n += NS) {
    #pragma unroll
    for (int i = 0; i < A_PT; ++i)
      if (i * 256 + t < NS * RA) as[i * 256 + t] = ra[i];
    #pragma unroll
    for (int i = 0; i < G_PT; ++i)
      if (i * 256 + t < NS * RG) gs[i * 256 + t] = rg[i];
    __syncthreads();
    if (n + NS < n1) fetch(n + NS);
    #pragma unroll
    for (int s = 0; s < NS; s += KS) {
      #pragma unroll
      for (int k = 0; k < D; ++k) {
        real av[FR], gv[FR];
        #pragma unroll
        for (int f = 0; f < FR; ++f) {
          av[f] = as[(s + hi) * RA + (wc * 32 + f * T + lo) * D + k];
          gv[f] = gs[(s + hi) * RG + (ww * 32 + f * T + lo) * D + k];
        }
        #pragma unroll
        for (int x = 0; x < FR; ++x)
          #pragma unroll
          for (int y = 0; y < FR; ++y) acc[x][y] = mma(av[x], gv[y], acc[x][y]);
      }
    }
    __syncthreads();
  }
  #pragma unroll
  for (int x = 0; x < FR; ++x)
    #pragma unroll
    for (int r = 0; r < AV; ++r)
      #pragma unroll
      for (int y = 0; y < FR; ++y)
        part[(wc * 32 + x * T + row_of(r, hi)) * TW + ww * 32 + y * T + lo] = acc[x][y][r];
}

// gW of one tile column block: 64 weights per workgroup, four lanes of splits.
template <int C, int MN, int TC, int TW>
__device__ __forceinline__ void reduce_tile(const real* __restrict__ part, const int* __restrict__ rows,
                                            real* __restrict__ gw, i64 tiles, i64 splits, int tile, int at,
                                            real* lds) {
  const int t = threadIdx.x, q = t >> 6, v = at + (t & 63);
  const real* p = part + (i64)tile * 4096 + v;
  real sum = 0;
  #pragma unroll 4
  for (i64 s = q; s < splits; s += 4) sum += p[s * tiles * 4096];
  lds[t] = sum;
  __syncthreads();
  if (q == 0) {
    sum = (lds[t] + lds[64 + t]) + (lds[128 + t] + lds[192 + t]);
    const int c = tile / ((MN + TW - 1) / TW) * TC + v / TW, w = tile % ((MN + TW - 1) / TW) * TW + v % TW;
    if (c < C && w < MN) gw[(i64)rows[c] + w] = sum;
  }
}
)";

std::string fmt(const char* text, std::initializer_list<long long> values) {
  // Replaces each @ in `text` by the next value.
  std::string out;
  auto it = values.begin();
  for (const char* c = text; *c; ++c) {
    if (*c == '@' && it != values.end())
      out += std::to_string(*it++);
    else
      out += *c;
  }
  return out;
}

// Starts of the weight rows of a block's channels.
std::vector<long> weight_rows(const CBlock& b) {
  std::vector<long> rows;
  for (const CPath& q : b.paths)
    for (int v = 0; v < q.mul2; ++v)
      for (int u = 0; u < q.mul1; ++u) rows.push_back(q.w_off + (long)(u * q.mul2 + v) * b.mul3);
  return rows;
}

// True when every run of `n` channels has consecutive weight rows.
bool linear_rows(const CBlock& b, int n) {
  const std::vector<long> rows = weight_rows(b);
  for (size_t c = 0; c < rows.size(); ++c)
    if (rows[c] != rows[c / n * n] + (long)(c % n) * b.mul3) return false;
  return true;
}

// Channels (forward) or outputs (SWAP) per staged chunk: 64 floats or 32
// doubles, half of that where only then a chunk's weight rows are consecutive
// (forward) or less is multiplied past the outputs (SWAP; 160 channels, lmax 3,
// 20,000 rows, gA and gW 3,562 -> 3,006 us).
int product_chunk(const CPlan& p, const CBlock& b, bool swap) {
  if (swap) return p.bits == 32 && (b.mul3 + 63) / 64 * 64 == (b.mul3 + 31) / 32 * 32 ? 64 : 32;
  const int kc = p.bits == 64 ? 32 : 64;
  return !linear_rows(b, kc) && linear_rows(b, kc / 2) ? kc / 2 : kc;
}

int lds_reals(const CPlan& p, bool grad) {
  int most = 256;
  for (const CBlock& b : p.blocks) {
    if (grad) {
      most = std::max(most, grad_stage(p, b) * (grad_tc(b) + grad_tw(b)) * b.d3);
      continue;
    }
    for (bool swap : {false, true}) {
      const int m = swap ? b.channels : b.mul3, kc = product_chunk(p, b, swap), tm = tile_m(m), nb = tile_nodes(p.bits, b, m);
      most = std::max(most, nb * (kc + 1) * b.d3 + std::max(kc, nb * b.d3) * (tm + 1));
    }
  }
  return most;
}

// Tiles of m per workgroup: the staged rows of a one-chunk product serve all
// of them, as long as about three workgroups per CU remain.
int64_t product_tiles(const CPlan& p, const CBlock& b, int64_t rows, bool swap) {
  const int mn = swap ? b.channels : b.mul3;
  return ceil_div(rows, tile_nodes(p.bits, b, mn)) * ceil_div(mn, tile_m(mn));
}
int product_group(const CPlan& p, int64_t rows, bool swap) {
  int64_t total = 0;
  for (const CBlock& b : p.blocks) total += product_tiles(p, b, rows, swap);
  return (int)std::max<int64_t>(1, std::min<int64_t>(8, total / 768));
}

std::string emit(const CPlan& p) {
  std::string s = fmt("#define BITS @\n", {p.bits}) + kBody;
  for (size_t n = 0; n < p.blocks.size(); ++n) {
    const CBlock& b = p.blocks[n];
    s += fmt("__device__ const int rows@[@] = {", {(long long)n, b.channels});
    for (long row : weight_rows(b)) s += std::to_string(row) + ",";
    s += "};\n";
  }
  // Forward and its transpose: the blocks' tiles one after the other over the grid.
  for (int swap = 0; swap < 2; ++swap) {
    s += std::string("extern \"C\" __global__ void __launch_bounds__(256) luna_con_") + (swap ? "ga" : "fwd") +
         "(const real* __restrict__ in, const real* __restrict__ wt, real* __restrict__ out, i64 N, int group) {\n";
    s += fmt("  __shared__ real lds[@];\n  i64 tile = blockIdx.x;\n", {lds_reals(p, false)});
    for (size_t n = 0; n < p.blocks.size(); ++n) {
      const CBlock& b = p.blocks[n];
      const int kn = swap ? b.mul3 : b.channels, mn = swap ? b.channels : b.mul3, tm = tile_m(mn);
      const int kc = product_chunk(p, b, swap), nb = tile_nodes(p.bits, b, mn), lin = linear_rows(b, swap ? tm : kc);
      const long long mt = ceil_div(mn, tm), io = swap ? b.out_off : b.a_off, oo = swap ? b.a_off : b.out_off;
      s += fmt("  { const int per = (@ + group - 1) / group;\n    const i64 nt = (N + @) / @ * per;\n",
               {mt, nb - 1, nb});
      s += fmt("    if (tile < nt) {\n      const i64 nb = tile / per; const int mt = (int)(tile - nb * per) * group;\n"
               "      product_tiles<@, @, @, @, @, @, @>(in + @, @, wt, rows@, out + @, @, nb * @, mt, "
               "mt + group < @ ? mt + group : @, N, lds); return; }\n",
               {b.d3, kn, mn, tm, kc, swap, lin, io, swap ? p.out : p.adim, (long long)n, oo, swap ? p.adim : p.out, nb,
                mt, mt});
      s += "    tile -= nt; }\n";
    }
    s += "}\n";
  }
  s += "extern \"C\" __global__ void __launch_bounds__(256) luna_con_gw(const real* __restrict__ a, "
       "const real* __restrict__ g, real* __restrict__ part, i64 N, i64 span) {\n";
  s += fmt("  __shared__ real lds[@];\n  i64 tile = blockIdx.x;\n", {lds_reals(p, true)});
  for (size_t n = 0; n < p.blocks.size(); ++n) {
    const CBlock& b = p.blocks[n];
    const long long tw = grad_tw(b), tc = grad_tc(b), wt = ceil_div(b.mul3, tw), nt = grad_tiles(b);
    const int ns = grad_stage(p, b);
    s += fmt("  { const i64 per = ((span + @) / @ + @) / @ * @, splits = (N + per - 1) / per;\n",
             {b.d3 - 1, b.d3, ns - 1, ns, ns});
    s += fmt("    if (tile < splits * @) {\n      const i64 sp = tile / @; const int ti = (int)(tile - sp * @);\n",
             {nt, nt, nt});
    s += fmt("      const int tc = ti / @, tw = ti - tc * @;\n", {wt, wt});
    s += fmt("      grad_tile<@, @, @, @, @, @>(a + @, @LL, g + @, @LL, part + tile * 4096, sp * per, "
             "sp * per + per < N ? sp * per + per : N, tc * @, tw * @, lds); return; }\n",
             {b.d3, b.channels, b.mul3, tc, tw, ns, b.a_off, p.adim, b.out_off, p.out, tc, tw});
    s += fmt("    tile -= splits * @; part += splits * @LL; }\n", {nt, nt * 4096});
  }
  s += "}\n";
  s += "extern \"C\" __global__ void __launch_bounds__(256) luna_con_gw_reduce(const real* __restrict__ part, "
       "real* __restrict__ gw, i64 N, i64 span) {\n  __shared__ real lds[256];\n"
       "  int tile = blockIdx.x / 64; const int at = blockIdx.x % 64 * 64;\n";
  for (size_t n = 0; n < p.blocks.size(); ++n) {
    const CBlock& b = p.blocks[n];
    const int ns = grad_stage(p, b);
    const long long nt = grad_tiles(b);
    s += fmt("  { const i64 per = ((span + @) / @ + @) / @ * @, splits = (N + per - 1) / per;\n",
             {b.d3 - 1, b.d3, ns - 1, ns, ns});
    s += fmt("    if (tile < @) { reduce_tile<@, @, @, @>(part, rows@, gw, @, splits, tile, at, lds); return; }\n",
             {nt, b.channels, b.mul3, grad_tc(b), grad_tw(b), (long long)n, nt});
    s += fmt("    tile -= @; part += splits * @LL; }\n", {nt, nt * 4096});
  }
  s += "}\n";
  return s;
}

hipFunction_t kernel_of(CPlan& p, int which) {
  static const char* const names[] = {"luna_con_fwd", "luna_con_ga", "luna_con_gw", "luna_con_gw_reduce"};
  return p.kernels.function(
      which, [] { return std::string("all"); }, [&](const std::string&) { return emit(p); },
      [&] { return std::string(names[which]); });
}

unsigned grid_x(int64_t tiles) {
  if (tiles > 0x7fffffffLL) fail("contraction: launch grid exceeds 2^31 workgroups");
  return (unsigned)tiles;
}

void product(CPlan& p, const void* in, const void* wt, void* out, int64_t rows, hipStream_t s, bool swap) {
  if (rows < 0) fail("negative problem size");
  if (rows == 0) return;
  if (!in || !wt || !out) fail("contraction: null tensor");
  int group = product_group(p, rows, swap);
  int64_t tiles = 0;
  for (const CBlock& b : p.blocks) {
    const int mn = swap ? b.channels : b.mul3;
    tiles += ceil_div(rows, tile_nodes(p.bits, b, mn)) * ceil_div(ceil_div(mn, tile_m(mn)), group);
  }
  void* args[] = {&in, &wt, &out, &rows, &group};
  launch(swap ? "con_ga" : "con_fwd", kernel_of(p, swap),
         dim3(grid_x(tiles)), dim3(256), s, args);
}

}  // namespace
}  // namespace luna

using namespace luna;

struct LunaConPlan {
  CPlan plan;
};

extern "C" {

int luna_con_plan_create(const char* spec, const char* cache_dir, LunaConPlan** out) {
  return guard_call([&] {
    if (!spec || !out) fail("luna_con_plan_create: null argument");
    auto holder = std::make_unique<LunaConPlan>();
    parse(holder->plan, spec);
    holder->plan.kernels.cache_dir = cache_dir ? cache_dir : "";
    holder->plan.kernels.tag = "con";
    *out = holder.release();
  });
}

int luna_con_plan_destroy(LunaConPlan* plan) {
  return guard_call([&] { delete plan; });
}

int luna_con_plan_precompile(LunaConPlan* plan) {
  return guard_call([&] {
    if (!plan) fail("luna_con_plan_precompile: null plan");
    plan->plan.kernels.code_for("all", [&] { return emit(plan->plan); });
  });
}

int luna_con_fwd(const LunaConPlan* plan, const void* a, const void* weight, void* out, int64_t rows,
                 LunaStream stream) {
  return guard_call([&] {
    if (!plan) fail("luna_con_fwd: null plan");
    product(const_cast<LunaConPlan*>(plan)->plan, a, weight, out, rows, (hipStream_t)stream, false);
  });
}

int luna_con_grad_a(const LunaConPlan* plan, const void* g, const void* weight, void* ga, int64_t rows,
                    LunaStream stream) {
  return guard_call([&] {
    if (!plan) fail("luna_con_grad_a: null plan");
    product(const_cast<LunaConPlan*>(plan)->plan, g, weight, ga, rows, (hipStream_t)stream, true);
  });
}

int luna_con_grad_w_workspace(const LunaConPlan* plan, int64_t rows, size_t* bytes) {
  return guard_call([&] {
    if (!plan || !bytes) fail("luna_con_grad_w_workspace: null argument");
    if (rows < 0) fail("negative problem size");
    *bytes = grad_partials(plan->plan, rows) * (plan->plan.bits / 8);
  });
}

int luna_con_grad_w(const LunaConPlan* cplan, const void* a, const void* g, void* gw, void* workspace,
                    size_t workspace_bytes, int64_t rows, LunaStream stream) {
  return guard_call([&] {
    if (!cplan) fail("luna_con_grad_w: null plan");
    CPlan& p = const_cast<LunaConPlan*>(cplan)->plan;
    if (rows < 0) fail("negative problem size");
    if (!gw || (rows > 0 && (!a || !g))) fail("luna_con_grad_w: null tensor");
    const size_t need = grad_partials(p, rows) * (p.bits / 8);
    if (need && (!workspace || workspace_bytes < need)) fail("luna_con_grad_w: workspace too small");
    int64_t span = grad_span(p, rows), groups = 0, tiles = 0;
    for (const CBlock& b : p.blocks) {
      groups += ceil_div(rows, grad_rows(p, b, span)) * grad_tiles(b);
      tiles += grad_tiles(b);
    }
    hipStream_t s = (hipStream_t)stream;
    if (rows > 0) {
      void* args[] = {&a, &g, &workspace, &rows, &span};
      launch("con_gw", kernel_of(p, 2), dim3(grid_x(groups)), dim3(256), s, args);
    }
    void* args[] = {&workspace, &gw, &rows, &span};
    launch("con_gw_reduce", kernel_of(p, 3), dim3(grid_x(tiles * 64)), dim3(256), s, args);
  });
}

}  // extern "C"
