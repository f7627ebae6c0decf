// fp64 matrix products whose operands are addressed by one stride per index (SplitParams).
//
// What bounds it: v_mfma_f64_16x16x4_f64 does not run beside other vector instructions.  A loop of nothing else
// reaches 55-60 TFLOP/s with one wavefront per SIMD (84 cycles per instruction instead of 64), 65-67 with two to four,
// and two integer instructions per MFMA take 67 down to 58.  So the K loop here has no vector instructions besides
// MFMAs and memory operations -- loads go through a buffer descriptor with a fixed offset per lane and a scalar one
// for the step, LDS addresses are fixed registers plus immediates -- and the tiles leave two to three blocks to a CU.
//
// A tile of an operand stands in LDS as [row][16 k], 16-byte pieces of two k; a lane's fragment of one read serves
// two MFMAs (any assignment of k to the steps will do as long as A and B agree).  Piece c of row r sits at position
// c ^ (r / 2 % 8), so that the 16 rows of a fragment read hit 64 different banks without padding.
#include "gemm_kernel.hpp"

using namespace hg;
using namespace hg::gemm;

namespace {

using d2 = double __attribute__((ext_vector_type(2)));
using u2 = uint32_t __attribute__((ext_vector_type(2)));
using u4 = uint32_t __attribute__((ext_vector_type(4)));
using Acc = MfmaF64::Acc;

constexpr int SK = 16;                      // k of one step

__device__ __forceinline__ int lds_at(int r, int c) { return r * 8 + (c ^ ((r >> 1) & 7)); }

// One operand's share of a tile: ROWS rows of SK elements, a lane owns NS pieces of two k.
template <int ROWS, bool KC>
struct Side {
  static constexpr int NS = ROWS * 8 / NT;
  static_assert(NS * NT == ROWS * 8, "whole pieces");
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t off[NS];                         // bytes
  int at[NS];
  uint32_t ks;                              // bytes between neighbouring k

  __device__ __forceinline__ static int row(int t, int i) { return KC ? (t + i * NT) / 8 : (t + i * NT) % ROWS; }
  __device__ __forceinline__ static int piece(int t, int i) { return KC ? (t + i * NT) % 8 : (t + i * NT) / ROWS; }

  __device__ __forceinline__ void init(int t, const double* base, uint32_t bytes, uint32_t rs, int r0, int rows, uint32_t stride) {
    rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, bytes, 0x00027000);
    ks = stride;
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      const int r = row(t, i), c = piece(t, i);
      off[i] = (uint32_t)(r0 + r < rows ? r0 + r : rows - 1) * rs + 2 * c * ks;      // (rows past the end: never stored)
      at[i] = lds_at(r, c);
    }
  }
  __device__ __forceinline__ static u4 both(u2 a, u2 b) { return u4{a[0], a[1], b[0], b[1]}; }
  // A whole step that starts at k0.
  __device__ __forceinline__ void load(int k0, u4* s) const {
    const uint32_t so = (uint32_t)k0 * ks;
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      if constexpr (KC) s[i] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off[i], so, 0));
      else
        s[i] = both(__builtin_bit_cast(u2, __builtin_amdgcn_raw_buffer_load_b64(rsrc, off[i], so, 0)),
                    __builtin_bit_cast(u2, __builtin_amdgcn_raw_buffer_load_b64(rsrc, off[i], so + ks, 0)));
    }
  }
  // The last step of a chunk when it is not a whole one: `left` elements of k, zeros behind them.
  __device__ __forceinline__ void load_tail(int t, int k0, int left, u4* s) const {
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      const int k = 2 * piece(t, i);
      u2 v[2];
#pragma unroll
      for (int j = 0; j < 2; ++j)
        v[j] = __builtin_bit_cast(u2, __builtin_amdgcn_raw_buffer_load_b64(rsrc, k + j < left ? off[i] + (k0 + j) * ks : 0xfffffff0u, 0, 0));
      s[i] = both(v[0], v[1]);
    }
  }
  __device__ __forceinline__ void store(const u4* s, u4* tile) const {
#pragma unroll
    for (int i = 0; i < NS; ++i) tile[at[i]] = s[i];
  }
};

// AKC, BKC: the operand is contiguous along k (lanes stage 16 bytes of a row; otherwise a row each, 8 bytes of two k).
// ROWS: the lanes also add up the elements of A they stage, eight lanes to a row (see gemm_split.hip); blocks of the first
// column of tiles do, for products that ask.
template <bool AKC, bool BKC, bool ROWS>
__device__ __forceinline__ void gemm_wide_f64_body(const SplitParams& p, const double* __restrict__ A, const double* __restrict__ B, double* __restrict__ C, int nr, int nsplits, int batch) {
  constexpr int WM = 2, WN = 2, TM = 2, TN = 2;          // wavefronts, and 16 x 16 blocks of each
  constexpr int BM = 16 * WM * TM, BN = 16 * WN * TN;
  __shared__ u4 lds[2][(BM + BN) * 8];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave / WN, wn = wave % WN;

  const auto share = split_share<BM, BN>(p, A, B, nr, nsplits, batch);
  const int m0 = share.m0, n0 = share.n0, kbeg = share.kbeg, kend = share.kend;

  Side<BM, AKC> sa;
  Side<BN, BKC> sb;
  sa.init(t, share.A, p.a_bytes, p.sam, m0, p.M, p.sak);
  sb.init(t, share.B, p.b_bytes, p.sbn, n0, p.N, p.sbk);
  constexpr int NA = Side<BM, AKC>::NS, NB = Side<BN, BKC>::NS;

  Acc acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = MfmaF64::zero();

  const int steps = (kend - kbeg + SK - 1) / SK, whole = (kend - kbeg) / SK;
  u4 ra[NA], rb[NB];
  static_assert(!ROWS || AKC, "the lanes of a row stage pieces of it");
  const bool sum_rows = ROWS && p.rows != nullptr && n0 == 0;
  double row_sum[NA], row_factor = 1;
#pragma unroll
  for (int i = 0; i < NA; ++i) row_sum[i] = 0;
  if (sum_rows && p.row_factor) row_factor = *(const double*)p.row_factor;
  auto store_a = [&](u4* to, int left) {      // left: elements of k that the step has, SK and more: all
    sa.store(ra, to);
    if (sum_rows) {
#pragma unroll
      for (int i = 0; i < NA; ++i) {
        const d2 x = __builtin_bit_cast(d2, ra[i]);
#pragma unroll
        for (int j = 0; j < 2; ++j)
          if (left >= SK || 2 * (t % 8) + j < left) row_sum[i] = __builtin_fma(x[j], row_factor, row_sum[i]);
      }
    }
  };
  auto fetch = [&](int i) {
    sa.load(kbeg + i * SK, ra);
    sb.load(kbeg + i * SK, rb);
  };
  auto fetch_tail = [&](int i) {
    sa.load_tail(t, kbeg + i * SK, kend - kbeg - i * SK, ra);
    sb.load_tail(t, kbeg + i * SK, kend - kbeg - i * SK, rb);
  };
  if (whole > 0) fetch(0);
  else fetch_tail(0);
  store_a(lds[0], kend - kbeg);
  sb.store(rb, lds[0] + BM * 8);
  __syncthreads();

  // where the lane's fragments of the two halves of a step start
  const int r = lane & 15, q = lane >> 4;
  int fa[2], fb[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    fa[h] = lds_at(wm * TM * 16 + r, 4 * h + q);
    fb[h] = BM * 8 + lds_at(wn * TN * 16 + r, 4 * h + q);
  }
  // One step on buffer `cur`.  next: 0 = there is none behind it, 1 = a whole step, 2 = the rest of K.
  auto step = [&](int i0, auto buffer, auto next) {
    constexpr int cur = decltype(buffer)::value;
    if constexpr (decltype(next)::value == 1) fetch(i0 + 1);
    if constexpr (decltype(next)::value == 2) fetch_tail(i0 + 1);
    __builtin_amdgcn_sched_barrier(0);      // (left to itself the compiler moves the loads down to their use)
    d2 a[2][TM], b[2][TN];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int i = 0; i < TM; ++i) a[h][i] = __builtin_bit_cast(d2, lds[cur][fa[h] + i * 128]);
#pragma unroll
      for (int j = 0; j < TN; ++j) b[h][j] = __builtin_bit_cast(d2, lds[cur][fb[h] + j * 128]);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = MfmaF64::run(a[h][i][u], b[h][j][u], acc[i][j]);
    if constexpr (decltype(next)::value != 0) {
      __builtin_amdgcn_sched_barrier(0);
      store_a(lds[cur ^ 1], decltype(next)::value == 1 ? SK : kend - kbeg - (i0 + 1) * SK);
      sb.store(rb, lds[cur ^ 1] + BM * 8);
    }
    __syncthreads();
  };
  constexpr std::integral_constant<int, 0> b0{};
  constexpr std::integral_constant<int, 1> b1{};
  constexpr std::integral_constant<int, 2> rest{};
  int i0 = 0;
#pragma unroll 1
  for (; i0 + 2 < whole; i0 += 2) {
    step(i0, b0, b1);
    step(i0 + 1, b1, b1);
  }
  // up to two whole steps and a last one that is not whole are left; i0 is even
  if (i0 + 1 < whole) {
    step(i0, b0, b1);
    if (i0 + 2 < steps) {
      step(i0 + 1, b1, rest);
      step(i0 + 2, b0, b0);
    } else {
      step(i0 + 1, b1, b0);
    }
  } else if (i0 + 1 < steps) {
    step(i0, b0, rest);
    step(i0 + 1, b1, b0);
  } else {
    step(i0, b0, b0);
  }

  if (sum_rows) {
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      double v = row_sum[i];
      for (int o = 1; o < 8; o <<= 1) v += __shfl_xor(v, o);
      const int m = m0 + (t + i * NT) / 8;
      if (t % 8 == 0 && m < p.M) p.rows[(int64_t)m * nsplits + share.s] = v;
    }
  }
  double* Cout = C + (int64_t)batch * p.bsc + (int64_t)share.s * p.c_split_stride;
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + (wn * TN + j) * 16 + MfmaF64::col(lane);
    if (n >= p.N) continue;
    double* col = Cout + (int64_t)n * p.scn;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + (wm * TM + i) * 16 + MfmaF64::row(lane, e);
        if (m < p.M) col[(int64_t)m * p.scm] = acc[i][j][e];
      }
  }
}

template <bool AKC, bool BKC>
__global__ void __launch_bounds__(NT, 4) k_gemm_wide_f64(SplitParams p, const double* __restrict__ A, const double* __restrict__ B, double* __restrict__ C) {
  gemm_wide_f64_body<AKC, BKC, false>(p, A, B, C, blockIdx.x + gridDim.x * blockIdx.y, gridDim.y, blockIdx.z);
}

template <bool AKC, bool BKC, bool ROWS>
__global__ void __launch_bounds__(NT, 4) k_gemm_wide_f64_group(SplitGroup g) {
  int nr;
  const int k = split_job(g, blockIdx.x, &nr);
  if (k < 0) return;
  const SplitJob& j = g.job[k];
  const int per_batch = j.tiles * j.splits, batch = nr / per_batch;
  gemm_wide_f64_body<AKC, BKC, ROWS>(j.p, (const double*)j.A, (const double*)j.B, (double*)j.C, nr - batch * per_batch, j.splits, batch);
}

}  // namespace

namespace hg {
namespace gemm {

void launch_wide_f64(const SplitParams& p, const LaunchArgs& a) {
  const double *A = (const double*)a.A, *B = (const double*)a.B;
  double* C = (double*)a.C;
  if (a.va && a.vb) launch_kernel(a, k_gemm_wide_f64<true, true>, p, A, B, C);
  else if (a.va) launch_kernel(a, k_gemm_wide_f64<true, false>, p, A, B, C);
  else if (a.vb) launch_kernel(a, k_gemm_wide_f64<false, true>, p, A, B, C);
  else launch_kernel(a, k_gemm_wide_f64<false, false>, p, A, B, C);
}

void launch_wide_f64_group(const SplitGroup& g, unsigned grid, bool akc, bool bkc, bool rows, hipStream_t stream) {
  auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(grid), dim3(NT), 0, stream, g); };
  if (rows && bkc) go(k_gemm_wide_f64_group<true, true, true>);
  else if (rows) go(k_gemm_wide_f64_group<true, false, true>);
  else if (akc && bkc) go(k_gemm_wide_f64_group<true, true, false>);
  else if (akc) go(k_gemm_wide_f64_group<true, false, false>);
  else if (bkc) go(k_gemm_wide_f64_group<false, true, false>);
  else go(k_gemm_wide_f64_group<false, false, false>);
}

}  // namespace gemm
}  // namespace hg
