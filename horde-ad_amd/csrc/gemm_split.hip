// fp32 matrix products on the bf16 matrix cores, without giving up fp32.
//
// An fp32 number is the exact sum of three bf16 numbers (8 + 8 + 8 significant
// bits): x = h + m + l, each part the nearest bf16 of what is left, so that
// |m| <= 2^-8 |x| and |l| <= 2^-17 |x|.  A product of two such sums has nine terms;
// the six largest are h h', h m', m h', m m', h l', l h', and the three left out
// (m l', l m', l l') together stay below 2^-24 of the product (plus 2^-34): as much as
// rounding the product to fp32 may cost.  Every term of the six is a product of
// two 8-bit numbers, exact in fp32.
//
// How the terms are added decides the rest.  The matrix cores drop low bits of what they add onto a larger number, so h h'
// is summed from zero, sixteen at a time, and goes to its accumulator with one rounded addition, and the five small terms
// have an accumulator of their own, on the matrix cores throughout (2^-7 of the other one: its lost bits do not
// count); the two meet in one addition at the end.  Error against fp64 in units of 2^-24 of the sum of magnitudes, mean (max),
// 2048 terms, beside v_mfma_f32_32x32x2_f32 and beside all six terms in one chain:
//     normally distributed      0.039 (0.34)   0.098 (0.65)   0.064 (0.38)
//     uniform in 0 .. 1         0.67  (3.8)    0.84  (4.7)    0.66  (3.5)
//     e^-uniform(0, 100)        0.24  (2.2)    0.27  (2.1)    0.29  (2.1)
//     one product, no others    0.366 (1.7)    0.361 (1.0)    0.457 (2.4)
// With m l' and l m' as well the last row is 0.361 (1.0) too, and a product on tiles of 128 x 128 takes a fifth longer
// (464 -> 557 us below): left at six there.  The thin tiles form all eight.
//
// Range.  Operands are multiplied by 2^23 on their way into the split (the first remainder is one fma, so it costs one
// multiplication an element), the sums by 2^-46 on their way out: the smallest fp32 number, 2^-149, is then 2^-126, and no
// part of any element is subnormal.  From above, the parts must not overflow, nor the sums of their products, which are
// 2^-7 larger than the products themselves while only h h' has been added.  Every block knows the largest element of each
// operand it has staged: where 2^23 of it or 2^46 K |a| |b| could pass 2^127 -- elements from 2^104, infinities, products from
// 2^81 / K -- the block computes its tile again with v_mfma_f32_32x32x2_f32, so such inputs give what they always gave.
// (Limits at 2^-100 and 2^127 on the elements alone, without the scaling, sent every tile that met a softmax
// probability under e^-69 the second way, 3.9 ms instead of 0.41 for 2048 x 8192 over 2048, and let products just
// below 2^128 overflow.)
//
// What bounds it: the mix of instructions beside the products and the power all of them draw.  Six bf16 instructions of
// 32 x 32 x 16 do the work of eight fp32 ones of 32 x 32 x 2.  Loops of nothing but the step's instructions, TFLOP/s of bf16 on
// normal numbers: products alone 1787, with the reads of LDS 1647, with the rounded additions too 1499, with the split's vector
// instructions (7 an element) 1324, with the writes to LDS 1230, with the barriers 1207, with loads that a step waits for 1027.
// The loads are a step ahead of their use: they go out when the registers of the step before are split (the compiler, left to itself,
// waited for loads of the same step behind a sixth of its products), 1033 -> 1064 here.  2048 x 8192 over 2048, normally
// distributed / behind a relu, one after another: 398 / 385 us with loads of the same step, 388 / 374 now (fp32 instruction 649 / 615
// on another card); three of 128 x 128 over 27 x 5000 in one launch 126 / 117, bound by their loads (377 MB).
// (256 x 256 tiles split an element half as often, but two sets of accumulators do not fit: all six terms in one
// chain, or the second set added up by vector instructions, were no faster; nor were 256 x 128 tiles.  Remainders formed
// by v_dot2_f32_bf16, two instructions less a remainder: wrong results.)
#include "gemm_kernel.hpp"

using namespace hg;
using namespace hg::gemm;

namespace {

using bf8 = __bf16 __attribute__((ext_vector_type(8)));
using bf2 = __bf16 __attribute__((ext_vector_type(2)));
using f2 = float __attribute__((ext_vector_type(2)));
using f4u = float __attribute__((ext_vector_type(4), aligned(4)));
using f16v = float __attribute__((ext_vector_type(16)));
using u4 = uint32_t __attribute__((ext_vector_type(4)));

constexpr int SK = 16;                      // k of one step: one MFMA deep

// Eight consecutive k of one row on their way to LDS.
struct Slot { float v[8]; };

constexpr int kScaleLog = 23;               // operands are split after multiplication by 2^23
constexpr float kScale = 8388608.0f, kUnscale = 1.0f / (8388608.0f * 8388608.0f);

__device__ __forceinline__ uint32_t pack(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{a, b}, bf2));
}

// the three parts of two neighbours, scaled
__device__ __forceinline__ void split2(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = pack(a * kScale, b * kScale);
  const float a1 = __builtin_fmaf(a, kScale, -__builtin_bit_cast(float, h << 16)), b1 = __builtin_fmaf(b, kScale, -__builtin_bit_cast(float, h & 0xffff0000u));
  m = pack(a1, b1);
  l = pack(a1 - __builtin_bit_cast(float, m << 16), b1 - __builtin_bit_cast(float, m & 0xffff0000u));
}

// Element (16 bytes) of row r, k half h within one part of a tile: rows of 32 bytes, the halves
// swapped in every other group of four rows so that eight neighbouring rows of one half lie in different banks.
__device__ __forceinline__ int lds_at(int r, int h) { return r * 2 + (h ^ ((r >> 3) & 1)); }

// One operand's share of a tile: ROWS rows of SK elements, a lane owns NS pieces of eight k each.
// Loads go through a buffer descriptor over the operand: a fixed 32-bit offset per lane plus a
// scalar one for the step, and whatever lies past the end (rows, k) reads as zero.
template <int ROWS, bool KC>
struct Side {
  static constexpr bool ALL = ROWS * 2 >= NT;      // every lane owns a piece
  static constexpr int NS = ALL ? ROWS * 2 / NT : 1;
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t off[NS];                         // bytes
  int at[NS];
  uint32_t ks;                              // bytes between neighbouring k

  __device__ __forceinline__ void init(int t, const float* base, uint32_t bytes, uint32_t rs, int r0, int rows, uint32_t stride) {
    rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, bytes, 0x00027000);
    ks = stride;
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      // lanes run along whichever of k and the rows is contiguous
      const int r = KC ? t / 2 + i * (NT / 2) : (t + i * NT) % ROWS;
      const int h = KC ? t & 1 : (t + i * NT) / ROWS;
      off[i] = (uint32_t)(r0 + r < rows ? r0 + r : rows - 1) * rs + 8 * h * ks;   // (rows past the end: never stored)
      at[i] = lds_at(r, h);
    }
    if (!ALL && t >= ROWS * 2) off[0] = 0x80000000u;      // (past the end with whatever is added)
  }
  // A whole step that starts at k0.
  __device__ __forceinline__ void load(int k0, Slot* s) const {
    const uint32_t so = (uint32_t)k0 * ks;
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      if constexpr (KC) {
        const f4u a = __builtin_bit_cast(f4u, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off[i], so, 0));
        const f4u b = __builtin_bit_cast(f4u, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off[i] + 16, so, 0));
#pragma unroll
        for (int j = 0; j < 4; ++j) { s[i].v[j] = a[j]; s[i].v[4 + j] = b[j]; }
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) s[i].v[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, off[i], so + j * ks, 0));
      }
    }
  }
  // The last step of a chunk when it is not a whole one: `left` elements of k.
  __device__ __forceinline__ void load_tail(int t, int k0, int left, Slot* s) const {
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      const int h = KC ? 8 * (t & 1) : 8 * ((t + i * NT) / ROWS);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        s[i].v[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, h + j < left ? off[i] + (k0 + j) * ks : 0xfffffff0u, 0, 0));
    }
  }
  // Elements 2 j and 2 j + 1 of a piece become theirs of its three parts.
  static __device__ __forceinline__ void split(const Slot& s, int j, u4* parts, float& largest) {
    uint32_t h, m, l;
    split2(s.v[2 * j], s.v[2 * j + 1], h, m, l);
    parts[0][j] = h;
    parts[1][j] = m;
    parts[2][j] = l;
    asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(largest) : "v"(s.v[2 * j]), "v"(s.v[2 * j + 1]));      // (passes NaNs over: their parts are NaNs)
  }
  // to: [3][ROWS * 2] of 16 bytes
  __device__ __forceinline__ void put(const u4* parts, int i, u4* to) const {
    if (!ALL && threadIdx.x >= ROWS * 2) return;
#pragma unroll
    for (int q = 0; q < 3; ++q) to[q * ROWS * 2 + at[i]] = parts[q];
  }
};

// Four consecutive k of one row from k on; zeros from kend on.
template <bool KC>
__device__ __forceinline__ void four(__amdgpu_buffer_rsrc_t rsrc, uint32_t row, uint32_t ks, int k, bool whole, int kend, float* v) {
  if (KC && whole) {
    const f4u x = __builtin_bit_cast(f4u, __builtin_amdgcn_raw_buffer_load_b128(rsrc, row + k * ks, 0, 0));
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = x[u];
  } else {
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, k + u < kend ? row + (k + u) * ks : 0xfffffff0u, 0, 0));
  }
}

// THIN: tiles of 128 x 32 for products with at most 32 columns (weight gradients of narrow layers), bound by the loads of A:
// a step is 10 KB of loads and eight instructions a wavefront, one step ahead, so four blocks (124 to 128 registers, 30 KB of
// LDS) hide one another's trips to memory (with six instructions the same products take 2 to 3 % less).  128 x 28 over 28 x 5000
// with its row sums, 87 MB, in the recurrent network's gradient: 30.1 us with loads of the same step, 26.5 now; the 32 x 32 tiles of the fp32
// instruction, which read A for every 32 rows of it and B four times, 33.0 without sums.
// ROWS: the lanes also add up, in fp64, the elements of A they stage: a bias gradient is the row sums of what the weight
// gradient multiplies.  Blocks of the first column of tiles do, for products that ask (split_job).  Reading A once more for
// them: 28 x 128 rows of 5000 17.5 us, 2048 rows of 8192 17.4; here
// they cost the recurrent network's products 3 to 4 us.
template <bool AKC, bool BKC, bool THIN, bool ROWS>
__device__ __forceinline__ void gemm_split_body(const SplitParams& p, const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C, int nr, int nsplits, int batch) {
  constexpr int WM = THIN ? 4 : 2, WN = THIN ? 1 : 2, TM = THIN ? 1 : 2, TN = THIN ? 1 : 2;          // wavefronts, and 32 x 32 blocks of each
  constexpr int BM = 32 * WM * TM, BN = 32 * WN * TN;
  constexpr int PA = 3 * BM * 2, PB = 3 * BN * 2;       // 16-byte elements of one buffer
  __shared__ u4 lds[2][PA + PB];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave / WN, wn = wave % WN;

  const auto share = split_share<BM, BN>(p, A, B, nr, nsplits, batch);
  const int m0 = share.m0, n0 = share.n0, kbeg = share.kbeg, kend = share.kend;

  Side<BM, AKC> sa;
  Side<BN, BKC> sb;
  sa.init(t, share.A, p.a_bytes, p.sam, m0, p.M, p.sak);
  sb.init(t, share.B, p.b_bytes, p.sbn, n0, p.N, p.sbk);
  constexpr int NA = Side<BM, AKC>::NS, NB = Side<BN, BKC>::NS;

  f16v acc[TM][TN], low[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = low[i][j][r] = 0;
  float top_a = 0, top_b = 0;               // the largest magnitude of each operand met so far

  const int steps = (kend - kbeg + SK - 1) / SK, whole = (kend - kbeg) / SK;
  Slot ra[NA], rb[NB];
  static_assert(!ROWS || (AKC && NA == 1 && BM * 2 == NT), "lane t stages a half of row t / 2");
  const bool sum_rows = ROWS && p.rows != nullptr && n0 == 0;
  double row_sum = 0, row_factor = 1;
  if (sum_rows && p.row_factor) row_factor = (double)*(const float*)p.row_factor;
  // Pair number w of what the block stages of a step: split; with the last one of a piece its parts go to LDS.
  // left: elements of k that the step has, 16 and more: all
  constexpr int PAIRS = 4 * (NA + NB);
  u4 parts[3];
  auto stage = [&](int w, u4* to, int left) {
    const int u = w / 4, j = w % 4;
    if (u < NA) {
      sa.split(ra[u], j, parts, top_a);
      if (sum_rows) {
#pragma unroll
        for (int e = 2 * j; e < 2 * j + 2; ++e)
          if (left >= SK || 8 * (t & 1) + e < left) row_sum = __builtin_fma((double)ra[u].v[e], row_factor, row_sum);      // (the product is exact)
      }
      if (j == 3) sa.put(parts, u, to);
    } else {
      sb.split(rb[u - NA], j, parts, top_b);
      if (j == 3) sb.put(parts, u - NA, to + PA);
    }
  };
  auto fetch = [&](int i) {                 // (chosen outside the main loop: a load on one side of a branch would be waited for where the sides meet)
    sa.load(kbeg + i * SK, ra);
    sb.load(kbeg + i * SK, rb);
  };
  auto fetch_tail = [&](int i) {
    sa.load_tail(t, kbeg + i * SK, kend - kbeg - i * SK, ra);
    sb.load_tail(t, kbeg + i * SK, kend - kbeg - i * SK, rb);
  };
  if (whole > 0) fetch(0);
  else fetch_tail(0);
#pragma unroll
  for (int w = 0; w < PAIRS; ++w) stage(w, lds[0], kend - kbeg);
  if (whole > 1) fetch(1);
  else if (steps > 1) fetch_tail(1);
  __syncthreads();

  const int fra = lds_at(wm * TM * 32 + (lane & 31), lane >> 5), frb = lds_at(wn * TN * 32 + (lane & 31), lane >> 5);
  // One step: its products are formed; behind them the next step's elements, which have been on their way for a
  // step, are split and stored to the other buffer, and as soon as a piece's registers are free the loads of the step after that go out.
  // next: the next step exists. load: 0 = the one after it does not, 1 = it is a whole one, 2 = the rest of K.
  auto step = [&](int i0, auto next, auto load) {
    constexpr bool more = decltype(next)::value != 0;
    constexpr int ld = decltype(load)::value;
    const int cur = i0 & 1;
    const u4* la = lds[cur] + fra;
    const u4* lb = lds[cur] + PA + frb;
    u4* ln = lds[cur ^ 1];
    const int left = ld ? SK : kend - kbeg - (i0 + 1) * SK;
    bf8 fa[TM][3], fb[TN][3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[i][q] = __builtin_bit_cast(bf8, la[q * BM * 2 + i * 64]);
#pragma unroll
      for (int j = 0; j < TN; ++j) fb[j][q] = __builtin_bit_cast(bf8, lb[q * BN * 2 + j * 64]);
    }
    constexpr int TERMS = THIN ? 8 : 6, PRODUCTS = TM * TN * TERMS;
    constexpr int FIRST = 3;               // (the loads have had a step to arrive; a little more does no harm)
    auto until = [&](int product) {          // pairs staged before the product after this one
      const int n = product < FIRST ? 0 : (product - FIRST + 1) * PAIRS / (PRODUCTS - FIRST - 1);
      return n < PAIRS ? n : PAIRS;
    };
    auto behind = [&](int product) {        // what is staged behind a product
      if constexpr (more) {
#pragma unroll
        for (int w = 0; w < PAIRS; ++w) {
          if (w < until(product - 1) || w >= until(product)) continue;
          stage(w, ln, left);
          if (w == 4 * NA - 1) {
            if constexpr (ld == 1) sa.load(kbeg + (i0 + 2) * SK, ra);
            if constexpr (ld == 2) sa.load_tail(t, kbeg + (i0 + 2) * SK, kend - kbeg - (i0 + 2) * SK, ra);
          }
          if (w == PAIRS - 1) {
            if constexpr (ld == 1) sb.load(kbeg + (i0 + 2) * SK, rb);
            if constexpr (ld == 2) sb.load_tail(t, kbeg + (i0 + 2) * SK, kend - kbeg - (i0 + 2) * SK, rb);
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int b = 0; b < TM * TN; ++b) {
      // h h' of 16 k is summed from zero and added with one rounded addition; the five smaller terms are summed on the
      // matrix cores, the smallest first.
      const int i = b % TM, j = b / TM;
      int n = b * TERMS;
      f16v zero;
#pragma unroll
      for (int r = 0; r < 16; ++r) zero[r] = 0;
      auto add = [&](int qa, int qb, const f16v& c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i][qa], fb[j][qb], c, 0, 0, 0); };
      const f16v c = add(0, 0, zero);
      behind(n++);
      if constexpr (THIN) {
        low[i][j] = add(2, 1, low[i][j]);
        behind(n++);
        low[i][j] = add(1, 2, low[i][j]);
        behind(n++);
      }
      low[i][j] = add(2, 0, low[i][j]);
      behind(n++);
      low[i][j] = add(0, 2, low[i][j]);
#pragma unroll
      for (int r = 0; r < 5; ++r) acc[i][j][r] += c[r];
      behind(n++);
      low[i][j] = add(1, 1, low[i][j]);
#pragma unroll
      for (int r = 5; r < 10; ++r) acc[i][j][r] += c[r];
      behind(n++);
      low[i][j] = add(1, 0, low[i][j]);
#pragma unroll
      for (int r = 10; r < 16; ++r) acc[i][j][r] += c[r];
      behind(n++);
      low[i][j] = add(0, 1, low[i][j]);
      behind(n++);
    }
    __syncthreads();
  };
  constexpr std::integral_constant<int, 0> none{};
  constexpr std::integral_constant<int, 1> full{};
  constexpr std::integral_constant<int, 2> rest{};
  int i0 = 0;
#pragma unroll 1
  for (; i0 + 2 < whole; ++i0) step(i0, full, full);
  if (i0 + 2 < steps) step(i0++, full, rest);
  if (i0 + 1 < steps) step(i0++, full, none);
  step(i0, none, none);

  if (sum_rows) {
    row_sum += __shfl_xor(row_sum, 1);
    if (!(t & 1) && m0 + t / 2 < p.M) p.rows[(int64_t)(m0 + t / 2) * nsplits + share.s] = row_sum;
  }
  float* Cout = C + (int64_t)batch * p.bsc + (int64_t)share.s * p.c_split_stride;
  auto put = [&](int i, int j, const f16v& c, float scale) {
    const int n = n0 + (wn * TN + j) * 32 + (lane & 31);
    if (n >= p.N) return;
    float* col = Cout + (int64_t)n * p.scn;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = m0 + (wm * TM + i) * 32 + MfmaF32W::row(lane, r);
      if (m < p.M) col[(int64_t)m * p.scm] = c[r] * scale;
    }
  };
  // what the largest elements of the whole block allow: see the head of the file
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    top_a = fmaxf(top_a, __shfl_xor(top_a, d));
    top_b = fmaxf(top_b, __shfl_xor(top_b, d));
  }
  float* tops = reinterpret_cast<float*>(lds[0]);      // (free: the last step ended with a barrier)
  if (lane == 0) {
    tops[2 * wave] = top_a;
    tops[2 * wave + 1] = top_b;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < WM * WN; ++w) {
    top_a = fmaxf(top_a, tops[2 * w]);
    top_b = fmaxf(top_b, tops[2 * w + 1]);
  }
  auto exponent = [](float x) { return (int)(__builtin_bit_cast(uint32_t, x) >> 23) - 126; };
  const int ea = exponent(top_a), eb = exponent(top_b);                           // |a| < 2^ea, |b| < 2^eb
  const int ek = 32 - __builtin_clz((uint32_t)(kend - kbeg));                      // K < 2^ek
  if (ea + kScaleLog > 127 || eb + kScaleLog > 127 || ea + eb + 2 * kScaleLog + ek + 1 > 127) {
    // elements or sums that could leave fp32's range: the tile again, on the fp32 instruction.  Fragments come straight from
    // memory, eight k ahead (bound by their loads where those run along the rows); each serves a wavefront's whole
    // row or column of blocks.  2048 x 8192 over 2048, one infinity / one in every tile: 930 / 1080 us (2380 for one
    // with a block of 32 x 32 at a time and single elements loaded; 600-640 on the fp32 instruction from the start).
    uint32_t ga[TM], gb[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int row = m0 + (wm * TM + i) * 32 + (lane & 31);
      ga[i] = (uint32_t)(row < p.M ? row : p.M - 1) * p.sam;
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int row = n0 + (wn * TN + j) * 32 + (lane & 31);
      gb[j] = (uint32_t)(row < p.N ? row : p.N - 1) * p.sbn;
    }
    struct Frag { float a[TM][4], b[TN][4]; };
    auto fetch8 = [&](int k0, Frag& f) {
#pragma unroll
      for (int i = 0; i < TM; ++i) four<AKC>(sa.rsrc, ga[i], sa.ks, k0 + 4 * (lane >> 5), k0 + 8 <= kend, kend, f.a[i]);
#pragma unroll
      for (int j = 0; j < TN; ++j) four<BKC>(sb.rsrc, gb[j], sb.ks, k0 + 4 * (lane >> 5), k0 + 8 <= kend, kend, f.b[j]);
    };
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;
    Frag now, next;
    fetch8(kbeg, now);
#pragma unroll 1
    for (int k0 = kbeg; k0 < kend; k0 += 8) {
      fetch8(k0 + 8, next);                 // (behind the end: zeros, without a fetch)
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(now.a[i][u], now.b[j][u], acc[i][j], 0, 0, 0);
      now = next;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) put(i, j, acc[i][j], 1.0f);
    return;
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) put(i, j, acc[i][j] + low[i][j], kUnscale);
}

template <bool AKC, bool BKC, bool THIN>
__global__ void __launch_bounds__(NT, THIN ? 4 : 2) k_gemm_split(SplitParams p, const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C) {
  gemm_split_body<AKC, BKC, THIN, false>(p, A, B, C, blockIdx.x + gridDim.x * blockIdx.y, gridDim.y, blockIdx.z);
}

template <bool AKC, bool BKC, bool THIN, bool ROWS>
__global__ void __launch_bounds__(NT, THIN ? 4 : 2) k_gemm_split_group(SplitGroup g) {
  int nr;
  const int k = split_job(g, blockIdx.x, &nr);
  if (k < 0) return;
  const SplitJob& j = g.job[k];
  const int per_batch = j.tiles * j.splits, batch = nr / per_batch;
  gemm_split_body<AKC, BKC, THIN, ROWS>(j.p, (const float*)j.A, (const float*)j.B, (float*)j.C, nr - batch * per_batch, j.splits, batch);
}

template <typename F>
void launch_as(const LaunchArgs& a, F kernel, const SplitParams& p) {
  const float* A = (const float*)a.A;
  const float* B = (const float*)a.B;
  float* C = (float*)a.C;
  if (a.ev_start || a.ev_stop) hipExtLaunchKernelGGL(kernel, a.grid, dim3(NT), 0, a.stream, a.ev_start, a.ev_stop, 0, p, A, B, C);
  else hipLaunchKernelGGL(kernel, a.grid, dim3(NT), 0, a.stream, p, A, B, C);
}

}  // namespace

namespace hg {
namespace gemm {

template <bool THIN>
static void launch_split(const SplitParams& p, const LaunchArgs& a) {
  if (a.va && a.vb) launch_as(a, k_gemm_split<true, true, THIN>, p);
  else if (a.va) launch_as(a, k_gemm_split<true, false, THIN>, p);
  else if (a.vb) launch_as(a, k_gemm_split<false, true, THIN>, p);
  else launch_as(a, k_gemm_split<false, false, THIN>, p);
}

void launch_split_f32(const SplitParams& p, const LaunchArgs& a, bool thin) {
  if (thin) launch_split<true>(p, a);
  else launch_split<false>(p, a);
}

template <bool THIN>
static void launch_split_group(const SplitGroup& g, unsigned grid, bool akc, bool bkc, bool rows, hipStream_t stream) {
  auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(grid), dim3(NT), 0, stream, g); };
  if (rows && bkc) go(k_gemm_split_group<true, true, THIN, true>);
  else if (rows) go(k_gemm_split_group<true, false, THIN, true>);
  else if (akc && bkc) go(k_gemm_split_group<true, true, THIN, false>);
  else if (akc) go(k_gemm_split_group<true, false, THIN, false>);
  else if (bkc) go(k_gemm_split_group<false, true, THIN, false>);
  else go(k_gemm_split_group<false, false, THIN, false>);
}

void launch_split_f32_group(const SplitGroup& g, unsigned grid, bool akc, bool bkc, bool thin, bool rows, hipStream_t stream) {
  if (thin) launch_split_group<true>(g, grid, akc, bkc, rows, stream);
  else launch_split_group<false>(g, grid, akc, bkc, rows, stream);
}

}  // namespace gemm
}  // namespace hg
