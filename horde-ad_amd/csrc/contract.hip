// Reductions and contractions over strided views:
//   out[o] = sum_r a[o,r] * b[o,r]
// which, with free views, is horde-ad's tssum / tssumN / tssum0 / tsdot0 /
// tsdot1In / tsmatvecmul / tsmatmul2 (src/HordeAd/Core/OpsConcrete.hs:215-242).
//
// This file holds the general path, bound by HBM bandwidth:
//   * lane-per-output: adjacent lanes own adjacent outputs and walk the
//     reduced index space with an odometer (coalesced when the kept innermost
//     dimension has unit stride: sums over outer dimensions);
//   * wave-per-output: the 64 lanes of a wavefront stride over the innermost
//     reduced dimension and combine with a shuffle tree (coalesced when the
//     reduced innermost dimension has unit stride: dot1In, sum0, dot0).
// Long reductions with few outputs are split into S chunks whose partial sums
// (double / int64 accumulators) are combined by a second launch, so the
// summation order is fixed by the shape alone: results are reproducible from
// run to run.  GEMM-shaped contractions are routed to the MFMA kernels first.
#include "common.hpp"

using namespace hg;

namespace hg {
// gemm.hip: returns HGPU_OK and sets *handled when the contraction was
// recognised as a matrix product and executed on the matrix cores.
int try_gemm(hgpu_ctx* ctx, const hgpu_array* a, const hgpu_array* b, int n_keep, hgpu_array* out, bool* handled,
             int n_terms = 0, const hgpu_array* const* as = nullptr, const hgpu_array* const* bs = nullptr, hgpu_array** partials_out = nullptr);
constexpr int kGemmMaxTerms = 32;   // products one launch of try_gemm sums (kMaxTerms of the kernels)
}

namespace {

constexpr int kBlock = 256;

template <typename T> struct acc_of { using type = int64_t; };
template <> struct acc_of<double> { using type = double; };
template <> struct acc_of<float> { using type = double; };

// Several products of one layout reduced by one launch (hgpu_contract_sum):
// the chunk index s of a work item also selects the term, s = term * s_per +
// chunk within the term, and the term's operands replace the kernel's pointer
// arguments.  n == 0: one product.
struct TermPtrs {
  int n, s_per;
  const void* a[hg::kGemmMaxTerms];
  const void* b[hg::kGemmMaxTerms];
};

template <typename A>
__device__ __forceinline__ A wave_sum(A v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    if constexpr (sizeof(A) == 8) {
      unsigned long long u = *reinterpret_cast<unsigned long long*>(&v);
      unsigned lo = __shfl_down((unsigned)(u & 0xffffffffu), off, 64);
      unsigned hi = __shfl_down((unsigned)(u >> 32), off, 64);
      unsigned long long w = ((unsigned long long)hi << 32) | lo;
      v += *reinterpret_cast<A*>(&w);
    } else {
      v += __shfl_down(v, off, 64);
    }
  }
  return v;
}

// Work item = (output o, chunk s); s-th chunk covers reduced linear indices
// [s*chunk, min(R, (s+1)*chunk)).  out is dense [n_out, S].
// A block takes 256 outputs of one chunk, so that all its lanes walk through the same reduced indices: their offsets are found
// once per 256 of them, each by one lane, and read from LDS, and eight loads per operand are in flight.  With an odometer of its own
// in every lane one load waited for the other.  us, before / so: 4096 columns of 4096 elements fp64 68.1 / 27.9, fp32 67.8 / 18.6, 20,000
// columns of 300 products fp32 26.7 / 9.6; a gradient of the convolution network at batch 7 (27 kernels, seven of them such
// reductions) with flat_sum below 314 / 272.
// (`bid` of `nb` blocks: the kernels below pass their own block index; the grouped kernel at the end of this
// file passes a block's place among the blocks of its problem.  tp == nullptr: one product.)
template <typename TI, typename TO, bool HASB, typename D>
__device__ __forceinline__ void lane_body(const D& keep, const D& red, int64_t n_out, int64_t R, int S, int64_t chunk,
                                          const TI* __restrict__ a0, const TI* __restrict__ b0, TO* __restrict__ out, const TermPtrs* tp, unsigned bid, unsigned nb) {
  using A = typename acc_of<TI>::type;
  constexpr int U = 8;
  __shared__ int64_t offs[HASB ? 2 : 1][kBlock];
  const int64_t per_chunk = (n_out + kBlock - 1) / kBlock, tiles = per_chunk * S;
  int64_t filled = -1;                 // the first of the indices whose offsets are there
  for (int64_t tile = bid; tile < tiles; tile += nb) {
    const int64_t s_all = tile / per_chunk, mine = (tile - s_all * per_chunk) * kBlock + threadIdx.x;
    const int64_t o = mine < n_out ? mine : n_out - 1;
    int64_t s = s_all;
    const TI* a = a0;
    const TI* b = b0;
    if (tp && tp->n) {
      int term = (int)(s / tp->s_per);
      s -= (int64_t)term * tp->s_per;
      a = (const TI*)tp->a[term];
      b = (const TI*)tp->b[term];
    }
    int64_t ko[2];
    decompose<2>(keep, o, ko);
    a += ko[0];
    if (HASB) b += ko[1];
    const int64_t r0 = s * chunk, r1 = r0 + chunk < R ? r0 + chunk : R;
    A acc = 0;
    for (int64_t r = r0; r < r1; r += kBlock) {
      const int m = r1 - r < kBlock ? (int)(r1 - r) : kBlock;
      if (r != filled) {               // (the same for all lanes)
        __syncthreads();
        if ((int)threadIdx.x < m) {
          int64_t ro[2];
          decompose<2>(red, r + threadIdx.x, ro);
          offs[0][threadIdx.x] = ro[0];
          if (HASB) offs[HASB ? 1 : 0][threadIdx.x] = ro[1];
        }
        __syncthreads();
        filled = r;
      }
      int k = 0;
      for (; k + U <= m; k += U) {
        A x[U], y[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          x[u] = (A)a[offs[0][k + u]];
          if (HASB) y[u] = (A)b[offs[HASB ? 1 : 0][k + u]];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (HASB) x[u] *= y[u];
          acc += x[u];
        }
      }
      for (; k < m; ++k) {
        A x = (A)a[offs[0][k]];
        if (HASB) x *= (A)b[offs[HASB ? 1 : 0][k]];
        acc += x;
      }
    }
    if (mine < n_out) out[o * S + s_all] = (TO)acc;
  }
}
template <typename TI, typename TO, bool HASB>
__global__ void __launch_bounds__(kBlock) k_contract_lane(Dims keep, Dims red, int64_t n_out, int64_t R, int S, int64_t chunk,
                                                           const TI* __restrict__ a0, const TI* __restrict__ b0, TO* __restrict__ out, TermPtrs tp) {
  lane_body<TI, TO, HASB>(keep, red, n_out, R, S, chunk, a0, b0, out, &tp, blockIdx.x, gridDim.x);
}

// Sum over j = j_first, j_first + 64, ... < j_end of a[j * sa] (* b[j * sb]): four
// independent accumulators keep four loads per operand in flight.
template <typename TI, typename A, bool HASB>
__device__ __forceinline__ A lane_strided_sum(const TI* __restrict__ pa, const TI* __restrict__ pb, int64_t sa, int64_t sb, int64_t j_first, int64_t j_end) {
  A acc0 = 0, acc1 = 0, acc2 = 0, acc3 = 0;
  int64_t j = j_first;
  for (; j + 192 < j_end; j += 256) {
    A x0 = (A)pa[j * sa], x1 = (A)pa[(j + 64) * sa], x2 = (A)pa[(j + 128) * sa], x3 = (A)pa[(j + 192) * sa];
    if (HASB) {
      x0 *= (A)pb[j * sb];
      x1 *= (A)pb[(j + 64) * sb];
      x2 *= (A)pb[(j + 128) * sb];
      x3 *= (A)pb[(j + 192) * sb];
    }
    acc0 += x0;
    acc1 += x1;
    acc2 += x2;
    acc3 += x3;
  }
  for (; j < j_end; j += 64) {
    A x = (A)pa[j * sa];
    if (HASB) x *= (A)pb[j * sb];
    acc0 += x;
  }
  return (acc0 + acc1) + (acc2 + acc3);
}

// The same sum over [j0, j1) where a lies side by side (and b does, or stays on one element, as the ones of a plain sum
// do): 16 bytes a load.  With four bytes a load, and b fetched for every element, rows of 5000 to 8192 fp32 went by at
// 3.4 TB/s: 2048 rows of 8192 19.5 -> 17.4 us, 28 x 128 rows of 5000 19.9 -> 16.3 us.  Element-aligned: rows start anywhere.
// For rows that fill one round of loads (4 KB): shorter ones are as fast either way.  Not in k_contract_group, whose
// reductions are mostly short and which the additional registers slow down (CNN: 326.6 -> 328.1 us).
template <typename TI> struct Vec16Of { using type = TI __attribute__((ext_vector_type(16 / sizeof(TI)), aligned(sizeof(TI)))); };
template <typename TI, typename A, bool HASB>
__device__ __forceinline__ A wide_sum(const TI* __restrict__ pa, const TI* __restrict__ pb, int64_t sb, int64_t j0, int64_t j1, int lane) {
  using V = typename Vec16Of<TI>::type;
  constexpr int N = 16 / sizeof(TI), U = 4;
  const bool vb = HASB && sb != 0;
  const A one_b = HASB && !vb ? (A)pb[0] : (A)1;
  A acc[U] = {0, 0, 0, 0};
  int64_t j = j0 + lane * N;
  auto add = [&](A& c, const V& x, const V& y) {
#pragma unroll
    for (int e = 0; e < N; ++e) c += HASB ? (A)x[e] * (vb ? (A)y[e] : one_b) : (A)x[e];
  };
  for (; j + (U - 1) * 64 * N + N <= j1; j += U * 64 * N) {
    V x[U], y[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = *reinterpret_cast<const V*>(pa + j + u * 64 * N);
    if (vb) {
#pragma unroll
      for (int u = 0; u < U; ++u) y[u] = *reinterpret_cast<const V*>(pb + j + u * 64 * N);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) add(acc[u], x[u], y[u]);
  }
  for (; j + N <= j1; j += 64 * N) {
    const V x = *reinterpret_cast<const V*>(pa + j);
    V y = x;
    if (vb) y = *reinterpret_cast<const V*>(pb + j);
    add(acc[0], x, y);
  }
  for (; j < j1; ++j) acc[1] += HASB ? (A)pa[j] * (vb ? (A)pb[j] : one_b) : (A)pa[j];      // (less than a vector, one lane's)
  return (acc[0] + acc[1]) + (acc[2] + acc[3]);
}
// Rows that the WIDE kernels take (not those that rows_sum takes four at a time).  Not fp64 beside a b that runs along too, where the additional registers cost more than the wide loads
// give: us, wide / not, 10,000 rows of 1000 29.5 / 27.7, 5000 of 3000 37.0 / 36.1, 1100 of 14712 38.9 / 40.1; fp32 18.7 / 18.4, 23.1 / 23.2,
// 24.6 / 25.5, 300 rows of 65000 28.4 / 30.8.
bool wide_rows(size_t es, int64_t Q, int64_t Lin, int64_t sa, const void* b, int64_t sb) {
  return (Q == 1 || Lin > 1024) && sa == 1 && (!b || sb == 0 || (sb == 1 && es == 4));
}
template <typename TI, typename A, bool HASB, bool WIDE>
__device__ __forceinline__ A row_sum(const TI* __restrict__ pa, const TI* __restrict__ pb, int64_t sa, int64_t sb, int64_t j0, int64_t j1, int lane) {
  if constexpr (WIDE && std::is_floating_point<TI>::value) {
    if (j1 - j0 >= 4096 / (int64_t)sizeof(TI)) return wide_sum<TI, A, HASB>(pa, pb, sb, j0, j1, lane);
  }
  return lane_strided_sum<TI, A, HASB>(pa, pb, sa, sb, j0 + lane, j1);
}

// (32-bit indices)
template <typename D>
__device__ __forceinline__ void decompose_small(const D& d, uint32_t r, int64_t& oa, int64_t& ob) {
  oa = ob = 0;
  for (int i = d.nd - 1; i > 0; --i) {
    const uint32_t s = (uint32_t)d.shape[i], q = r / s, c = r - q * s;
    r = q;
    oa += (int64_t)c * d.st[0][i];
    ob += (int64_t)c * d.st[1][i];
  }
  oa += (int64_t)r * d.st[0][0];
  ob += (int64_t)r * d.st[1][0];
}

// Sum over the elements f = first, first + step, ... < f1 of rows that lie in one (row f / Lin, element f % Lin): rows shorter than a
// wavefront, which would leave lanes idle, four elements a lane in flight.  us, before / so: 300 sums of 10,000 rows of 6 fp64
// 1121 / 74, of 2000 rows of 32 231 / 45, 36 of 168 rows of 24 (four to a launch) 5.6 / 3.2, 500 of 500 rows of 30 33.4 / 14.5.
// (Rows of 64 and more fill the wavefront, and an index less to find for each element counts once the memory is what bounds it.)
template <typename TI, typename A, bool HASB, typename D>
__device__ __forceinline__ A flat_sum(const D& red, uint32_t Lin, const TI* __restrict__ a, const TI* __restrict__ b, int64_t sa_in, int64_t sb_in, uint32_t first, uint32_t step, uint32_t f1) {
  constexpr uint32_t U = 4;
  A c[U] = {0, 0, 0, 0};
  for (uint32_t f = first; f < f1; f += U * step) {
    A x[U], y[U];
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
      const bool in = f + u * step < f1;
      const uint32_t g = in ? f + u * step : f, q = g / Lin, j = g - q * Lin;
      int64_t oa, ob;
      decompose_small(red, q, oa, ob);
      x[u] = (A)a[oa + j * sa_in];
      if (!in) x[u] = 0;
      if (HASB) y[u] = in ? (A)b[ob + j * sb_in] : (A)0;
    }
#pragma unroll
    for (uint32_t u = 0; u < U; ++u) {
      if (HASB) x[u] *= y[u];
      c[u] += x[u];
    }
  }
  return (c[0] + c[1]) + (c[2] + c[3]);
}
// (indices up to f1 + 4 * step are formed)
__device__ __forceinline__ bool flat_rows(int64_t Q, int64_t Lin) { return Q > 1 && Lin < 64 && Q * Lin < ((int64_t)1 << 30); }

// Sum over the rows q = first, first + step, ... < q1, four at a time where they are short, so that a lane has four loads per operand
// in flight although a row gives it only a few elements.
template <typename TI, typename A, bool HASB, bool WIDE, typename D>
__device__ __forceinline__ A rows_sum(const D& red, int64_t first, int64_t step, int64_t q1, const TI* __restrict__ a, const TI* __restrict__ b, int64_t sa_in, int64_t sb_in,
                                      int64_t j0, int64_t j1, bool in_fours, int lane) {
  A acc = 0;
  int64_t q = first;
  if (!WIDE && in_fours) {
    for (; q + 3 * step < q1; q += 4 * step) {
      const TI* pa[4];
      const TI* pb[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        int64_t oa, ob;
        decompose_small(red, (uint32_t)(q + u * step), oa, ob);
        pa[u] = a + oa;
        pb[u] = HASB ? b + ob : nullptr;
      }
      A c[4] = {0, 0, 0, 0};
      for (int64_t j = j0 + lane; j < j1; j += 64) {
        A x[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = (A)pa[u][j * sa_in];
        if (HASB) {
#pragma unroll
          for (int u = 0; u < 4; ++u) x[u] *= (A)pb[u][j * sb_in];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) c[u] += x[u];
      }
      acc += (c[0] + c[1]) + (c[2] + c[3]);
    }
  }
  for (; q < q1; q += step) {
    int64_t ro[2];
    decompose<2>(red, q, ro);
    acc += row_sum<TI, A, HASB, WIDE>(a + ro[0], HASB ? b + ro[1] : nullptr, sa_in, sb_in, j0, j1, lane);
  }
  return acc;
}

// One wavefront per work item.  `red` has its innermost dim split off:
// Lin = extent, (sa_in, sb_in) = strides; `red` keeps the outer reduced dims
// with Q = their product.  Chunks split Q when Q > 1, else Lin.
template <typename TI, typename TO, bool HASB, bool WIDE, typename D>
__device__ __forceinline__ void wave_body(const D& keep, const D& red, int64_t n_out, int64_t Q, int64_t Lin, int64_t sa_in, int64_t sb_in,
                                          int S, int64_t chunk, const TI* __restrict__ a0, const TI* __restrict__ b0, TO* __restrict__ out, const TermPtrs* tp, unsigned bid, unsigned nb) {
  using A = typename acc_of<TI>::type;
  const int lane = threadIdx.x & 63;
  int64_t wave = ((int64_t)bid * kBlock + threadIdx.x) >> 6;
  int64_t nwaves = ((int64_t)nb * kBlock) >> 6;
  int64_t items = n_out * S;
  for (int64_t item = wave; item < items; item += nwaves) {
    int64_t o = item / S;
    int s = (int)(item - o * S);
    const TI* a = a0;
    const TI* b = b0;
    if (tp && tp->n) {
      int term = s / tp->s_per;
      s -= term * tp->s_per;
      a = (const TI*)tp->a[term];
      b = (const TI*)tp->b[term];
    }
    int64_t ko[2];
    decompose<2>(keep, o, ko);
    int64_t q0 = 0, q1 = Q, j0 = 0, j1 = Lin;
    if (Q > 1) { q0 = s * chunk; q1 = q0 + chunk; if (q1 > Q) q1 = Q; }
    else { j0 = s * chunk; j1 = j0 + chunk; if (j1 > Lin) j1 = Lin; }
    const TI *pa = a + ko[0], *pb = HASB ? b + ko[1] : nullptr;
    A acc;
    if (!WIDE && flat_rows(Q, Lin)) acc = flat_sum<TI, A, HASB>(red, (uint32_t)Lin, pa, pb, sa_in, sb_in, (uint32_t)(q0 * Lin) + lane, 64, q1 > q0 ? (uint32_t)(q1 * Lin) : 0);
    else acc = rows_sum<TI, A, HASB, WIDE>(red, q0, 1, q1, pa, pb, sa_in, sb_in, j0, j1, Lin <= 1024 && Q <= INT32_MAX, lane);
    acc = wave_sum<A>(acc);
    if (lane == 0) out[item] = (TO)acc;
  }
}
template <typename TI, typename TO, bool HASB, bool WIDE>
__global__ void __launch_bounds__(kBlock) k_contract_wave(Dims keep, Dims red, int64_t n_out, int64_t Q, int64_t Lin, int64_t sa_in, int64_t sb_in,
                                                           int S, int64_t chunk, const TI* __restrict__ a0, const TI* __restrict__ b0, TO* __restrict__ out, TermPtrs tp) {
  wave_body<TI, TO, HASB, WIDE>(keep, red, n_out, Q, Lin, sa_in, sb_in, S, chunk, a0, b0, out, &tp, blockIdx.x, gridDim.x);
}

// One block of four wavefronts per output: for a few hundred outputs with a few
// thousand reduced elements each, where one wavefront per output leaves most of
// the device idle and splitting into chunks would cost a second launch.  The
// wavefronts take every fourth outer reduced index (or a quarter of the inner
// dim when there is no outer one; the lanes every 256th element of short rows)
// and combine through LDS in a fixed order.
template <typename TI, typename TO, bool HASB, bool WIDE, typename D>
__device__ __forceinline__ void block_body(const D& keep, const D& red, int64_t n_out, int64_t Q, int64_t Lin, int64_t sa_in, int64_t sb_in,
                                           const TI* __restrict__ a, const TI* __restrict__ b, TO* __restrict__ out, unsigned bid, unsigned nb) {
  using A = typename acc_of<TI>::type;
  __shared__ A part[kBlock / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  constexpr int NW = kBlock / 64;
  for (int64_t o = bid; o < n_out; o += nb) {
    int64_t ko[2];
    decompose<2>(keep, o, ko);
    const TI *pa = a + ko[0], *pb = HASB ? b + ko[1] : nullptr;
    A acc = 0;
    if (!WIDE && flat_rows(Q, Lin)) {
      acc = flat_sum<TI, A, HASB>(red, (uint32_t)Lin, pa, pb, sa_in, sb_in, threadIdx.x, kBlock, (uint32_t)(Q * Lin));
    } else if (Q > 1) {
      acc = rows_sum<TI, A, HASB, WIDE>(red, w, NW, Q, pa, pb, sa_in, sb_in, 0, Lin, Lin <= 1024 && Q <= INT32_MAX, lane);
    } else {
      const int64_t quarter = (Lin + NW - 1) / NW;
      const int64_t j0 = w * quarter, j1 = j0 + quarter < Lin ? j0 + quarter : Lin;
      acc = row_sum<TI, A, HASB, WIDE>(pa, pb, sa_in, sb_in, j0, j1, lane);
    }
    acc = wave_sum<A>(acc);
    if (lane == 0) part[w] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
      A t = part[0];
#pragma unroll
      for (int k = 1; k < NW; ++k) t += part[k];
      out[o] = (TO)t;
    }
    __syncthreads();
  }
}
template <typename TI, typename TO, bool HASB, bool WIDE>
__global__ void __launch_bounds__(kBlock) k_contract_block(Dims keep, Dims red, int64_t n_out, int64_t Q, int64_t Lin, int64_t sa_in, int64_t sb_in,
                                                            const TI* __restrict__ a, const TI* __restrict__ b, TO* __restrict__ out) {
  block_body<TI, TO, HASB, WIDE>(keep, red, n_out, Q, Lin, sa_in, sb_in, a, b, out, blockIdx.x, gridDim.x);
}

// Sums the partial results of a split reduction: out[i] = sum_s part[s * stride + i].  A block owns
// OPB consecutive outputs; its 256 / OPB groups of lanes each take every
// (256 / OPB)-th partial (coalesced rows of OPB elements), several loads in
// flight at a time, and combine through LDS in a fixed order.  Few outputs get
// the narrow blocks: more of them, and fewer partials for a lane to walk through.
struct SumArgs {
  const void* part;
  const void* other;  // kSumPair: the second of two
  void* out;
  void* out2;         // outputs from n1 on
  int64_t n, n1, stride;
  int S, kind;
  unsigned grid, pad_;
};

template <typename T, int OPB>
__device__ __forceinline__ void partials_body(const SumArgs& a, unsigned bid, unsigned nb) {
  constexpr int G = 256 / OPB;
  __shared__ T red[G][OPB + 1];
  const T* __restrict__ part = (const T*)a.part;
  const int ol = threadIdx.x % OPB, g = threadIdx.x / OPB;
  for (int64_t base = (int64_t)bid * OPB; base < a.n; base += (int64_t)nb * OPB) {
    int64_t i = base + ol;
    T acc = T(0);
    if (i < a.n) {
#pragma unroll 8
      for (int s = g; s < a.S; s += G) acc += part[(int64_t)s * a.stride + i];
    }
    red[g][ol] = acc;
    __syncthreads();
    if (g == 0 && i < a.n) {
      T t = red[0][ol];
#pragma unroll
      for (int k = 1; k < G; ++k) t += red[k][ol];
      if (i < a.n1) ((T*)a.out)[i] = t;
      else ((T*)a.out2)[i - a.n1] = t;
    }
    __syncthreads();
  }
}

// The same sum with an output per lane: for a handful of partials (S <= 8), where the blocks above would leave most of
// their lane groups without one, and for many outputs, where they would go around several times and wait for their loads
// each time (300 x 784 outputs of 15 fp64 partials with five other problems of a group: 23.7 us in such blocks, 18.2 so; 2048 x 784 of 9
// fp32 ones, 4.5 to launch among them, 22 and 16).  Up to eight are added one after another (0 + p0 + p1 + ...),
// more of them in eight interleaved chains, eight to fifteen loads in flight.  (Chains as short as those of the blocks above, which meet
// in pairs: the error is 0.8 to 0.9 of theirs; four chains and the rest of S one after another had 1.1 to 1.5 of it.)
template <typename T>
__device__ __forceinline__ void partials_lane_body(const SumArgs& g, unsigned bid, unsigned nb) {
  const int64_t step = (int64_t)nb * 256;
  auto put = [&](int64_t i, T v) {
    if (i < g.n1) ((T*)g.out)[i] = v;
    else ((T*)g.out2)[i - g.n1] = v;
  };
  const int64_t first = (int64_t)bid * 256 + threadIdx.x;
  // (Two loops, the end of S asked for first: in one loop, and with the end behind the eights, an output's loads waited for the
  // store of the one before.  2048 x 784 of 9 and 2048 x 2048 of 2 fp32 partials in one launch, us: 39.4, so 32.3.)
  if (g.S <= 8) {
    for (int64_t i = first; i < g.n; i += step) {
      const T* p = (const T*)g.part + i;
      T x[8], acc = T(0);
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = u == 0 || u < g.S ? p[(int64_t)u * g.stride] : T(0);      // (a sum that begins with +0 is never -0)
#pragma unroll
      for (int u = 0; u < 8; ++u) acc += x[u];
      put(i, acc);
    }
    return;
  }
  const int whole = g.S / 8 * 8;
  for (int64_t i = first; i < g.n; i += step) {
    const T* p = (const T*)g.part + i;
    T x[8], rest[8], c[8] = {};
#pragma unroll
    for (int u = 0; u < 8; ++u) rest[u] = whole + u < g.S ? p[(int64_t)(whole + u) * g.stride] : T(0);
    for (int s = 0; s < whole; s += 8) {
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = p[(int64_t)(s + u) * g.stride];
#pragma unroll
      for (int u = 0; u < 8; ++u) c[u] += x[u];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) c[u] += rest[u];
    put(i, ((c[0] + c[4]) + (c[2] + c[6])) + ((c[1] + c[5]) + (c[3] + c[7])));
  }
}

// Partial sums in doubles that lie side by side, S for an output: a wavefront per output.
template <typename T>
__device__ __forceinline__ void partials_row_body(const SumArgs& g, unsigned bid, unsigned nb) {
  const int lane = threadIdx.x & 63;
  const int64_t nwaves = ((int64_t)nb * kBlock) >> 6;
  for (int64_t o = ((int64_t)bid * kBlock + threadIdx.x) >> 6; o < g.n; o += nwaves) {
    const double* p = (const double*)g.part + o * g.S;
    double acc = lane_strided_sum<double, double, false>(p, nullptr, 1, 0, lane, g.S);
    acc = wave_sum<double>(acc);
    if (lane == 0) ((T*)g.out)[o] = (T)acc;
  }
}

// Two results that are added up, the first dense: vectors of 16 bytes where both start at multiples of that.  A second one
// that is a view (a row's sum, repeated along the row) has rows of n1 elements, `stride` apart, their elements S apart.
template <typename T>
__device__ __forceinline__ void pair_body(const SumArgs& g, unsigned bid, unsigned nb) {
  constexpr int V = 16 / sizeof(T);
  typedef T Vec __attribute__((ext_vector_type(V)));
  const T *a = (const T*)g.part, *b = (const T*)g.other;
  T* o = (T*)g.out;
  const int64_t at = (int64_t)bid * 256 + threadIdx.x, step = (int64_t)nb * 256;
  if (g.n1 != g.n) {
    for (int64_t i = at; i < g.n; i += step) {
      const int64_t r = i / g.n1;
      o[i] = a[i] + b[r * g.stride + (i - r * g.n1) * g.S];
    }
    return;
  }
  const bool wide = (((uintptr_t)a | (uintptr_t)b | (uintptr_t)o) & 15) == 0;
  const int64_t nv = wide ? g.n / V : 0;
  for (int64_t i = at; i < nv; i += step) ((Vec*)o)[i] = ((const Vec*)a)[i] + ((const Vec*)b)[i];
  for (int64_t i = nv * V + at; i < g.n; i += step) o[i] = a[i] + b[i];
}

// See try_tiny_map.
template <typename T>
__device__ __forceinline__ void tiny_body(const SumArgs& g) {
#pragma clang fp contract(off)
  if (threadIdx.x >= g.n) return;
  const uint64_t code = (uint64_t)g.stride;
  T v[6];
  v[0] = ((const T*)g.part)[code >> 48 & 1 ? threadIdx.x : 0];
  v[1] = ((const T*)g.other)[code >> 49 & 1 ? threadIdx.x : 0];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    v[2 + k] = k > 0 ? v[1 + k] : v[0];
    if (k >= g.S) continue;
    const unsigned q = (unsigned)(code >> (12 * k)) & 0xfff, op = q & 15;
    T x = v[0], y = v[0];
#pragma unroll
    for (int u = 1; u < 2 + k; ++u) {
      if ((q >> 4 & 15) == (unsigned)u) x = v[u];
      if ((q >> 8 & 15) == (unsigned)u) y = v[u];
    }
    v[2 + k] = op == 0 ? -x : op == 1 ? x + y : op == 2 ? x - y : x * y;
  }
  ((T*)g.out)[threadIdx.x] = v[5];
}

template <typename T>
__device__ __forceinline__ void sum_body(const SumArgs& s, unsigned bid) {
  if (s.kind == RedJob::kSumTiny) tiny_body<T>(s);
  else if (s.kind == RedJob::kSumPair) pair_body<T>(s, bid, s.grid);
  else if (s.kind == RedJob::kSumRows) partials_row_body<T>(s, bid, s.grid);
  else if (s.kind == RedJob::kSumLane) partials_lane_body<T>(s, bid, s.grid);
  else if (s.kind == RedJob::kSum32) partials_body<T, 32>(s, bid, s.grid);
  else partials_body<T, 8>(s, bid, s.grid);
}

template <typename T, int KIND>
__global__ void __launch_bounds__(kBlock) k_sum_partials(SumArgs s) {
  if (KIND == RedJob::kSumTiny) tiny_body<T>(s);
  else if (KIND == RedJob::kSumPair) pair_body<T>(s, blockIdx.x, gridDim.x);
  else if (KIND == RedJob::kSumRows) partials_row_body<T>(s, blockIdx.x, gridDim.x);
  else if (KIND == RedJob::kSumLane) partials_lane_body<T>(s, blockIdx.x, gridDim.x);
  else if (KIND == RedJob::kSum32) partials_body<T, 32>(s, blockIdx.x, gridDim.x);
  else partials_body<T, 8>(s, blockIdx.x, gridDim.x);
}

// Up to four single-launch reductions and twelve sums of partial results of one element type as one kernel: the first
// blocks are problem 0's, the next ones problem 1's, ...; every block runs the code of the kernel its problem would have
// been launched with.  A launch costs 4.5 to 5 us in a recorded graph however little it does, and nobody waits for the
// sums of a reverse pass.  Gradients, us, each sum as a launch of its own / so: two recurrent layers of width 128 over 28 steps,
// fp32 batch 5000 636 / 608, fp64 batch 150 319 / 303; CNN 28 x 28 fp64 batch 1000 327 / 320, its training step at batch 250
// fp32 152 / 144; dense 784-300-100-10 fp64 batch 5000 214 / 209; wide dense network fp32 1730 / 1720.
struct RedArgs {
  Dims2 keep, red;
  int64_t n_out, R, Q, Lin, sa, sb, chunk;
  int variant, hasb;
  unsigned grid, pad_;
  const void* a;
  const void* b;
  void* out;
};
struct RedGroup {
  int n, n_sums;
  RedArgs j[kMaxGroupReductions];
  SumArgs s[kMaxGroupSums];
};
static_assert(sizeof(RedGroup) <= 4000, "the grouped reduction's arguments must fit the kernel argument block");

template <typename T>
__global__ void __launch_bounds__(kBlock) k_contract_group(RedGroup args) {
  // read where the launch has put it: with this many uses of a by-value argument the compiler copies all of it to every lane's memory
  // (3248 bytes of scratch; 1500 sums of 30 rows of 28, four to a launch: 5.9 -> 63.7 us)
  const RedGroup& g = *(const RedGroup*)__builtin_amdgcn_kernarg_segment_ptr();
  unsigned bid = blockIdx.x;
  int k = 0;
  while (k < g.n && bid >= g.j[k].grid) { bid -= g.j[k].grid; ++k; }
  if (k == g.n) {
    k = 0;
    while (k < g.n_sums - 1 && bid >= g.s[k].grid) { bid -= g.s[k].grid; ++k; }
    sum_body<T>(g.s[k], bid);
    return;
  }
  const RedArgs& r = g.j[k];
  const T* a = (const T*)r.a;
  const T* b = (const T*)r.b;
  T* out = (T*)r.out;
  if (r.variant == 0) {
    if (r.hasb) block_body<T, T, true, false>(r.keep, r.red, r.n_out, r.Q, r.Lin, r.sa, r.sb, a, b, out, bid, r.grid);
    else block_body<T, T, false, false>(r.keep, r.red, r.n_out, r.Q, r.Lin, r.sa, r.sb, a, b, out, bid, r.grid);
  } else if (r.variant == 1) {
    if (r.hasb) wave_body<T, T, true, false>(r.keep, r.red, r.n_out, r.Q, r.Lin, r.sa, r.sb, 1, r.chunk, a, b, out, nullptr, bid, r.grid);
    else wave_body<T, T, false, false>(r.keep, r.red, r.n_out, r.Q, r.Lin, r.sa, r.sb, 1, r.chunk, a, b, out, nullptr, bid, r.grid);
  } else {
    if (r.hasb) lane_body<T, T, true>(r.keep, r.red, r.n_out, r.R, 1, r.chunk, a, b, out, nullptr, bid, r.grid);
    else lane_body<T, T, false>(r.keep, r.red, r.n_out, r.R, 1, r.chunk, a, b, out, nullptr, bid, r.grid);
  }
}

// First (want_max = 0: minimal, 1: maximal) element along the last dim.
template <typename T>
__global__ void __launch_bounds__(kBlock) k_argminmax(Dims keep, int64_t n_out, int64_t L, int64_t sl, int want_max, const T* __restrict__ a, int64_t* __restrict__ out, T* __restrict__ vals) {
  int64_t step = (int64_t)gridDim.x * kBlock;
  for (int64_t o = (int64_t)blockIdx.x * kBlock + threadIdx.x; o < n_out; o += step) {
    int64_t ko[1];
    decompose<1>(keep, o, ko);
    const T* p = a + ko[0];
    T best = p[0];
    int64_t bi = 0;
    for (int64_t j = 1; j < L; ++j) {
      T x = p[j * sl];
      bool better = want_max ? (x > best) : (x < best);
      if (better) { best = x; bi = j; }
    }
    out[o] = bi;
    if (vals) vals[o] = best;
  }
}

// Where a row's elements are shared out between lanes: a NaN is neither greater nor smaller than anything, so it is no
// candidate (bi stays INT64_MAX until a number comes), but in the first place of its row, where it stays.
template <typename T>
__device__ __forceinline__ bool takes(T x, T best, int64_t bi, int want_max) {
  return bi == INT64_MAX ? x == x : (want_max ? (x > best) : (x < best));
}
template <typename T>
__device__ __forceinline__ void put_extremum(T first, T best, int64_t bi, int64_t* out, T* val) {
  const bool keep_first = !(first == first);
  *out = keep_first ? 0 : bi;
  if (val) *val = keep_first ? first : best;
}

// The same with one wavefront per row, for long rows: every lane scans a
// strided subsequence keeping its first extremum, then lanes combine; on equal
// values the smaller index wins, which keeps "first occurrence".
template <typename T>
__global__ void __launch_bounds__(kBlock) k_argminmax_wave(Dims keep, int64_t n_out, int64_t L, int64_t sl, int want_max, const T* __restrict__ a, int64_t* __restrict__ out, T* __restrict__ vals) {
  const int lane = threadIdx.x & 63;
  int64_t wave = ((int64_t)blockIdx.x * kBlock + threadIdx.x) >> 6;
  int64_t nwaves = ((int64_t)gridDim.x * kBlock) >> 6;
  for (int64_t o = wave; o < n_out; o += nwaves) {
    int64_t ko[1];
    decompose<1>(keep, o, ko);
    const T* p = a + ko[0];
    T best = T(0);
    int64_t bi = INT64_MAX;
    for (int64_t j = lane; j < L; j += 64) {
      T x = p[j * sl];
      if (takes(x, best, bi, want_max)) { best = x; bi = j; }
    }
    for (int off = 32; off > 0; off >>= 1) {
      long long o_bi = __shfl_down((long long)bi, off, 64);
      T o_best;
      if constexpr (sizeof(T) == 8) {
        unsigned long long u = *reinterpret_cast<unsigned long long*>(&best);
        unsigned lo = __shfl_down((unsigned)(u & 0xffffffffu), off, 64);
        unsigned hi = __shfl_down((unsigned)(u >> 32), off, 64);
        unsigned long long w = ((unsigned long long)hi << 32) | lo;
        o_best = *reinterpret_cast<T*>(&w);
      } else if constexpr (sizeof(T) == 4) {
        unsigned u = *reinterpret_cast<unsigned*>(&best);
        unsigned w = __shfl_down(u, off, 64);
        o_best = *reinterpret_cast<T*>(&w);
      } else {
        int w = __shfl_down((int)best, off, 64);
        o_best = (T)w;
      }
      if (o_bi != INT64_MAX && (takes(o_best, best, bi, want_max) || (o_best == best && o_bi < bi))) { best = o_best; bi = o_bi; }
    }
    if (lane == 0) put_extremum(p[0], best, bi, out + o, vals ? vals + o : nullptr);
  }
}

// One block of 1024 lanes per row, for a few very long rows (the minimum of a
// whole tensor): lanes scan strided subsequences, then combine through LDS with
// the same "smaller index wins ties" rule.
template <typename T>
__global__ void __launch_bounds__(1024) k_argminmax_block(Dims keep, int64_t L, int64_t sl, int want_max, const T* __restrict__ a, int64_t* __restrict__ out, T* __restrict__ vals) {
  __shared__ T sbest[1024];
  __shared__ int64_t sidx[1024];
  int64_t ko[1];
  decompose<1>(keep, blockIdx.x, ko);
  const T* p = a + ko[0];
  const int t = threadIdx.x;
  T best = t < L ? p[(int64_t)t * sl] : T(0);
  int64_t bi = t < L && best == best ? t : INT64_MAX;
  // eight loads in flight; the comparisons keep the order of the positions
  int64_t j = (int64_t)t + 1024;
  for (; j + 7 * 1024 < L; j += 8 * 1024) {
    T x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) x[u] = p[(j + u * 1024) * sl];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (takes(x[u], best, bi, want_max)) { best = x[u]; bi = j + u * 1024; }
    }
  }
  for (; j < L; j += 1024) {
    T x = p[j * sl];
    if (takes(x, best, bi, want_max)) { best = x; bi = j; }
  }
  sbest[t] = best;
  sidx[t] = bi;
  __syncthreads();
  for (int off = 512; off > 0; off >>= 1) {
    if (t < off) {
      T ob = sbest[t + off];
      int64_t oi = sidx[t + off];
      if (oi != INT64_MAX) {
        bool mine = sidx[t] != INT64_MAX;
        bool better = !mine || (want_max ? (ob > sbest[t]) : (ob < sbest[t])) || (ob == sbest[t] && oi < sidx[t]);
        if (better) { sbest[t] = ob; sidx[t] = oi; }
      }
    }
    __syncthreads();
  }
  if (t == 0) put_extremum(p[0], sbest[0], sidx[0], out + blockIdx.x, vals ? vals + blockIdx.x : nullptr);
}

// A few very long rows whose data one CU cannot fetch fast enough (a block
// draws some tens of GB/s): G blocks per row scan consecutive pieces, then one
// wavefront per row, of the block that finishes last (`tickets`: a counter per row, 128 bytes apart, zero between launches),
// picks among the G candidates, the earlier piece winning ties.  The candidates travel as the
// partial sums of the fused sums do: exchanged in by atomics of device scope, the returned value says that they have arrived,
// then the ticket is drawn.  One row of 50,000 fp64: 9.9 us in two launches, 7.3 in one, with 48 pieces for 24 6.6.
// The extremum of a row among its G candidates, by one wavefront.
template <typename T, typename V, typename I>
__device__ __forceinline__ void pick_body(int G, int want_max, const V& value_of, const I& index_of, T first, int64_t* __restrict__ out, T* __restrict__ vals) {
  const int lane = threadIdx.x & 63;
  T best = T(0);
  int64_t bi = INT64_MAX;
  for (int g = lane; g < G; g += 64) {
    T x = value_of(g);
    int64_t xi = index_of(g);
    if (xi == INT64_MAX) continue;
    bool better = bi == INT64_MAX || (want_max ? (x > best) : (x < best));    // pieces of a lane come in ascending order
    if (better) { best = x; bi = xi; }
  }
  for (int off = 32; off > 0; off >>= 1) {
    T ob = __shfl_down(best, off);
    int64_t oi = __shfl_down(bi, off);
    if (oi != INT64_MAX) {
      bool better = bi == INT64_MAX || (want_max ? (ob > best) : (ob < best)) || (ob == best && oi < bi);
      if (better) { best = ob; bi = oi; }
    }
  }
  if (lane == 0) put_extremum(first, best, bi, out, vals);
}
template <typename T>
__global__ void __launch_bounds__(kBlock) k_argminmax_pieces(Dims keep, int64_t L, int64_t sl, int want_max, int G, int64_t piece, const T* __restrict__ a,
                                                              unsigned long long* handed, unsigned* tickets, int64_t* __restrict__ out, T* __restrict__ vals) {
  __shared__ T sbest[kBlock];
  __shared__ int64_t sidx[kBlock];
  const int row = blockIdx.x / G, g = blockIdx.x % G;
  int64_t ko[1];
  decompose<1>(keep, row, ko);
  const T* p = a + ko[0];
  const int t = threadIdx.x;
  const int64_t j0 = (int64_t)g * piece, j1 = j0 + piece < L ? j0 + piece : L;
  T best = T(0);
  int64_t bi = INT64_MAX;
  int64_t j = j0 + t;
  for (; j + 3 * kBlock < j1; j += 4 * kBlock) {
    T x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) x[u] = p[(j + u * kBlock) * sl];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (takes(x[u], best, bi, want_max)) { best = x[u]; bi = j + u * kBlock; }
    }
  }
  for (; j < j1; j += kBlock) {
    T x = p[j * sl];
    if (takes(x, best, bi, want_max)) { best = x; bi = j; }
  }
  sbest[t] = best;
  sidx[t] = bi;
  __syncthreads();
  for (int off = kBlock / 2; off > 0; off >>= 1) {
    if (t < off) {
      T ob = sbest[t + off];
      int64_t oi = sidx[t + off];
      if (oi != INT64_MAX) {
        bool mine = sidx[t] != INT64_MAX;
        bool better = !mine || (want_max ? (ob > sbest[t]) : (ob < sbest[t])) || (ob == sbest[t] && oi < sidx[t]);
        if (better) { sbest[t] = ob; sidx[t] = oi; }
      }
    }
    __syncthreads();
  }
  __shared__ bool last;
  if (t == 0) {
    unsigned long long bits = 0;
    __builtin_memcpy(&bits, &sbest[0], sizeof(T));
    const unsigned long long v = __hip_atomic_exchange(handed + 2 * blockIdx.x, bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const unsigned long long i = __hip_atomic_exchange(handed + 2 * blockIdx.x + 1, (unsigned long long)sidx[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("" :: "v"(v), "v"(i) : "memory");      // uses of the returned values: nothing below starts before they are there
    unsigned* ticket = tickets + 32 * row;
    last = __hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)G - 1;
    if (last) __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);      // for the next launch
  }
  __syncthreads();
  if (!last || t >= 64) return;
  asm volatile("" ::: "memory");
  auto load = [&](int at) { return __hip_atomic_load(handed + 2 * (int64_t)row * G + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
  pick_body<T>(G, want_max, [&](int c) { const unsigned long long u = load(2 * c); T x; __builtin_memcpy(&x, &u, sizeof(T)); return x; },
               [&](int c) { return (int64_t)load(2 * c + 1); }, p[0], out + row, vals ? vals + row : nullptr);
}

// A few very long rows, in pieces: see k_argminmax_pieces (the caller's guard is held; `scratch` holds 16 bytes per piece).
// (One row of 10,000 fp64: ten pieces 6.6 us, one block of 1024 lanes 6.4.)
constexpr int64_t kPiecesFrom = 16384, kPiece = 1024, kPiecesRows = 16;
int pieces_of(int64_t L) { return (int)std::min<int64_t>(128, L / kPiece); }
template <typename T>
void extremum_pieces(hgpu_ctx* ctx, const Dims& keep, int64_t n_out, int64_t L, int64_t sl, int want_max, const void* a, void* scratch, unsigned* tickets, void* out, void* vp) {
  const int G = pieces_of(L);
  const int64_t piece = (L + G - 1) / G;
  hipLaunchKernelGGL(k_argminmax_pieces<T>, dim3((unsigned)(n_out * G)), dim3(kBlock), 0, ctx->stream, keep, L, sl, want_max, G, piece, (const T*)a,
                     (unsigned long long*)scratch, tickets, (int64_t*)out, (T*)vp);
}

// The buffers of a reduction whose launch may be held back (see RedJob): what it reads and what it writes.
struct HoldBufs { hgpu_buffer* a; hgpu_buffer* b; hgpu_buffer* out; };

template <typename TI, typename TO>
int launch_stage(hgpu_ctx* ctx, bool use_wave, const Dims& keep, const Dims& red_full, int64_t n_out, int64_t R, int S, const void* a, const void* b, void* out,
                 const TermPtrs* terms = nullptr, const HoldBufs* hold = nullptr, int dtype = -1, bool fresh = true) {
  // with terms, S counts the chunks of all of them; each term is cut into s_per
  // (fresh: out is a new array, see LaunchGuard)
  TermPtrs tp;
  tp.n = 0;
  tp.s_per = S;
  if (terms) tp = *terms;
  const int S_per = tp.n ? tp.s_per : S;
  const char* label = b ? (use_wave ? "contract_dot_wave" : "contract_dot_lane") : (use_wave ? "contract_sum_wave" : "contract_sum_lane");
  if (ctx->profiling && ctx->profile_shapes) {
    char buf[160];
    int n = snprintf(buf, sizeof buf, "%s[out%lld,R%lld,S%d,red", label, (long long)n_out, (long long)R, S);
    for (int i = 0; i < red_full.nd && n < (int)sizeof buf - 40; ++i)
      n += snprintf(buf + n, sizeof buf - n, "_%lld:%lld/%lld", (long long)red_full.shape[i], (long long)red_full.st[0][i], (long long)red_full.st[1][i]);
    n += snprintf(buf + n, sizeof buf - n, ",keep");
    for (int i = 0; i < keep.nd && n < (int)sizeof buf - 40; ++i)
      n += snprintf(buf + n, sizeof buf - n, "_%lld:%lld/%lld", (long long)keep.shape[i], (long long)keep.st[0][i], (long long)keep.st[1][i]);
    snprintf(buf + n, sizeof buf - n, "]");
    label = intern_label(ctx, buf);
  }
  const double nterms = tp.n ? tp.n : 1;
  // algorithmic bytes: every operand's distinct elements once (an operand that stands still along a dim is not read again along it)
  auto distinct = [&](int k) {
    double n = 1;
    for (int i = 0; i < keep.nd; ++i) if (keep.st[k][i] != 0) n *= (double)keep.shape[i];
    for (int i = 0; i < red_full.nd; ++i) if (red_full.st[k][i] != 0) n *= (double)red_full.shape[i];
    return n;
  };
  const double bytes = (distinct(0) + (b ? distinct(1) : 0.0)) * sizeof(TI) * nterms + (double)n_out * (S > 0 ? S : 1) * sizeof(TO),
               flops = (double)n_out * R * (b ? 2 : 1) * nterms;
  int maxb = ctx->num_cu * 8;
  // A single-launch reduction of at most eight million terms is held back: the next ones that do not read its result share its launch.
  if (hold && !terms && S <= 1 && std::is_same<TI, TO>::value && (double)n_out * (double)R <= 8.0e6) {
    RedJob j;
    j.dtype = dtype;
    j.hasb = b ? 1 : 0;
    j.keep = keep;
    j.red = red_full;
    j.n_out = n_out;
    j.R = R;
    j.a = a;
    j.b = b;
    j.out = out;
    j.label = label;
    j.bytes = bytes;
    j.flops = flops;
    if (use_wave) {
      int last = j.red.nd - 1;
      j.Lin = j.red.shape[last];
      j.sa = j.red.st[0][last];
      j.sb = j.red.st[1][last];
      j.Q = R / j.Lin;
      if (j.red.nd > 1) { j.red.nd -= 1; } else { j.red.shape[0] = 1; j.red.st[0][0] = j.red.st[1][0] = 0; }
      if (S == 0) {
        j.variant = 0;
        j.grid = (unsigned)(n_out < (int64_t)maxb ? n_out : maxb);
      } else {
        j.variant = 1;
        j.chunk = j.Q > 1 ? j.Q : j.Lin;
        j.grid = grid_for(n_out * 64, kBlock, maxb);
      }
    } else {
      j.variant = 2;
      j.chunk = R;
      j.grid = grid_for(n_out, kBlock, maxb);
    }
    hgpu_buffer* reads[2] = {hold->a, hold->b};
    if (hold_reduction(ctx, j, reads, hold->b ? 2 : 1, hold->out)) return HGPU_OK;
  }
  Reads reads{a, b};
  if (tp.n) {
    reads.add(tp.a, tp.a + tp.n);
    reads.add(tp.b, tp.b + tp.n);
  }
  LaunchGuard lg(ctx, label, bytes, flops, fresh ? &reads : nullptr);
  if (use_wave && S == 0) {       // one block per output, no partials
    Dims red = red_full;
    int last = red.nd - 1;
    int64_t Lin = red.shape[last], sa = red.st[0][last], sb = red.st[1][last];
    int64_t Q = R / Lin;
    if (red.nd > 1) { red.nd -= 1; } else { red.shape[0] = 1; red.st[0][0] = red.st[1][0] = 0; }
    unsigned g = (unsigned)(n_out < (int64_t)maxb ? n_out : maxb);
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(g), dim3(kBlock), 0, ctx->stream, keep, red, n_out, Q, Lin, sa, sb, (const TI*)a, (const TI*)b, (TO*)out); };
    const bool wide = wide_rows(sizeof(TI), Q, Lin, sa, b, sb);
    if (b && wide) go(k_contract_block<TI, TO, true, true>);
    else if (b) go(k_contract_block<TI, TO, true, false>);
    else if (wide) go(k_contract_block<TI, TO, false, true>);
    else go(k_contract_block<TI, TO, false, false>);
  } else if (use_wave) {
    Dims red = red_full;
    int last = red.nd - 1;
    int64_t Lin = red.shape[last], sa = red.st[0][last], sb = red.st[1][last];
    int64_t Q = R / Lin;
    if (red.nd > 1) { red.nd -= 1; } else { red.shape[0] = 1; red.st[0][0] = red.st[1][0] = 0; }
    int64_t span = Q > 1 ? Q : Lin;
    int64_t chunk = (span + S_per - 1) / S_per;
    int64_t items = n_out * S;
    unsigned g = grid_for(items * 64, kBlock, maxb);
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(g), dim3(kBlock), 0, ctx->stream, keep, red, n_out, Q, Lin, sa, sb, S, chunk, (const TI*)a, (const TI*)b, (TO*)out, tp); };
    const bool wide = wide_rows(sizeof(TI), Q, Lin, sa, b, sb);
    if (b && wide) go(k_contract_wave<TI, TO, true, true>);
    else if (b) go(k_contract_wave<TI, TO, true, false>);
    else if (wide) go(k_contract_wave<TI, TO, false, true>);
    else go(k_contract_wave<TI, TO, false, false>);
  } else {
    int64_t chunk = (R + S_per - 1) / S_per;
    unsigned g = grid_for((n_out + kBlock - 1) / kBlock * kBlock * S, kBlock, maxb);
    if (b) hipLaunchKernelGGL((k_contract_lane<TI, TO, true>), dim3(g), dim3(kBlock), 0, ctx->stream, keep, red_full, n_out, R, S, chunk, (const TI*)a, (const TI*)b, (TO*)out, tp);
    else hipLaunchKernelGGL((k_contract_lane<TI, TO, false>), dim3(g), dim3(kBlock), 0, ctx->stream, keep, red_full, n_out, R, S, chunk, (const TI*)a, (const TI*)nullptr, (TO*)out, tp);
  }
  HG_CHECK_LAUNCH(ctx, "contract");
  return HGPU_OK;
}

}  // namespace

namespace hg {
hipError_t launch_extremum_row(hgpu_ctx* ctx, int dtype, int64_t n, int want_max, const void* a, void* index, void* value) {
  Dims keep;
  memset(&keep, 0, sizeof keep);
  keep.nd = 1;
  for (auto& e : keep.shape) e = 1;
  if (dtype == HGPU_F64) hipLaunchKernelGGL(k_argminmax_block<double>, dim3(1), dim3(1024), 0, ctx->stream, keep, n, (int64_t)1, want_max, (const double*)a, (int64_t*)index, (double*)value);
  else hipLaunchKernelGGL(k_argminmax_block<float>, dim3(1), dim3(1024), 0, ctx->stream, keep, n, (int64_t)1, want_max, (const float*)a, (int64_t*)index, (float*)value);
  return hipGetLastError();
}

static SumArgs sum_args(const RedJob& j) {
  SumArgs s;
  memset(&s, 0, sizeof s);
  s.part = j.a;
  s.other = j.b;
  s.out = j.out;
  s.out2 = j.out2;
  s.n = j.n_out;
  s.n1 = j.n1;
  s.stride = j.sa;
  s.S = (int)j.R;
  s.kind = j.variant;
  s.grid = j.grid;
  return s;
}

template <typename T>
static void launch_sum(hgpu_ctx* ctx, const RedJob& j) {
  const SumArgs s = sum_args(j);
  auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(j.grid), dim3(kBlock), 0, ctx->stream, s); };
  if (j.variant == RedJob::kSumTiny) go(k_sum_partials<T, RedJob::kSumTiny>);
  else if (j.variant == RedJob::kSumPair) go(k_sum_partials<T, RedJob::kSumPair>);
  else if (j.variant == RedJob::kSumRows) go(k_sum_partials<T, RedJob::kSumRows>);
  else if (j.variant == RedJob::kSumLane) go(k_sum_partials<T, RedJob::kSumLane>);
  else if (j.variant == RedJob::kSum32) go(k_sum_partials<T, RedJob::kSum32>);
  else go(k_sum_partials<T, RedJob::kSum8>);
}

// Partial results of more than this are added up at once: such a sum is long enough for a launch of its own, and its
// memory is better given back.
constexpr double kMaxHeldPartials = 64.0 * (1 << 20);

static int queue_sum(hgpu_ctx* ctx, RedJob& j, hgpu_buffer* part, const hgpu_array* out1, const hgpu_array* out2, const char* label = nullptr) {
  j.a = part->ptr;
  j.out = data_ptr(out1);
  j.out2 = out2 ? data_ptr(out2) : nullptr;
  j.label = label ? label : "gemm_sum_partials";
  j.flops = label ? 0 : (double)j.n_out * j.R;
  // (Submitted one by one, an objective's value goes out at once: the device would come to it only when the host asks.)
  if (out1->buf && (!out2 || out2->buf) && (double)part->bytes <= kMaxHeldPartials && (ctx->cap || j.n_out >= 16) &&
      hold_reduction(ctx, j, &part, 1, out1->buf, out2 ? out2->buf : nullptr)) return HGPU_OK;
  const Reads reads{j.a};
  LaunchGuard ls(ctx, j.label, j.bytes, j.flops, &reads);
  if (j.dtype == HGPU_F64) launch_sum<double>(ctx, j);
  else launch_sum<float>(ctx, j);
  HG_CHECK_LAUNCH(ctx, "gemm_sum_partials");
  return HGPU_OK;
}

int sum_partials(hgpu_ctx* ctx, int dtype, int64_t n, int parts, hgpu_buffer* part, const hgpu_array* out1, int64_t n1, const hgpu_array* out2, const char* label) {
  const size_t es = dtype_size(dtype);
  RedJob j;
  j.dtype = dtype;
  j.n_out = n;
  j.n1 = n1 < 0 ? n : n1;
  j.R = parts;
  j.sa = n;
  j.bytes = (double)n * (parts + 1) * es;
  // Rows of 8 for few outputs only: the recurrent network's three sums of 16384 fp64 outputs, 54 partials each, with rows of 8 /
  // of 32 18.1 / 12.0 us in their group.
  // fp32: rows of 32 are whole 128-byte lines (16384 outputs x 270 partials: 12.9 us with rows of 8, 7.1 us with rows of 32)
  j.variant = parts <= 8 || (parts <= 64 && n >= 65536) ? RedJob::kSumLane : (es == 4 || n > 8192 || parts < 32) ? RedJob::kSum32 : RedJob::kSum8;
  j.grid = grid_for(n, j.variant == RedJob::kSumLane ? 256 : j.variant == RedJob::kSum32 ? 32 : 8, ctx->num_cu * 8);
  return queue_sum(ctx, j, part, out1, out2, label);
}

// A row of S sums in doubles for every output.
static int sum_partial_rows(hgpu_ctx* ctx, int dtype, int64_t n, int64_t S, hgpu_buffer* part, const hgpu_array* out) {
  RedJob j;
  j.dtype = dtype;
  j.variant = RedJob::kSumRows;
  j.n_out = j.n1 = n;
  j.R = S;
  j.bytes = (double)n * (S * 8.0 + dtype_size(dtype));
  j.grid = grid_for(n * 64, kBlock, ctx->num_cu * 8);
  return queue_sum(ctx, j, part, out, nullptr);
}

hipError_t launch_reduction_group(hgpu_ctx* ctx, const RedJob* const* jobs, int n) {
  if (n == 1 && jobs[0]->is_sum()) {
    if (jobs[0]->dtype == HGPU_F64) launch_sum<double>(ctx, *jobs[0]);
    else launch_sum<float>(ctx, *jobs[0]);
    return hipGetLastError();
  }
  RedGroup g;
  memset(&g, 0, sizeof g);
  unsigned grid = 0;
  auto two = [](const Dims& d) {
    Dims2 e;
    memset(&e, 0, sizeof e);
    e.nd = d.nd;
    for (int i = 0; i < d.nd; ++i) { e.shape[i] = d.shape[i]; e.st[0][i] = d.st[0][i]; e.st[1][i] = d.st[1][i]; }
    return e;
  };
  for (int i = 0; i < n; ++i) {
    const RedJob& j = *jobs[i];
    grid += j.grid;
    if (j.is_sum()) { g.s[g.n_sums++] = sum_args(j); continue; }
    RedArgs& r = g.j[g.n++];
    r.keep = two(j.keep);
    r.red = two(j.red);
    r.n_out = j.n_out;
    r.R = j.R;
    r.Q = j.Q;
    r.Lin = j.Lin;
    r.sa = j.sa;
    r.sb = j.sb;
    r.chunk = j.chunk;
    r.variant = j.variant;
    r.hasb = j.hasb;
    r.grid = j.grid;
    r.a = j.a;
    r.b = j.b;
    r.out = j.out;
  }
  if (jobs[0]->dtype == HGPU_F64) hipLaunchKernelGGL((k_contract_group<double>), dim3(grid), dim3(kBlock), 0, ctx->stream, g);
  else hipLaunchKernelGGL((k_contract_group<float>), dim3(grid), dim3(kBlock), 0, ctx->stream, g);
  return hipGetLastError();
}
}  // namespace hg

namespace {

int64_t min_abs_nonzero(const Dims& d, int dim) {
  int64_t m = INT64_MAX;
  for (int k = 0; k < 2; ++k) {
    int64_t s = d.st[k][dim];
    if (s < 0) s = -s;
    if (s != 0 && s < m) m = s;
  }
  return m;
}

// The HBM-bound path of hgpu_contract: out[o] = sum_r a[o,r] * b[o,r] (b may be
// null) written densely at `out`.  Long reductions with few outputs are split
// into S chunks whose partial sums a second launch adds up.  The partial sums
// live in `scratch` when the caller brings one (then nothing is allocated here,
// and a request whose partial sums exceed scratch_bytes is refused), else in a
// block from the context's allocator.
int reduce_views(hgpu_ctx* ctx, const hgpu_array* a, const hgpu_array* b, int n_keep, void* out, void* scratch, size_t scratch_bytes, const hgpu_array* out_arr = nullptr) {
  int64_t n_out = 1, R = 1;
  for (int i = 0; i < n_keep; ++i) n_out *= a->shape[i];
  for (int i = n_keep; i < a->rank; ++i) R *= a->shape[i];
  int64_t zero[HGPU_MAX_RANK] = {0};
  const int64_t* bst = b ? b->strides : zero;
  const int64_t* ks[2] = {a->strides, bst};
  const int64_t* rs[2] = {a->strides + n_keep, bst + n_keep};
  Dims keep, red;
  if (!collapse(n_keep, a->shape, 2, ks, &keep) || !collapse(a->rank - n_keep, a->shape + n_keep, 2, rs, &red))
    return fail(ctx, HGPU_ERR_UNSUPPORTED, "contract: more than %d merged dims", HG_KDIMS);
  // Which way is memory contiguous: along the kept or along the reduced index?
  int64_t sr = min_abs_nonzero(red, red.nd - 1);
  int64_t sk = min_abs_nonzero(keep, keep.nd - 1);
  int64_t Lin = red.shape[red.nd - 1];
  bool use_wave;
  if (n_out < 2048) use_wave = true;
  else if (sr <= sk && Lin >= 16) use_wave = true;
  else use_wave = false;
  // Enough work items to fill the device, chunks of at least 512 elements.
  int64_t want_items = (int64_t)ctx->num_cu * (use_wave ? 16 : 1024);
  int64_t S = 1;
  if (n_out < want_items) {
    S = (want_items + n_out - 1) / n_out;
    int64_t span = use_wave ? ((R / Lin) > 1 ? (R / Lin) : Lin) : R;
    int64_t per = use_wave ? ((R / Lin) > 1 ? 512 / (Lin < 512 ? Lin : 512) : 1024) : 256;
    if (per < 1) per = 1;
    int64_t maxS = span / per;
    if (maxS < 1) maxS = 1;
    if (S > maxS) S = maxS;
    if (S > 4096) S = 4096;
  }
  // A caller's scratch bounds the partial sums: fewer chunks when they would not
  // fit, none (one launch, every output summed whole) when not even two do.
  if (scratch && S > 1 && (size_t)n_out * (size_t)S * 8 > scratch_bytes) {
    S = (int64_t)(scratch_bytes / ((size_t)n_out * 8));
    if (S < 2) S = 1;
  }
  const void* pa = data_ptr(a);
  const void* pb = b ? data_ptr(b) : nullptr;
  int rc = HGPU_OK;
  // (a caller that brings its own scratch wants its result written by the time the call returns to the stream: not held)
  HoldBufs hb{a->buf, b ? b->buf : nullptr, out_arr ? out_arr->buf : nullptr};
  const bool fresh = scratch == nullptr;
  const HoldBufs* hold = (hb.out && !scratch && a->buf && (!b || b->buf) && (a->dtype == HGPU_F64 || a->dtype == HGPU_F32)) ? &hb : nullptr;
  if (use_wave && ((n_out >= 64 && (n_out <= 1024 || S > 1) && R >= 1024 && R <= 65536) || (n_out < 64 && S > 1 && R >= 1024 && R <= 16384))) {
    // a few hundred outputs of a few thousand elements (or a handful of outputs, or so many that a wavefront each
    // leaves the device half empty, that would otherwise take a launch for partial sums and a second one to add them):
    // a block per output, one launch.  2048 rows of 8192 fp32: 17.2 us in two chunks a row and 4.7 to add them, 19.0 so.
    // Gradients, us, chunks / a block per output: wide dense network 1602 / 1557, recurrent network at batch 5000 (1280
    // outputs of 5000) 881 / 863.
    HG_DISPATCH_DTYPE(a->dtype, T, rc = (launch_stage<T, T>(ctx, true, keep, red, n_out, R, 0, pa, pb, out, nullptr, hold, a->dtype, fresh)));
  } else if (S == 1) {
    HG_DISPATCH_DTYPE(a->dtype, T, rc = (launch_stage<T, T>(ctx, use_wave, keep, red, n_out, R, 1, pa, pb, out, nullptr, hold, a->dtype, fresh)));
  } else {
    // stage 1: partials [n_out, S] in the accumulator type; stage 2 sums them.
    const size_t need = (size_t)n_out * (size_t)S * 8;
    hgpu_buffer* part = nullptr;
    void* pp = scratch;
    if (scratch) {
      if (need > scratch_bytes)   // cannot happen after the clamp above; kept as the guard of the fixed array
        return fail(ctx, HGPU_ERR_UNSUPPORTED, "contract: %lld outputs in %lld chunks need %zu bytes of partial sums, the fixed scratch holds %zu",
                    (long long)n_out, (long long)S, need, scratch_bytes);
    } else {
      rc = buffer_alloc(ctx, need, &part);
      if (rc) return rc;
      pp = part->ptr;
    }
    int64_t psh[2] = {n_out, S}, pst[2] = {S, 1};
    const bool few_long = n_out < 256 && S >= 256;
    HG_DISPATCH_DTYPE(a->dtype, T, { using A = typename acc_of<T>::type;  rc = (launch_stage<T, A>(ctx, use_wave, keep, red, n_out, R, (int)S, pa, pb, pp, nullptr, nullptr, -1, fresh)); });
    if (!rc && hold && n_out < 65536 && !few_long) {
      rc = sum_partial_rows(ctx, a->dtype, n_out, S, part, out_arr);
    } else if (!rc) {
      Dims k2, r2;
      int64_t z1[1] = {0};
      const int64_t* ks2[2] = {pst, z1};
      const int64_t* rs2[2] = {pst + 1, z1};
      collapse(1, psh, 2, ks2, &k2);
      collapse(1, psh + 1, 2, rs2, &r2);
      bool wave2 = n_out < 65536;
      // few outputs under many partial sums: a block each (one output, 4096 partial sums: 8.0 us with a wavefront, 4.4 with a block)
      HG_DISPATCH_DTYPE(a->dtype, T, { using A = typename acc_of<T>::type; rc = (launch_stage<A, T>(ctx, wave2, k2, r2, n_out, S, few_long ? 0 : 1, pp, nullptr, out, nullptr, nullptr, -1, fresh)); });
    }
    if (part) buffer_release(part);
  }
  return rc;
}

// Partial sums of hgpu_contract_noalloc: one array per device, held until the
// process ends.  In host code the name below is only a stand-in for the symbol:
// the device address comes from hipGetSymbolAddress, once per device.
constexpr size_t kScratchBytes = 1u << 20;
constexpr int kMaxDevices = 64;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];
static void* g_scratch_ptr[kMaxDevices];
static std::mutex g_scratch_mu;

int scratch_of(hgpu_ctx* ctx, void** out) {
  if (ctx->device < 0 || ctx->device >= kMaxDevices) return fail(ctx, HGPU_ERR_UNSUPPORTED, "contract_noalloc: device %d", ctx->device);
  std::lock_guard<std::mutex> g(g_scratch_mu);
  if (!g_scratch_ptr[ctx->device]) {
    hipError_t e = hipSetDevice(ctx->device);
    void* p = nullptr;
    if (e == hipSuccess) e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) return check_hip(ctx, e == hipSuccess ? hipErrorInvalidSymbol : e, "hipGetSymbolAddress(scratch)");
    g_scratch_ptr[ctx->device] = p;
  }
  *out = g_scratch_ptr[ctx->device];
  return HGPU_OK;
}

}  // namespace

namespace hg {
// A program over a few elements that an objective ends with (`negate sum * c`) joins the launch of a gradient's last sums: a
// pass of its own is 4 us in a graph.  One or two operands, up to four negations, additions, subtractions and
// multiplications: 12 bits each, in the order of the program, and above them which operands move.  Submitted one by one it
// goes out at once, by the same kernel: the host is about to ask for an objective's value, and what waits starts when it does.
bool try_tiny_map(hgpu_ctx* ctx, int n_in, const hgpu_array* const* in, int n_instr, const hgpu_fused_instr* prog, const hgpu_array* out) {
  const int64_t n = nelem(out);
  if (n_in < 1 || n_in > 2 || n_instr < 1 || n_instr > 4 || !dtype_is_float(out->dtype) || n < 1 || n > 64 || !out->buf) return false;
  uint64_t code = 0;
  for (int k = 0; k < n_instr; ++k) {
    const hgpu_fused_instr& q = prog[k];
    uint64_t op;
    if (q.kind == HGPU_FUSED_OP1 && q.op == HGPU_NEG) op = 0;
    else if (q.kind == HGPU_FUSED_OP2 && q.op == HGPU_ADD) op = 1;
    else if (q.kind == HGPU_FUSED_OP2 && q.op == HGPU_SUB) op = 2;
    else if (q.kind == HGPU_FUSED_OP2 && q.op == HGPU_MUL) op = 3;
    else return false;
    // (slots of this kernel: the operands are 0 and 1, results follow)
    auto slot = [&](int s) { return (uint64_t)(s < n_in ? s : s - n_in + 2); };
    code |= (op | slot(q.a) << 4 | (op ? slot(q.b) : 0) << 8) << (12 * k);
  }
  hgpu_buffer* reads[2] = {nullptr, nullptr};
  for (int i = 0; i < n_in; ++i) {
    if (in[i]->dtype != out->dtype || !in[i]->buf) return false;
    bool still = true;
    for (int d = 0; d < in[i]->rank; ++d) still = still && (in[i]->shape[d] == 1 || in[i]->strides[d] == 0);
    if (!still && !is_dense(in[i])) return false;
    if (!still) code |= 1ull << (48 + i);
    reads[i] = in[i]->buf;
  }
  RedJob j;
  j.dtype = out->dtype;
  j.variant = RedJob::kSumTiny;
  j.n_out = j.n1 = n;
  j.R = n_instr;
  j.sa = (int64_t)code;
  j.grid = 1;
  j.bytes = (double)n * (n_in + 1) * dtype_size(out->dtype);
  j.flops = (double)n * n_instr;
  j.label = "tiny_map";
  j.a = data_ptr(in[0]);
  j.b = n_in > 1 ? data_ptr(in[1]) : j.a;
  j.out = data_ptr(out);
  if (ctx->cap) return hold_reduction(ctx, j, reads, n_in, out->buf);
  const Reads from{j.a, j.b};
  LaunchGuard lg(ctx, j.label, j.bytes, j.flops, &from);
  if (j.dtype == HGPU_F64) launch_sum<double>(ctx, j);
  else launch_sum<float>(ctx, j);
  return hipGetLastError() == hipSuccess;
}

// *acc += x, taking over x (the first term becomes the accumulator).
int add_into(hgpu_ctx* ctx, hgpu_array** acc, hgpu_array* x) {
  if (!*acc) { *acc = x; return HGPU_OK; }
  hgpu_array* sum = nullptr;
  int rc = HGPU_OK;
  const int64_t n = nelem(x);
  // Both are results that may be held back: so is their sum, which joins the others' launch (the first step of a
  // recurrence, its state a constant, apart from the other steps: the sum of the two sent every held sum before it).
  const hgpu_array *first = *acc, *second = x;
  if (!is_dense(first)) std::swap(first, second);
  Dims d;
  const int64_t* st[1] = {second->strides};
  const bool rows = n > 0 && collapse(x->rank, x->shape, 1, st, &d) && d.nd <= 2 && d.st[0][d.nd - 1] >= INT32_MIN && d.st[0][d.nd - 1] <= INT32_MAX;
  if (dtype_is_float(x->dtype) && n > 0 && n <= (1 << 20) && is_dense(first) && rows) {
    rc = new_dense(ctx, x->dtype, x->rank, x->shape, &sum);
    RedJob j;
    j.dtype = x->dtype;
    j.variant = RedJob::kSumPair;
    j.n_out = j.n1 = n;
    j.R = 2;
    if (!is_dense(second)) {
      j.n1 = d.nd == 2 ? d.shape[1] : 1;
      j.sa = d.st[0][0];
      j.R = d.nd == 2 ? d.st[0][1] : 0;
    }
    j.grid = grid_for(n, 256 * 16 / (int)dtype_size(x->dtype), ctx->num_cu * 8);
    j.bytes = 3.0 * n * dtype_size(x->dtype);
    j.flops = (double)n;
    j.label = "gemm_sum_pair";
    if (!rc) {
      j.a = data_ptr(first);
      j.b = data_ptr(second);
      j.out = data_ptr(sum);
      hgpu_buffer* reads[2] = {(*acc)->buf, x->buf};
      if (!hold_reduction(ctx, j, reads, 2, sum->buf)) { hgpu_release(sum); sum = nullptr; }
    }
  }
  if (!rc && !sum) rc = hgpu_ewise2(ctx, HGPU_ADD, *acc, x, &sum);
  hgpu_release(*acc);
  hgpu_release(x);
  *acc = rc ? nullptr : sum;
  return rc;
}
}  // namespace hg

namespace {

// out = sum_t contract(as[t], bs[t]) for terms of one layout that are not a
// matrix product: the terms' chunks are reduced by one launch into partials
// [n_out, n * S], a second launch adds the partials up.
int contract_terms(hgpu_ctx* ctx, int n, const hgpu_array* const* as, const hgpu_array* const* bs, int n_keep, hgpu_array* o) {
  const hgpu_array* a = as[0];
  const hgpu_array* b = bs[0];
  int64_t n_out = nelem(o), R = 1;
  for (int i = n_keep; i < a->rank; ++i) R *= a->shape[i];
  const int64_t* ks[2] = {a->strides, b->strides};
  const int64_t* rs[2] = {a->strides + n_keep, b->strides + n_keep};
  Dims keep, red;
  if (!collapse(n_keep, a->shape, 2, ks, &keep) || !collapse(a->rank - n_keep, a->shape + n_keep, 2, rs, &red))
    return fail(ctx, HGPU_ERR_UNSUPPORTED, "contract_sum: more than %d merged dims", HG_KDIMS);
  int64_t sr = min_abs_nonzero(red, red.nd - 1), sk = min_abs_nonzero(keep, keep.nd - 1);
  int64_t Lin = red.shape[red.nd - 1];
  bool use_wave = n_out < 2048 || (sr <= sk && Lin >= 16);
  int64_t want_items = (int64_t)ctx->num_cu * (use_wave ? 16 : 1024);
  int64_t S = 1;
  if (n_out * n < want_items) {
    S = (want_items + n_out * n - 1) / (n_out * n);
    int64_t span = use_wave ? ((R / Lin) > 1 ? (R / Lin) : Lin) : R;
    int64_t per = use_wave ? ((R / Lin) > 1 ? 512 / (Lin < 512 ? Lin : 512) : 1024) : 256;
    if (per < 1) per = 1;
    int64_t maxS = span / per;
    if (maxS < 1) maxS = 1;
    if (S > maxS) S = maxS;
    if (S > 128) S = 128;
  }
  TermPtrs tp;
  tp.n = n;
  tp.s_per = (int)S;
  for (int t = 0; t < n; ++t) { tp.a[t] = data_ptr(as[t]); tp.b[t] = data_ptr(bs[t]); }
  const int64_t S_all = S * n;
  int accdt = dtype_is_float(a->dtype) ? HGPU_F64 : HGPU_I64;
  int64_t psh[2] = {n_out, S_all};
  hgpu_array* part = nullptr;
  int rc = new_dense(ctx, accdt, 2, psh, &part);
  if (rc) return rc;
  HG_DISPATCH_DTYPE(a->dtype, T, { using A = typename acc_of<T>::type; rc = (launch_stage<T, A>(ctx, use_wave, keep, red, n_out, R, (int)S_all, tp.a[0], tp.b[0], data_ptr(part), &tp)); });
  if (!rc && n_out < 65536 && dtype_is_float(a->dtype)) {
    rc = sum_partial_rows(ctx, a->dtype, n_out, S_all, part->buf, o);
  } else if (!rc) {
    Dims k2, r2;
    int64_t z1[1] = {0};
    const int64_t* ks2[2] = {part->strides, z1};
    const int64_t* rs2[2] = {part->strides + 1, z1};
    collapse(1, psh, 2, ks2, &k2);
    collapse(1, psh + 1, 2, rs2, &r2);
    bool wave2 = n_out < 65536;
    HG_DISPATCH_DTYPE(a->dtype, T, { using A = typename acc_of<T>::type; rc = (launch_stage<A, T>(ctx, wave2, k2, r2, n_out, S_all, 1, data_ptr(part), nullptr, data_ptr(o))); });
  }
  hgpu_release(part);
  return rc;
}

// Sums of rows: rows of floats side by side, all terms alike (the caller's: one shape, one set of strides), the other factor
// (where there is one) one element, the same for all terms.
struct RowView { int64_t rows, K, stride; const void* factor; hgpu_buffer* factor_buf; };
static bool row_view(int n, const hgpu_array* const* as, const hgpu_array* const* bs, int n_keep, const hgpu_array* out, RowView* v) {
  const hgpu_array* a = as[0];
  if (!dtype_is_float(a->dtype) || n > kGemmMaxTerms || !out->buf || nelem(a) == 0 || nelem(out) >= 65536) return false;
  const hgpu_array* b = bs ? bs[0] : nullptr;
  for (int t = 0; b && t < n; ++t) {
    if (data_ptr(bs[t]) != data_ptr(b)) return false;
    for (int d = 0; d < b->rank; ++d)
      if (b->shape[d] > 1 && bs[t]->strides[d] != 0) return false;
  }
  Dims keep, red;
  const int64_t* ks[1] = {a->strides};
  const int64_t* rs[1] = {a->strides + n_keep};
  if (!collapse(n_keep, a->shape, 1, ks, &keep) || !collapse(a->rank - n_keep, a->shape + n_keep, 1, rs, &red)) return false;
  if (keep.nd != 1 || red.nd != 1 || red.st[0][0] != 1 || keep.st[0][0] < 0) return false;
  *v = {keep.shape[0], red.shape[0], keep.st[0][0], b ? data_ptr(b) : nullptr, b ? b->buf : nullptr};
  return true;
}

// Row sums of what a held product multiplies (the bias gradient beside a weight gradient, in a recording): that product's blocks add
// them up as they stage its operand (gemm_split.hip, gemm_wide_f64.hip).  Its terms are all there are of this sum.
static int rows_with_product(hgpu_ctx* ctx, int n, const hgpu_array* const* as, const hgpu_array* const* bs, int n_keep, const hgpu_array* out, bool* handled) {
  const hgpu_array* a = as[0];
  RowView v;
  if (!ctx->cap || !row_view(n, as, bs, n_keep, out, &v)) return HGPU_OK;
  const void* ptrs[kGemmMaxTerms];
  for (int t = 0; t < n; ++t) ptrs[t] = data_ptr(as[t]);
  hgpu_buffer* part = nullptr;
  int shares = 0;
  if (!join_wide_rows(ctx, a->dtype, n, ptrs, v.rows, v.K, v.stride, v.factor_buf, v.factor, &part, &shares)) return HGPU_OK;
  const int rc = sum_partial_rows(ctx, a->dtype, v.rows, shares, part, out);
  buffer_release(part);
  *handled = !rc;
  return rc;
}

// Sums of rows over several terms, each element times one factor: a bias gradient of an unrolled recurrence where no held
// product reads the same rows.  A block per output row, whose wavefronts take whole terms, four at a time; doubles, in a fixed
// order; the result itself, no partial sums.  What bounds it is the launch and a few trips to memory: the kernel that takes
// any reduction is 13 KB of code, with 64-bit divisions on its way, and the device fetches them anew for every launch in
// another kernel's wake.  28 terms of 128 rows of 150 fp64 inside a recording: 15.5 us (the second such sum 7.7) and their part
// of the sums of partial results.
constexpr int kRowWaves = 8;
struct RowTerms {
  const void* a[kGemmMaxTerms];
  int n, K;
  int64_t stride;             // elements between rows
  const void* factor;         // one element; null: 1
  void* out;
};
template <typename T>
__global__ void __launch_bounds__(64 * kRowWaves) k_row_terms(RowTerms p) {
  __shared__ double part[kRowWaves];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t at = (int64_t)blockIdx.x * p.stride;
  const double f = p.factor ? (double)*(const T*)p.factor : 1.0;
  double c[4] = {0, 0, 0, 0};
  for (int t = w; t < p.n; t += 4 * kRowWaves) {
    const T* row[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) row[u] = (const T*)p.a[t + u * kRowWaves < p.n ? t + u * kRowWaves : p.n - 1] + at;
    for (int k0 = 0; k0 < p.K; k0 += 128) {
      T x[4][2];
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          const int k = k0 + 64 * v + lane;
          x[u][v] = row[u][k < p.K ? k : p.K - 1];
        }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int v = 0; v < 2; ++v)
          if (t + u * kRowWaves < p.n && k0 + 64 * v + lane < p.K) c[u] = __builtin_fma((double)x[u][v], f, c[u]);
    }
  }
  const double s = wave_sum<double>((c[0] + c[1]) + (c[2] + c[3]));
  if (lane == 0) part[w] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    double tot = part[0];
#pragma unroll
    for (int k = 1; k < kRowWaves; ++k) tot += part[k];
    ((T*)p.out)[blockIdx.x] = (T)tot;
  }
}

// Rows side by side, all terms alike, the other factor one element and the same for all terms; short enough for a block to a
// row (16384 elements: 32 of a lane), rows enough to fill a part of the device.
static int row_terms(hgpu_ctx* ctx, int n, const hgpu_array* const* as, const hgpu_array* const* bs, int n_keep, const hgpu_array* out, bool* handled) {
  const hgpu_array* a = as[0];
  RowView v;
  if (!row_view(n, as, bs, n_keep, out, &v) || v.rows < 16 || (double)n * (double)v.K > 16384) return HGPU_OK;
  RowTerms p;
  memset(&p, 0, sizeof p);
  for (int t = 0; t < n; ++t) p.a[t] = data_ptr(as[t]);
  p.n = n;
  p.K = (int)v.K;
  p.stride = v.stride;
  p.factor = v.factor;
  p.out = data_ptr(out);
  Reads reads;
  reads.add(p.a, p.a + n);
  if (p.factor) reads.push_back(p.factor);
  LaunchGuard lg(ctx, "row_terms", ((double)n * (double)v.K * (double)v.rows + (double)v.rows) * (double)dtype_size(a->dtype), (double)n * (double)v.K * (double)v.rows, &reads);
  if (a->dtype == HGPU_F64) hipLaunchKernelGGL(k_row_terms<double>, dim3((unsigned)v.rows), dim3(64 * kRowWaves), 0, ctx->stream, p);
  else hipLaunchKernelGGL(k_row_terms<float>, dim3((unsigned)v.rows), dim3(64 * kRowWaves), 0, ctx->stream, p);
  HG_CHECK_LAUNCH(ctx, "row_terms");
  *handled = true;
  return HGPU_OK;
}

}  // namespace

extern "C" {

int hgpu_contract_sum(hgpu_ctx* ctx, int n, const hgpu_array* const* as, const hgpu_array* const* bs, int n_keep, hgpu_array** out) {
  if (!ctx || !as || !bs || !out || n < 1) return HGPU_ERR_INVALID;
  for (int t = 0; t < n; ++t) {
    if (!as[t] || !bs[t]) return HGPU_ERR_INVALID;
    if (as[t]->dtype != as[0]->dtype || bs[t]->dtype != as[0]->dtype) return fail(ctx, HGPU_ERR_INVALID, "contract_sum: dtypes differ");
    if (!same_shape(as[t], as[0]) || !same_shape(bs[t], as[0])) return fail(ctx, HGPU_ERR_INVALID, "contract_sum: shapes differ");
  }
  const hgpu_array* a = as[0];
  if (n_keep < 0 || n_keep > a->rank) return fail(ctx, HGPU_ERR_INVALID, "contract_sum: n_keep %d of rank %d", n_keep, a->rank);
  if (n == 1) return hgpu_contract(ctx, as[0], bs[0], n_keep, out);
  // Terms of one layout go out together, 32 to a launch: when such a group is a
  // matrix product the K chunks of all its terms are summed in one fixed order
  // by one kernel.  Groups are formed in order of first appearance and their
  // results added in that order.
  const bool groupable = nelem(a) > 0 && (a->dtype == HGPU_F64 || a->dtype == HGPU_F32);
  auto same_layout = [&](int s, int t) {
    for (int d = 0; d < a->rank; ++d)
      if (as[s]->strides[d] != as[t]->strides[d] || bs[s]->strides[d] != bs[t]->strides[d]) return false;
    return true;
  };
  std::vector<char> taken((size_t)n, 0);
  hgpu_array* acc = nullptr;
  for (int t0 = 0; t0 < n; ++t0) {
    if (taken[(size_t)t0]) continue;
    std::vector<const hgpu_array*> ga{as[t0]}, gb{bs[t0]};
    taken[(size_t)t0] = 1;
    for (int t = t0 + 1; t < n && groupable && ga.size() < (size_t)kGemmMaxTerms; ++t)
      if (!taken[(size_t)t] && same_layout(t0, t)) { ga.push_back(as[t]); gb.push_back(bs[t]); taken[(size_t)t] = 1; }
    hgpu_array* part = nullptr;
    int rc = HGPU_OK;
    size_t done = 0;
    if (ga.size() > 1) {
      rc = new_dense(ctx, a->dtype, n_keep, a->shape, &part);
      bool handled = false;
      if (!rc) rc = try_gemm(ctx, ga[0], gb[0], n_keep, part, &handled, (int)ga.size(), ga.data(), gb.data());
      if (!rc && !handled) rc = rows_with_product(ctx, (int)ga.size(), ga.data(), gb.data(), n_keep, part, &handled);
      if (!rc && !handled) rc = row_terms(ctx, (int)ga.size(), ga.data(), gb.data(), n_keep, part, &handled);
      if (!rc && !handled && nelem(part) > 0) {   // not a matrix product: the grouped reduction
        rc = contract_terms(ctx, (int)ga.size(), ga.data(), gb.data(), n_keep, part);
        handled = !rc;
      }
      if (rc || !handled) { if (part) hgpu_release(part); part = nullptr; }
      else done = ga.size();
    }
    for (size_t t = done; t < ga.size() && !rc; ++t) {   // not a matrix product (or a single term): one by one
      hgpu_array* one = nullptr;
      rc = hgpu_contract(ctx, ga[t], gb[t], n_keep, &one);
      if (!rc) rc = add_into(ctx, &part, one);
    }
    if (!rc) rc = add_into(ctx, &acc, part), part = nullptr;
    if (rc) { if (part) hgpu_release(part); if (acc) hgpu_release(acc); return rc; }
  }
  *out = acc;
  return HGPU_OK;
}

int hgpu_contract(hgpu_ctx* ctx, const hgpu_array* a, const hgpu_array* b, int n_keep, hgpu_array** out) {
  if (!ctx || !a || !out) return HGPU_ERR_INVALID;
  if (n_keep < 0 || n_keep > a->rank) return fail(ctx, HGPU_ERR_INVALID, "contract: n_keep %d of rank %d", n_keep, a->rank);
  if (b) {
    if (b->dtype != a->dtype) return fail(ctx, HGPU_ERR_INVALID, "contract: dtypes differ");
    if (!same_shape(a, b)) return fail(ctx, HGPU_ERR_INVALID, "contract: shapes differ");
  }
  if (a->dtype == HGPU_BOOL) return fail(ctx, HGPU_ERR_INVALID, "contract: Bool arrays have no sum");
  // A kept dim along which neither operand moves (both replicated) repeats the
  // same values: compute once without it, replicate the result as a view.
  {
    bool repeats = false;
    int64_t sh1[HGPU_MAX_RANK];
    for (int i = 0; i < a->rank; ++i) {
      sh1[i] = a->shape[i];
      if (i < n_keep && a->shape[i] > 1 && a->strides[i] == 0 && (!b || b->strides[i] == 0)) { sh1[i] = 1; repeats = true; }
    }
    bool empty = false;
    for (int i = 0; i < a->rank; ++i) empty = empty || a->shape[i] == 0;
    if (repeats && !empty) {
      hgpu_array* a1 = new_view(ctx, a->buf, a->dtype, a->rank, sh1, a->strides, a->offset);
      hgpu_array* b1 = b ? new_view(ctx, b->buf, b->dtype, b->rank, sh1, b->strides, b->offset) : nullptr;
      hgpu_array* small = nullptr;
      int rc1 = hgpu_contract(ctx, a1, b1, n_keep, &small);
      hgpu_release(a1);
      if (b1) hgpu_release(b1);
      if (rc1) return rc1;
      int64_t st[HGPU_MAX_RANK];
      for (int i = 0; i < n_keep; ++i) st[i] = sh1[i] != a->shape[i] ? 0 : small->strides[i];
      *out = new_view(ctx, small->buf, small->dtype, n_keep, a->shape, st, small->offset);
      hgpu_release(small);
      return HGPU_OK;
    }
  }
  hgpu_array* o = nullptr;
  int64_t n_out = 1, R = 1;
  for (int i = 0; i < n_keep; ++i) n_out *= a->shape[i];
  for (int i = n_keep; i < a->rank; ++i) R *= a->shape[i];
  int rc;
  if (n_out == 0 || R == 0) {
    rc = new_zeros(ctx, a->dtype, n_keep, a->shape, &o);
    if (rc) return rc;
    *out = o;
    return HGPU_OK;
  }
  rc = new_dense(ctx, a->dtype, n_keep, a->shape, &o);
  if (!rc && b && n_keep == 0) {
    bool handled = false;
    rc = try_gather_dot(ctx, a, b, o, &handled);
    if (rc) { hgpu_release(o); return rc; }
    if (handled) { *out = o; return HGPU_OK; }
  }
  if (rc) return rc;

  bool handled = false;
  rc = try_gemm(ctx, a, b, n_keep, o, &handled);
  if (rc) { hgpu_release(o); return rc; }
  if (handled) { *out = o; return HGPU_OK; }

  rc = rows_with_product(ctx, 1, &a, b ? &b : nullptr, n_keep, o, &handled);
  if (!rc && !handled) rc = reduce_views(ctx, a, b, n_keep, data_ptr(o), nullptr, 0, o);
  if (rc) { hgpu_release(o); return rc; }
  *out = o;
  return HGPU_OK;
}

int hgpu_contract_noalloc(hgpu_ctx* ctx, const hgpu_array* a, const hgpu_array* b, int n_keep, hgpu_array* out) {
  if (!ctx || !a || !out) return HGPU_ERR_INVALID;
  if (n_keep < 0 || n_keep > a->rank) return fail(ctx, HGPU_ERR_INVALID, "contract_noalloc: n_keep %d of rank %d", n_keep, a->rank);
  if (b) {
    if (b->dtype != a->dtype) return fail(ctx, HGPU_ERR_INVALID, "contract_noalloc: dtypes differ");
    if (!same_shape(a, b)) return fail(ctx, HGPU_ERR_INVALID, "contract_noalloc: shapes differ");
  }
  if (a->dtype == HGPU_BOOL) return fail(ctx, HGPU_ERR_INVALID, "contract_noalloc: Bool arrays have no sum");
  if (out->dtype != a->dtype || out->rank != n_keep || !is_dense(out)) return fail(ctx, HGPU_ERR_INVALID, "contract_noalloc: the result array must be dense, of the operands' dtype and of the kept shape");
  for (int i = 0; i < n_keep; ++i)
    if (out->shape[i] != a->shape[i]) return fail(ctx, HGPU_ERR_INVALID, "contract_noalloc: the result array must have the kept shape");
  if (out->buf && (out->buf == a->buf || (b && out->buf == b->buf))) return fail(ctx, HGPU_ERR_INVALID, "contract_noalloc: the result shares memory with an operand");
  int64_t n_out = nelem(out), R = 1;
  for (int i = n_keep; i < a->rank; ++i) R *= a->shape[i];
  if (n_out == 0) return HGPU_OK;
  if (R == 0) {   // an empty sum: zeros (the fill rounds up to 16 bytes, which stays inside a block only from its start)
    if (out->offset != 0) return fail(ctx, HGPU_ERR_UNSUPPORTED, "contract_noalloc: an empty sum into a view that does not start its block");
    return zero_fill(ctx, data_ptr(out), (size_t)n_out * dtype_size(out->dtype));
  }
  void* sp = nullptr;
  if (int rc = scratch_of(ctx, &sp)) return rc;
  return reduce_views(ctx, a, b, n_keep, data_ptr(out), sp, kScratchBytes);
}

int hgpu_extremum_last(hgpu_ctx* ctx, const hgpu_array* a, int want_max, hgpu_array** values, hgpu_array** out) {
  if (!ctx || !a || !out) return HGPU_ERR_INVALID;
  if (a->rank < 1) return fail(ctx, HGPU_ERR_INVALID, "argminmax: rank 0");
  int64_t L = a->shape[a->rank - 1];
  if (L < 1) return fail(ctx, HGPU_ERR_INVALID, "argminmax: empty last dim");
  hgpu_array* o = nullptr;
  int rc = new_dense(ctx, HGPU_I64, a->rank - 1, a->shape, &o);
  if (rc) return rc;
  hgpu_array* v = nullptr;
  if (values) {
    rc = new_dense(ctx, a->dtype, a->rank - 1, a->shape, &v);
    if (rc) { hgpu_release(o); return rc; }
  }
  int64_t n_out = nelem(o);
  if (n_out > 0) {
    const int64_t* ks[1] = {a->strides};
    Dims keep;
    if (!collapse(a->rank - 1, a->shape, 1, ks, &keep)) { hgpu_release(o); if (v) hgpu_release(v); return fail(ctx, HGPU_ERR_UNSUPPORTED, "argminmax: too many dims"); }
    if (v && n_out == 1 && try_hold_extremum(ctx, a, want_max, o, v)) {
      *out = o;
      *values = v;
      return HGPU_OK;
    }
    const bool pieces = L >= kPiecesFrom && n_out <= kPiecesRows;
    void* tickets = nullptr;
    hgpu_buffer* scratch = nullptr;
    if (pieces) rc = ticket_block(ctx, &tickets);
    if (pieces && !rc) rc = buffer_alloc(ctx, (size_t)(n_out * pieces_of(L)) * 16, &scratch);
    if (rc) { hgpu_release(o); if (v) hgpu_release(v); return rc; }
    const Reads reads = reads_of(1, &a);
    LaunchGuard lg(ctx, "argminmax", (double)n_out * (L * dtype_size(a->dtype) + 8 + (v ? dtype_size(a->dtype) : 0)), (double)n_out * L, &reads);
    void* vp = v ? data_ptr(v) : nullptr;
    if (pieces) {
      // very few, very long rows: pieces of a row to many blocks, then one pick per row
      HG_DISPATCH_DTYPE(a->dtype, T, extremum_pieces<T>(ctx, keep, n_out, L, a->strides[a->rank - 1], want_max, data_ptr(a), scratch->ptr, (unsigned*)tickets, data_ptr(o), vp));
      buffer_release(scratch);
    } else if (L >= 512 && n_out <= 64) {
      // few long rows: a whole block per row (one row of 2500 fp32, a minibatch's logits: a wavefront, load after load, takes
      // 14.4 us, a block 5.8; one of 1500 fp64 9.9 and 5.0)
      HG_DISPATCH_DTYPE(a->dtype, T, hipLaunchKernelGGL(k_argminmax_block<T>, dim3((unsigned)n_out), dim3(1024), 0, ctx->stream, keep, L, a->strides[a->rank - 1], want_max, (const T*)data_ptr(a), (int64_t*)data_ptr(o), (T*)vp));
    } else if (L >= 256 && n_out < (int64_t)ctx->num_cu * 64) {
      unsigned g = grid_for(n_out * 64, kBlock, ctx->num_cu * 8);
      HG_DISPATCH_DTYPE(a->dtype, T, hipLaunchKernelGGL(k_argminmax_wave<T>, dim3(g), dim3(kBlock), 0, ctx->stream, keep, n_out, L, a->strides[a->rank - 1], want_max, (const T*)data_ptr(a), (int64_t*)data_ptr(o), (T*)vp));
    } else {
      unsigned g = grid_for(n_out, kBlock, ctx->num_cu * 8);
      HG_DISPATCH_DTYPE(a->dtype, T, hipLaunchKernelGGL(k_argminmax<T>, dim3(g), dim3(kBlock), 0, ctx->stream, keep, n_out, L, a->strides[a->rank - 1], want_max, (const T*)data_ptr(a), (int64_t*)data_ptr(o), (T*)vp));
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) { hgpu_release(o); if (v) hgpu_release(v); return check_hip(ctx, e, "argminmax"); }
  }
  *out = o;
  if (values) *values = v;
  return HGPU_OK;
}

int hgpu_argminmax_last(hgpu_ctx* ctx, const hgpu_array* a, int want_max, hgpu_array** out) {
  return hgpu_extremum_last(ctx, a, want_max, nullptr, out);
}

}  // extern "C"
