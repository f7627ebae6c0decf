// Matrix-core (MFMA) path of hgpu_contract.
//
// horde-ad's `Concrete` backend computes matmul2 as "dot over the innermost
// dim of two broadcast views" (src/HordeAd/Core/OpsConcrete.hs:237-242) and
// convolutions as the same contraction over gathered windows
// (test/simplified/TestMnistPP.hs:735).  Seen through strides these are all ONE
// pattern:  every kept dim advances only A (an "M" dim), only B (an "N" dim) or
// both (a batch dim), and every reduced dim advances both (a "K" dim).  Then
//     A[m, k] sits at  offAm(m) + offAk(k),   B[n, k] at  offBn(n) + offBk(k),
//     C[m, n] at  offCm(m) + offCn(n),
// with m, n, k multi-indices -- a matrix product whose operands are addressed
// through separable offset maps.  No operand is copied or re-laid-out: the
// im2col "patch matrix" of a convolution exists only as such a map.
//
// Kernel: 256 threads = 4 wavefronts, K-step 16; the block tile ranges from
// 128x128 (wavefronts 2x2, each 4x4 MFMA tiles of 16x16) down to 256x16 / 16x256
// and 32x32 for skinny or tiny outputs (a convolution with 16 output channels
// has N = 16).  v_mfma_f64_16x16x4_f64 / v_mfma_f32_16x16x4_f32, accumulators
// in registers.
// Operand tiles are staged through LDS in [k][m] order (one element of padding
// per row keeps both the transposing stores and the MFMA-fragment loads free
// of bank conflicts); the global loads of tile t+1 are issued before the MFMAs
// of tile t.  Lanes run along whichever of m or k is contiguous in memory, so
// loads coalesce for both plain and transposed operands.  Tiles are numbered
// so that each XCD (blockIdx mod 8) works on a contiguous run of tiles and its
// L2 sees neighbouring rows of A.  Small outputs with long K are split along K
// into partial products summed by a second launch (fixed order: reproducible).
#include <algorithm>
#include <cmath>

#include "gemm_kernel.hpp"

namespace hg {
// A product of gemm_single_dims that is held back.
struct WideJob {
  bool f64, akc, bkc, thin;
  gemm::SplitJob j;
};
static_assert(kMaxWideJobs == gemm::kMaxSplitGroup, "");
}  // namespace hg

using namespace hg;
using namespace hg::gemm;

namespace {

// K offset tables of both operands, Kp >= K entries: entries past K repeat the
// last four valid k (so that a 4-element vector load at a padded entry stays
// inside the operand).
__global__ void k_koff(Group k, int64_t K, int64_t Kp, int64_t* __restrict__ ka, int64_t* __restrict__ kb) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < Kp) {
    int64_t idx = i;
    if (i >= K) {
      idx = K >= 4 ? K - 4 + (i & 3) : K - 1;
      if (idx > K - 1) idx = K - 1;
    }
    int64_t a, b, c;
    group_off(k, idx, &a, &b, &c);
    ka[i] = a;
    kb[i] = b;
  }
}

// Appends dim (extent e, strides a, b, c) to a group, merging with the previous dim when all strides allow.
bool push_dim(Group& g, int64_t e, int64_t a, int64_t b, int64_t c) {
  if (e == 1) return true;
  if (g.nd > 0) {
    int p = g.nd - 1;
    if (g.sa[p] == a * e && g.sb[p] == b * e && g.sc[p] == c * e) {
      g.shape[p] *= e;
      g.sa[p] = a;
      g.sb[p] = b;
      g.sc[p] = c;
      return true;
    }
  }
  if (g.nd == GD) return false;
  g.shape[g.nd] = e;
  g.sa[g.nd] = a;
  g.sb[g.nd] = b;
  g.sc[g.nd] = c;
  g.nd++;
  return true;
}

void finish(Group& g) {
  if (g.nd == 0) {
    g.nd = 1;
    g.shape[0] = 1;
    g.sa[0] = g.sb[0] = g.sc[0] = 0;
  }
  for (int i = g.nd; i < GD; ++i) {
    g.shape[i] = 1;
    g.sa[i] = g.sb[i] = g.sc[i] = 0;
  }
}

int64_t total(const Group& g) {
  int64_t n = 1;
  for (int i = 0; i < g.nd; ++i) n *= g.shape[i];
  return n;
}

// What a product's launch reads: see LaunchGuard.
Reads product_reads(const void* pa, const void* pb, int n_terms, const void* const* as, const void* const* bs) {
  Reads r{pa, pb};
  r.add(as, as + n_terms);
  r.add(bs, bs + n_terms);
  return r;
}

// True when 16-byte loads along the direction the staging lanes run are safe
// for one operand: unit stride there and an extent that is a multiple of the
// vector, so that the elements of a vector are neighbours in memory.  The
// vectors need element alignment only.
bool vector_ok(size_t es, const Group& run, int run_dim, const int64_t* run_st) {
  const int64_t v = (int64_t)(16 / es);
  return run_st[run_dim] == 1 && run.shape[run_dim] % v == 0;
}
// Products with at most 32 rows or columns: the LDS-free kernel, the small side as N.
int gemm_direct(hgpu_ctx* ctx, GemmParams p, int dtype, const void* pa, const void* pb, hgpu_array* out, bool* handled, int n_terms) {
  if (p.N > 32) {   // swap the roles of the operands: C^T = B A^T
    std::swap(p.m, p.n);
    std::swap(p.M, p.N);
    std::swap(pa, pb);
    for (int t = 0; t < n_terms; ++t) std::swap(p.a_term[t], p.b_term[t]);
    for (Group* g : {&p.m, &p.n, &p.k, &p.bt})
      for (int i = 0; i < GD; ++i) std::swap(g->sa[i], g->sb[i]);
  }
  const int tn = p.N <= 16 ? 1 : 2, tm = p.M <= 16 ? 1 : (p.M <= 32 ? 2 : 4);
  const int64_t tiles = ((p.M + 16 * tm - 1) / (16 * tm)) * ((p.N + 16 * tn - 1) / (16 * tn));
  if (tiles > 0x3fffffff) return HGPU_OK;
  // one wavefront per (tile, K chunk): aim at one per SIMD (more, shorter chunks
  // measured slower: set-up and partial sums per wavefront), chunks of at least 64
  const int64_t want = (int64_t)ctx->num_cu * 4;
  const int64_t out_elems = p.M * p.N * p.BT;
  const int64_t nt = n_terms > 0 ? n_terms : 1;      // products summed by this launch
  int64_t split = 1;
  if (tiles * p.BT * nt * 2 <= want && p.K >= 128) {
    split = (want + tiles * p.BT * nt - 1) / (tiles * p.BT * nt);
    int64_t cap = (int64_t)((double)(p.M + p.N) * p.K * p.BT / (2.0 * out_elems));   // partials stay small next to the operands
    if (cap > 4096) cap = 4096;
    if (split > cap) split = cap;
    if (split > p.K / 64) split = p.K / 64;
    if (split < 1) split = 1;
  }
  p.kchunk = ((p.K + split - 1) / split + 15) / 16 * 16;
  p.term_split = (int)((p.K + p.kchunk - 1) / p.kchunk);
  p.n_terms = n_terms;
  p.split = (int)(p.term_split * nt);                // K chunks of all terms
  split = p.split;
  p.a_kc = p.b_kc = 0;
  p.c_rows_contig = 0;

  const size_t es = dtype_size(dtype);
  const int64_t out_n = nelem(out);
  const void* zero_tab = nullptr;
  int rc = zero_block(ctx, &zero_tab);
  if (rc) return rc;
  hgpu_buffer* koff = nullptr;
  const int64_t Kp = (p.K + 15) / 16 * 16 + 32;   // padded tables (see k_gemm_direct)
  rc = buffer_alloc(ctx, (size_t)Kp * 16, &koff);
  if (rc) return rc;
  hgpu_buffer* part = nullptr;
  if (split > 1) {
    rc = buffer_alloc(ctx, (size_t)out_n * split * es, &part);
    if (rc) { buffer_release(koff); return rc; }
  }
  p.c_split_stride = split > 1 ? out_n : 0;
  int64_t* ka = (int64_t*)koff->ptr;
  int64_t* kb = ka + Kp;
  dim3 grid((unsigned)((tiles * split + 3) / 4), 1, (unsigned)p.BT);
  {
    double flops = 2.0 * p.M * p.N * p.K * p.BT * nt;
    double bytes = (((double)p.M * p.K + (double)p.N * p.K) * nt + (double)p.M * p.N) * p.BT * es;
    const char* label = dtype == HGPU_F64 ? "gemm_f64" : "gemm_f32";
    if (ctx->profiling && ctx->profile_shapes) {
      char buf[128];
      snprintf(buf, sizeof buf, "%s[M%lldxN%lldxK%lldxB%lld,s%d,direct,t%dx%d,k%lld:%lld/%lld]", label, (long long)p.M, (long long)p.N, (long long)p.K, (long long)p.BT, (int)split, 16 * tm, 16 * tn, (long long)p.k.shape[p.k.nd - 1], (long long)p.k.sa[p.k.nd - 1], (long long)p.k.sb[p.k.nd - 1]);
      label = intern_label(ctx, buf);
    }
    // the helper launches are timed under their own names, the label times the MFMA kernel alone
    if (p.k.nd > 1) {
      const Reads none;
      LaunchGuard lk(ctx, "gemm_k_offsets", (double)Kp * 16, 0, &none);
      hipLaunchKernelGGL(k_koff, dim3((unsigned)((Kp + 255) / 256)), dim3(256), 0, ctx->stream, p.k, p.K, Kp, ka, kb);
      p.kmask = -1;
      p.ksa = p.ksb = 0;
    } else {   // single K dim: offsets are k * stride, the table a block of zeros
      ka = kb = (int64_t*)zero_tab;
      p.kmask = 0;
      p.ksa = p.k.sa[0];
      p.ksb = p.k.sb[0];
    }
    void* cdst = split > 1 ? part->ptr : data_ptr(out);
    // an operand contiguous along K is read four elements at a time
    auto k_vector = [&](const void* base, const void* const* terms, const int64_t* ks, const int64_t* rs, const Group& rows, const int64_t* bs) {
      const int64_t v = (int64_t)(16 / es);
      const int kd = p.k.nd - 1;
      for (int t = 0; t < n_terms; ++t)
        if (((uintptr_t)terms[t] & 15) != 0) return false;
      if (((uintptr_t)base & 15) != 0 || p.K < 16 || ks[kd] != 1 || p.k.shape[kd] % 4 != 0) return false;
      for (int i = 0; i < kd; ++i) if (ks[i] % v != 0) return false;
      for (int i = 0; i < rows.nd; ++i) if (rs[i] % v != 0) return false;
      for (int i = 0; i < p.bt.nd; ++i) if (bs[i] % v != 0) return false;
      return true;
    };
    const bool va = k_vector(pa, p.a_term, p.k.sa, p.m.sa, p.m, p.bt.sa), vb = k_vector(pb, p.b_term, p.k.sb, p.n.sb, p.n, p.bt.sb);
    LaunchArgs la{ctx->stream, -1, tm, tn, va, vb, grid, pa, pb, cdst, ka, kb};
    {
      const Reads reads = product_reads(pa, pb, n_terms, p.a_term, p.b_term);
      LaunchGuard lg(ctx, label, bytes, flops, &reads);
      la.ev_start = lg.start_event();
      la.ev_stop = lg.stop_event();
      if (dtype == HGPU_F64) launch_f64(p, la);
      else launch_f32(p, la);
    }
    if (split > 1) rc = sum_partials(ctx, dtype, out_n, (int)split, part, out);
  }
  hipError_t e = hipGetLastError();
  buffer_release(koff);
  if (part) buffer_release(part);
  if (rc) return rc;
  if (e != hipSuccess) return check_hip(ctx, e, "gemm");
  *handled = true;
  return HGPU_OK;
}

int wide_chunk(int K, int shares) { return ((K + shares - 1) / shares + 15) / 16 * 16; }

// Products whose row, column, contracted and batch indices are single dims with strides that a 32-bit byte offset
// reaches: fp32 on the bf16 matrix cores (gemm_split.hip), fp64 in tiles without address arithmetic (gemm_wide_f64.hip).
int gemm_single_dims(hgpu_ctx* ctx, const GemmParams& p, int dtype, const void* pa, const void* pb, hgpu_array* out, bool* handled, int n_terms, hgpu_array** partials_out,
                     const std::vector<hgpu_buffer*>& operands) {
  if (p.m.nd != 1 || p.n.nd != 1 || p.k.nd != 1 || p.bt.nd != 1) return HGPU_OK;
  const int64_t nt = n_terms > 0 ? n_terms : 1;
  const bool f64 = dtype == HGPU_F64;
  const int64_t es = f64 ? 8 : 4;
  SplitParams q{};
  int64_t sam = p.m.sa[0], sak = p.k.sa[0], sbn = p.n.sb[0], sbk = p.k.sb[0], scm = p.m.sc[0], scn = p.n.sc[0], M = p.M, N = p.N;
  int64_t bsa = p.bt.sa[0], bsb = p.bt.sb[0];
  const bool thin = !f64 && std::min(M, N) <= 32;
  bool swap = thin ? M < N : scm == 1 && scn != 1;          // the lanes of a result block run along its columns; a thin side is its columns
  if (swap) {
    std::swap(sam, sbn);
    std::swap(sak, sbk);
    std::swap(scm, scn);
    std::swap(M, N);
    std::swap(bsa, bsb);
  }
  if (sam < 0 || sak < 0 || sbn < 0 || sbk < 0 || p.K > (1 << 24)) return HGPU_OK;
  const int64_t a_bytes = ((M - 1) * sam + (p.K - 1) * sak + 1) * es, b_bytes = ((N - 1) * sbn + (p.K - 1) * sbk + 1) * es;
  if (a_bytes > 0x7fffff00 || b_bytes > 0x7fffff00 || M > 0x3fffffff || N > 0x3fffffff) return HGPU_OK;
  q.M = (int)M;
  q.N = (int)N;
  q.K = (int)p.K;
  q.sam = (uint32_t)(sam * es);
  q.sak = (uint32_t)(sak * es);
  q.sbn = (uint32_t)(sbn * es);
  q.sbk = (uint32_t)(sbk * es);
  q.scm = scm;
  q.scn = scn;
  q.bsa = bsa;
  q.bsb = bsb;
  q.bsc = p.bt.sc[0];
  q.a_bytes = (uint32_t)a_bytes;
  q.b_bytes = (uint32_t)b_bytes;
  q.n_terms = n_terms;
  for (int t = 0; t < n_terms; ++t) {
    q.a_term[t] = swap ? p.b_term[t] : p.a_term[t];
    q.b_term[t] = swap ? p.a_term[t] : p.b_term[t];
  }
  const int64_t out_n = nelem(out);
  int split = 1;
  if (f64) {
    // Microseconds, as measured: a step of 16 k of a 64 x 64 tile takes 0.62 alone on its CU, 0.56 with another one
    // there, 0.5 with more; 5 for the launch; partial results as below.  (300 x 784 over 5000, main kernel / with the
    // sums: 4 chunks = 260 blocks 82 / 89, 7 = 455 56 / 63, 10 = 650 54 / 63, 32 = 2080 52 / 65.)
    // Partial results at 4 TB/s, between other kernels that want the caches too (6 TB/s when nothing else runs): gradients of dense 784-300-100-10, batch 5000, 6 / 4 TB/s 197.4 / 190.8 us (15 / 11 shares
    // of the first weights' gradient), 784-2000-300-10, batch 1500, 385 / 380, 784-128-900-10, batch 3000, 192 / 187; at 2.5 TB/s
    // 784-650-333-10, batch 4000, goes from 374 to 408.  Two or three of them that the pass behind the product reads itself (a layer's forward
    // product) at 6 TB/s: no launch adds them up.  One layer in fifty takes other shares for it; gradients of dense 784-523-64-10, batch 1815, with 4 / 6 TB/s
    // 156.2 / 147.5 us, 784-325-64-10, 2905, 154.3 / 145.5, 784-1202-915-10, 2452, 596 / 583, 784-1814-895-10, 658, 316 / 298, 784-470-1995-10, 584, 225 / 226.
    double best = 1e300;
    const int64_t tiles = ((M + 63) / 64) * ((N + 63) / 64) * p.BT * nt;
    for (int64_t sp = 1; sp <= 64 && sp <= p.K / 64; ++sp) {
      const int64_t per_cu = (tiles * sp + ctx->num_cu - 1) / ctx->num_cu, steps = ((p.K + sp - 1) / sp + 15) / 16;
      const double step = per_cu == 1 ? 0.62 : per_cu == 2 ? 1.12 : 0.5 * per_cu;
      const double us = 5 + steps * step + (sp * nt > 1 ? 6 + (double)out_n * (sp * nt + 1) * 8 / (partials_out && sp * nt <= 3 ? 6e6 : 4e6) : 0);
      if (us < best) { best = us; split = (int)sp; }
    }
  } else if (thin) {
    // Two blocks on a CU, four where two would have 512 k and more to walk each (their loads are what counts; more blocks
    // leave more partial results).  us with the sums, two / four: 128 x 28 over 28 x 5000 (278 k) 25.7 / 26.8, 784 x 32 over
    // 8192 (128) 16.6 / 17.6, 784 x 28 over 8 x 5000 (556) 41.2 / 37.0, 784 x 10 over 8 x 10000 (1112) 75.4 / 55.5.
    const int64_t tiles = ((M + 127) / 128) * p.BT * nt;
    auto chunks = [&](int64_t per_cu) { return std::max<int64_t>(1, std::min<int64_t>(per_cu * ctx->num_cu / tiles, p.K / 64)); };
    split = (int)(p.K >= 512 * chunks(2) ? chunks(4) : chunks(2));
  } else {
    // Microseconds, as they were while the loop waited for its loads: a step of 16 k of a 128 x 128 tile 1.4 alone on its CU and 0.92 for each of
    // several; 8 for the launch with its first loads and last stores; for partial results a second launch and their bytes once
    // out and once in.  (With loads a step ahead it is 0.89 alone and 0.78 for each of two, 2048 x 2048 and 2048 x 4096 over 2048 to 8192; 2048 x 784 over
    // 8192 198 us without the sums, then 217, 300 x 5000 over 784 30 for 29.  Shares and the line below are still by the old steps, whose
    // choices are the ones measured; products just short of the line may be faster here by now.)
    double best = 1e300;
    const int64_t tiles = ((M + 127) / 128) * ((N + 127) / 128) * p.BT * nt;
    for (int64_t sp = 1; sp <= 64 && sp <= p.K / 64; ++sp) {
      const int64_t per_cu = (tiles * sp + ctx->num_cu - 1) / ctx->num_cu, steps = ((p.K + sp - 1) / sp + 15) / 16;
      const double step = per_cu == 1 ? 1.4 : 0.92 * per_cu;
      const double us = 8 + steps * step + (sp * nt > 1 ? 6 + (double)out_n * (sp * nt + 1) * 4 / 3.2e6 : 0);
      if (us < best) { best = us; split = (int)sp; }
    }
    // Small products are left to the tiles of the fp32 instruction, which submitted one after another come to 6 us and a
    // microsecond for six million multiplications of whole 64 x 64 tiles.  165 products of 8 to 1000 million, batches and long K: where this
    // says no they took 1.46 to 0.96 times as long here (3 x 125 x 194 over 141 13.6 against 9.5 us, 122 x 113 over 1251
    // 12.7 / 10.0), where it says yes 0.57 to 1.18 (52 x 101 x 264 over 107 13.8 / 24.3, 441 x 208 over 3108 20.8 / 26.5).
    const double work = (double)((M + 63) / 64 * 64) * (double)((N + 63) / 64 * 64) * (double)p.K * (double)(p.BT * nt);
    if (best >= 6 + work / 6e6) return HGPU_OK;
  }
  const int64_t BM = f64 ? 64 : 128, BN = thin ? 32 : BM;
  const int64_t tiles = ((M + BM - 1) / BM) * ((N + BN - 1) / BN);
  q.kchunk = wide_chunk(q.K, split);
  q.term_split = (int)((p.K + q.kchunk - 1) / q.kchunk);
  split = (int)(q.term_split * nt);
  if (split > 65535 || tiles * split > 0x3fffffff || (split > 1 && (double)out_n * split > 5e8)) return HGPU_OK;
  hgpu_buffer* part = nullptr;
  int rc = HGPU_OK;
  if (split > 1) {
    rc = buffer_alloc(ctx, (size_t)(out_n * split * es), &part);
    if (rc) return rc;
  }
  q.c_split_stride = split > 1 ? out_n : 0;
  {
    const double flops = 2.0 * M * N * p.K * p.BT * nt;
    const double bytes = (((double)M * p.K + (double)N * p.K) * nt + (double)M * N) * p.BT * es;
    const char* label = f64 ? "gemm_f64" : "gemm_f32";
    if (ctx->profiling && ctx->profile_shapes) {
      char buf[128];
      char terms[24] = "";
      if (nt > 1) snprintf(terms, sizeof terms, ",terms%lld", (long long)nt);
      snprintf(buf, sizeof buf, "%s[M%lldxN%lldxK%lldxB%lld,s%d,%s%s,%s,t%lldx%lld%s]", label, (long long)M, (long long)N, (long long)p.K, (long long)p.BT, split,
               sak == 1 ? "K" : "M", sbk == 1 ? "K" : "N", f64 ? "wide" : "split3", (long long)BM, (long long)BN, terms);
      label = intern_label(ctx, buf);
    }
    void* cdst = split > 1 ? part->ptr : data_ptr(out);
    LaunchArgs la{ctx->stream, 0, 0, 0, sak == 1, sbk == 1, dim3((unsigned)tiles, (unsigned)split, (unsigned)p.BT), swap ? pb : pa, swap ? pa : pb, cdst, nullptr, nullptr};
    // While a recording is open a product of a few rounds of blocks waits for others of its kernel, where nobody is about to
    // read its result: a reverse pass's weight gradients.  (Submitted one by one, the device would idle meanwhile.)
    static const bool hold = getenv("HORDEAD_NO_GROUPED_LAUNCH") == nullptr;
    if (hold && ctx->cap && !partials_out && !operands.empty() && tiles * split * p.BT <= 4 * ctx->num_cu) {
      auto job = std::make_shared<WideJob>();
      job->f64 = f64;
      job->akc = sak == 1;
      job->bkc = sbk == 1;
      job->thin = thin;
      job->j = SplitJob{q, la.A, la.B, cdst, (int)tiles, split, (int)p.BT};
      hold_wide(ctx, std::move(job), (thin ? 8 : f64 ? 4 : 0) + (sak == 1 ? 2 : 0) + (sbk == 1 ? 1 : 0), label, bytes, flops, operands, split > 1 ? part : out->buf);
    } else {
      const Reads reads = product_reads(pa, pb, n_terms, p.a_term, p.b_term);
      LaunchGuard lg(ctx, label, bytes, flops, &reads);
      la.ev_start = lg.start_event();
      la.ev_stop = lg.stop_event();
      if (f64) launch_wide_f64(q, la);
      else launch_split_f32(q, la, thin);
    }
    if (split > 1 && partials_out && split <= 3 && is_dense(out)) {
      int64_t sh[HGPU_MAX_RANK + 1], st[HGPU_MAX_RANK + 1];
      sh[0] = split;
      for (int d = 0; d < out->rank; ++d) sh[d + 1] = out->shape[d];
      dense_strides(out->rank + 1, sh, st);
      *partials_out = new_view(ctx, part, dtype, out->rank + 1, sh, st, 0);
    } else if (split > 1) {
      rc = sum_partials(ctx, dtype, out_n, (int)split, part, out);
    }
  }
  const hipError_t e = hipGetLastError();
  if (part) buffer_release(part);
  if (rc) return rc;
  if (e != hipSuccess) {
    if (partials_out && *partials_out) { hgpu_release(*partials_out); *partials_out = nullptr; }
    return check_hip(ctx, e, "gemm");
  }
  *handled = true;
  return HGPU_OK;
}

}  // namespace

namespace hg {

int try_footprint(hgpu_ctx* ctx, const GemmParams& p, int dtype, const void* pa, const void* pb, hgpu_array* out, bool* handled);
int try_smallk(hgpu_ctx* ctx, int n_terms, const hgpu_array* const* as, const hgpu_array* const* bs, int n_keep, int n_in, const hgpu_array* const* in, int c_slot,
               int n_instr, const hgpu_fused_instr* prog, const std::vector<int>& dt, int n_out, const int* out_slots, hgpu_array* const* outs, bool* handled);

// The dims of a contraction out[kept] = sum a[kept, red] * b[kept, red] sorted
// into row (M), column (N), reduced (K) and batch groups by which operand moves
// along them; false when the strides do not make it a matrix product.
bool classify_contraction(int rank, const int64_t* shape, const int64_t* st_a, const int64_t* st_b, const int64_t* st_c, int n_keep, GemmParams* p) {
  p->m.nd = p->n.nd = p->k.nd = p->bt.nd = 0;
  // Classify the dims.  The dims of a group are an index SET: any order works
  // as long as A, B and C agree, so each group is sorted with the dim that is
  // most contiguous in memory last (innermost) -- that is the dim the lanes of
  // a load run along -- and only then merged.
  struct DimRec { int64_t e, sa, sb, sc; };
  std::vector<DimRec> gm, gn, gk, gb;
  for (int i = 0; i < n_keep; ++i) {
    int64_t e = shape[i], sa = st_a[i], sb = st_b[i], sc = st_c[i];
    if (e == 1) continue;
    if (sa != 0 && sb == 0) gm.push_back({e, sa, 0, sc});
    else if (sa == 0 && sb != 0) gn.push_back({e, 0, sb, sc});
    else if (sa != 0 && sb != 0) gb.push_back({e, sa, sb, sc});
    else return false;  // an output dim neither operand depends on
  }
  for (int i = n_keep; i < rank; ++i) {
    int64_t e = shape[i], sa = st_a[i], sb = st_b[i];
    if (e == 1) continue;
    if (sa == 0 || sb == 0) return false;  // a plain sum hidden in the contraction
    gk.push_back({e, sa, sb, 0});
  }
  auto mag = [](int64_t v) { return v < 0 ? -v : v; };
  std::stable_sort(gm.begin(), gm.end(), [&](const DimRec& x, const DimRec& y) { return mag(x.sa) > mag(y.sa); });
  std::stable_sort(gn.begin(), gn.end(), [&](const DimRec& x, const DimRec& y) { return mag(x.sb) > mag(y.sb); });
  {
    // K: follow the operand that has a unit-stride K dim; when both or neither
    // do, the one that is larger (more rows to stream)
    int64_t rows_a = 1, rows_b = 1;
    for (auto& d : gm) rows_a *= d.e;
    for (auto& d : gn) rows_b *= d.e;
    bool a_unit = false, b_unit = false;
    for (auto& d : gk) { a_unit = a_unit || mag(d.sa) == 1; b_unit = b_unit || mag(d.sb) == 1; }
    bool by_a = (a_unit != b_unit) ? a_unit : rows_a >= rows_b;
    std::stable_sort(gk.begin(), gk.end(), [&](const DimRec& x, const DimRec& y) { return by_a ? mag(x.sa) > mag(y.sa) : mag(x.sb) > mag(y.sb); });
  }
  for (auto& d : gm) if (!push_dim(p->m, d.e, d.sa, d.sb, d.sc)) return false;
  for (auto& d : gn) if (!push_dim(p->n, d.e, d.sa, d.sb, d.sc)) return false;
  for (auto& d : gk) if (!push_dim(p->k, d.e, d.sa, d.sb, d.sc)) return false;
  for (auto& d : gb) if (!push_dim(p->bt, d.e, d.sa, d.sb, d.sc)) return false;
  finish(p->m);
  finish(p->n);
  finish(p->k);
  finish(p->bt);
  p->M = total(p->m);
  p->N = total(p->n);
  p->K = total(p->k);
  p->BT = total(p->bt);
  return true;
}

// Sums of as many products are a recurrence's; those of fewer keep, in a recording too, the shares of K and so the bits that
// they have submitted one by one.
constexpr int kRecurrenceTerms = 8;

// Shares of K for fp32 products on tiles of 128 x 128 that go out together: each was cut to fill the device alone, and together they
// take several rounds of short blocks, which fetch their first operands and leave partial results each.  Longer shares where
// the model of the single product (gemm_single_dims: 0.92 us a step for each of two blocks on a CU) says so; never more of them, so that the partial results have their memory.  False:
// as they are.  The three products of 128 x 128 over 27 x 5000 of a recurrence, 18 / 9 / 6 / 5 / 4 / 3 shares a term (504 to 84 blocks each), us of its whole
// gradient: 569 / 543 / 530 / 530 / 532 / 554.   (Products whose blocks differ in
// length fill one another's gaps: 2048 x 784 and 2048 x 2048 over 8192, 57 and 256 steps, lost 12 us of their gradient by this model.  fp64 and thin products come
// with more blocks to a CU, whose sums are short: not looked at.)
// The gradients' error against fp64 does not grow (weights of 128 x 128 at batch 3000 to 5000, 28 steps: 8.8e-8 to 9.6e-8 of the
// result before, 7.9e-8 to 9.5e-8 with fewer fp32 results to add up).
bool longer_wide_shares(hgpu_ctx* ctx, const WideJob* const* jobs, int n, int* shares) {
  const int slots = 2 * ctx->num_cu;
  double first = 0, best = 1e300;
  for (int d = 1; d <= 8; ++d) {
    int64_t blocks = 0, steps = 0, least = INT64_MAX;
    double sums = 0;
    int cut[kMaxWideJobs];
    for (int k = 0; k < n; ++k) {
      const SplitJob& j = jobs[k]->j;
      if (jobs[k]->f64 || jobs[k]->thin || j.p.n_terms < kRecurrenceTerms) return false;
      cut[k] = (j.p.term_split + d - 1) / d;
      const int64_t chunk = wide_chunk(j.p.K, cut[k]);
      cut[k] = (int)((j.p.K + chunk - 1) / chunk);
      const int64_t all = (int64_t)cut[k] * std::max(j.p.n_terms, 1);
      blocks += j.tiles * all * j.batches;
      steps = std::max(steps, chunk / 16);
      least = std::min(least, chunk / 16);
      sums += (double)j.p.c_split_stride * (double)all * 4 / 3.2e6;
    }
    const double us = (double)((blocks + slots - 1) / slots) * (double)steps * 1.84 + sums;
    if (d == 1) {
      if (4 * steps > 5 * least) return false;      // (blocks of different length fill one another's gaps)
      first = us;
    }
    if (us >= best) continue;
    best = us;
    std::copy(cut, cut + n, shares);
  }
  return best < 0.97 * first;
}
void set_wide_shares(WideJob& job, int shares) {
  job.j.p.kchunk = wide_chunk(job.j.p.K, shares);
  job.j.p.term_split = shares;
  job.j.splits = shares * std::max(job.j.p.n_terms, 1);
}
int wide_shares(const WideJob& job) { return job.j.splits; }
const void* wide_partials(const WideJob& job) { return job.j.C; }
const void* wide_row_partials(const WideJob& job) { return job.j.p.rows; }

hipError_t launch_wide_group(hgpu_ctx* ctx, const WideJob* const* jobs, int n) {
  SplitGroup g;
  memset(&g, 0, sizeof g);
  const SplitJob* js[kMaxSplitGroup];
  for (int k = 0; k < n; ++k) js[k] = &jobs[k]->j;
  bool rows = false;
  for (int k = 0; k < n; ++k) rows = rows || js[k]->p.rows;
  if (n == 1 && !rows) {
    const SplitJob& j = *js[0];
    LaunchArgs la{ctx->stream, 0, 0, 0, jobs[0]->akc, jobs[0]->bkc, dim3((unsigned)j.tiles, (unsigned)j.splits, (unsigned)j.batches), j.A, j.B, j.C, nullptr, nullptr};
    if (jobs[0]->f64) launch_wide_f64(j.p, la);
    else launch_split_f32(j.p, la, jobs[0]->thin);
    return hipGetLastError();
  }
  const unsigned grid = split_group(js, n, &g);
  if (jobs[0]->f64) launch_wide_f64_group(g, grid, jobs[0]->akc, jobs[0]->bkc, rows, ctx->stream);
  else launch_split_f32_group(g, grid, jobs[0]->akc, jobs[0]->bkc, jobs[0]->thin, rows, ctx->stream);
  return hipGetLastError();
}

// The shares of K of a held product that can also hand out the sums of the rows at `as` (n terms of M x K elements, rows
// `row_stride` apart); 0: it cannot.  The terms may come in another order: each is added up by itself and all meet in one sum.
// (fp64: only of several terms, which would be a launch of their own, 4.7 us for the rows of 28 x 128 x 150 where the products
// take 1.1 more for them.  A single term's sum waits with the other reductions of its kind, and fp64 additions hold the matrix cores
// up: rows of 300 x 5000 and 100 x 5000 cost their products 4.4 us, that launch 1.6.)
int wide_row_shares(const WideJob& job, int dtype, int n, const void* const* as, int64_t M, int64_t K, int64_t row_stride) {
  const SplitParams& p = job.j.p;
  if (job.f64 != (dtype == HGPU_F64) || (job.f64 && n < 2) || !job.akc || p.rows || job.j.batches != 1 || p.M != M || p.K != K || p.sam != (uint64_t)row_stride * dtype_size(dtype) || std::max(p.n_terms, 1) != n) return 0;
  std::vector<const void*> x(as, as + n), y(1, job.j.A);
  if (p.n_terms > 0) y.assign(p.a_term, p.a_term + n);
  std::sort(x.begin(), x.end());
  std::sort(y.begin(), y.end());
  return x == y ? job.j.splits : 0;
}

bool wide_takes_rows(const WideJob& job) { return job.j.p.rows != nullptr; }
void wide_take_rows(WideJob& job, void* part, const void* factor) {
  job.j.p.rows = (double*)part;
  job.j.p.row_factor = factor;
}

int try_gemm(hgpu_ctx* ctx, const hgpu_array* a, const hgpu_array* b, int n_keep, hgpu_array* out, bool* handled,
             int n_terms, const hgpu_array* const* as, const hgpu_array* const* bs, hgpu_array** partials_out) {
  // n_terms > 0: out = sum_t contract(as[t], bs[t]); all terms have the shapes,
  // strides and dtype of a = as[0], b = bs[0] (the caller has checked).
  // partials_out: a caller that runs an elementwise pass over the result anyway
  // takes the two or three partial results of a product split along K instead
  // (an array of shape [parts, kept dims...]; `out` is then left unwritten) and
  // adds them in that pass.
  *handled = false;
  if (partials_out) *partials_out = nullptr;
  if (!b) return HGPU_OK;
  if (a->dtype != HGPU_F64 && a->dtype != HGPU_F32) return HGPU_OK;
  GemmParams p;
  if (!classify_contraction(a->rank, a->shape, a->strides, b->strides, out->strides, n_keep, &p)) return HGPU_OK;
  // Worth the matrix cores only when there is reuse on both sides.
  if (p.K < 4 || p.M * p.N < 256) return HGPU_OK;
  if (p.BT > 65535) return HGPU_OK;
  // (all terms of a sum together: 28 products of 128 x 28 over 150, a minibatch's input weight gradient, ran as one
  // reduction per output, 58 us; the recurrent network at that batch, fp64: 402 -> 373 us)
  if ((double)p.M * p.N * p.K * p.BT * (n_terms > 0 ? n_terms : 1) < 2.0e6) return HGPU_OK;
  // a thousand outputs under a long K (the last layer's weight gradient: 100 x 10
  // over 5000): the split-K kernels have a handful of wavefronts to work with,
  // a wavefront per output in the reduction kernels has a thousand
  if ((p.M <= 16 || p.N <= 16) && p.K > 1024 && (double)p.M * p.N * p.K * p.BT < 2.0e7) return HGPU_OK;

  const void* pa = data_ptr(a);
  const void* pb = data_ptr(b);
  std::vector<hgpu_buffer*> operands{a->buf, b->buf};
  for (int t = 0; t < n_terms; ++t) { operands.push_back(as[t]->buf); operands.push_back(bs[t]->buf); }
  // A small output under a long K (weight gradients, the last layer of a
  // classifier) is better served by independent wavefronts than by staged tiles.
  static_assert(kMaxTerms == 32, "hgpu_contract_sum groups 32 terms to a launch");
  if (n_terms > kMaxTerms) return HGPU_OK;
  p.n_terms = n_terms;
  p.term_loop = 0;
  for (int t = 0; t < n_terms; ++t) { p.a_term[t] = data_ptr(as[t]); p.b_term[t] = data_ptr(bs[t]); }
  if (n_terms == 0) {   // windows into small footprints: operands from LDS
    int rc = try_footprint(ctx, p, a->dtype, pa, pb, out, handled);
    if (rc || *handled) return rc;
  }
  // (a side under 96 leaves more than a quarter of a 128-wide tile empty: the smaller tiles of the fp32 instruction; fp64: a side under 64)
  const bool tiled = (a->dtype == HGPU_F32 ? p.M >= 96 && p.N >= 96 : p.M >= 64 && p.N >= 64) && p.K >= 64;
  // fp64 with four 64 x 64 tiles for every CU: those run faster than the kernel over a short K, which is at its best with
  // few tiles or a program over the result (1024 x 4096 over 128 / 256 / 500: 25.6 / 42.8 / 79 us against 28.9 / 48.8 / 91;
  // 700 x 300 over 500: 18.0 against 10.2)
  const bool early = tiled && a->dtype == HGPU_F64 && ((p.M + 63) / 64) * ((p.N + 63) / 64) * p.BT >= 4 * (int64_t)ctx->num_cu;
  if (early) {
    int rc = gemm_single_dims(ctx, p, a->dtype, pa, pb, out, handled, n_terms, partials_out, operands);
    if (rc || *handled) return rc;
  }
  if ((p.K <= 512 || (p.K <= 1024 && p.M * p.N <= 160000)) && p.BT == 1) {   // the whole contracted dim in LDS: no K loop, no K table
    const hgpu_array* const* ta = n_terms > 0 ? as : &a;
    const hgpu_array* const* tb = n_terms > 0 ? bs : &b;
    const hgpu_array* none = nullptr;
    const int slot = 0;
    int rc = try_smallk(ctx, n_terms > 0 ? n_terms : 1, ta, tb, n_keep, 1, &none, 0, 0, nullptr, std::vector<int>{a->dtype}, 1, &slot, &out, handled);
    if (rc || *handled) return rc;
  }
  // Weight gradients of narrow layers, fp32: 8 to 32 rows or columns under a long K, bound by the loads of the long side, which
  // a tile of 128 x 32 reads once.  us with the sums, tiles of the fp32 instruction / so: 128 x 28 over 28 x 5000 34.9 / 25.7,
  // 50 x 28 over 20 x 1000 9.4 / 8.4, 2048 x 10 over 8192 26.1 / 21.4, 784 x 32 over 8192 24.5 / 16.6 (with six part products a tile;
  // with all eight, as now, 2 to 3 % more); error against fp64 0.4 to 0.6 of what it was, a sum of one product that product rounded,
  // as there.  Fewer columns leave the tile empty (784 x 4 over 8 x 10000 61 / 83); with rows further apart than 65536
  // elements the wider tiles read longer pieces (1000 x 20 over 50000 57.6 / 54.0, over 100,000 101 / 104).
  const int64_t k_all = p.K * (n_terms > 0 ? n_terms : 1);
  const bool thin = a->dtype == HGPU_F32 && std::min(p.M, p.N) >= 8 && std::min(p.M, p.N) <= 32 && std::max(p.M, p.N) > 32 && p.K >= 64 && p.K <= 65536 && k_all >= 4096;
  if ((tiled && !early) || thin) {
    int rc = gemm_single_dims(ctx, p, a->dtype, pa, pb, out, handled, n_terms, partials_out, operands);
    if (rc || *handled) return rc;
  }
  // (under a long K the staged kernels' coalesced tile loads win even with most of a 32-wide tile empty: 128 x 28 over 28 x 5000, 52 -> 45 us)
  if ((p.M <= 32 || p.N <= 32) && p.M <= 1024 && p.N <= 1024 && k_all < 4096) return gemm_direct(ctx, p, a->dtype, pa, pb, out, handled, n_terms);

  const int64_t nt = n_terms > 0 ? n_terms : 1;      // products summed by this launch
  const int64_t out_elems = p.M * p.N * p.BT;
  // K chunks for a tile shape, and how well the blocks then fill the device
  // (blocks / places of the rounds they take)
  auto plan_split = [&](int c, double* fill_out) {
    const int64_t bm = kTiles[c].wgm * kTiles[c].tm * 16, bn = kTiles[c].wgn * kTiles[c].tn * 16;
    const int64_t tl = ((p.M + bm - 1) / bm) * ((p.N + bn - 1) / bn);
    // small tiles do little work per K step and hide the latency of a step only
    // behind other blocks on the CU: ask for more of them
    const int64_t per_cu = bm * bn >= 128 * 64 ? 2 : (bm * bn >= 64 * 64 ? 4 : 8);
    const double slots = (double)ctx->num_cu * per_cu;
    auto fill = [&](int cand) {
      const double blocks = (double)tl * p.BT * nt * cand;
      return blocks / (std::ceil(blocks / slots) * slots);
    };
    int split = 1;
    const int64_t want = (int64_t)ctx->num_cu * per_cu;
    if (tl * p.BT * nt < want && p.K >= 8 * BK) {
      split = (int)((want + tl * p.BT * nt - 1) / (tl * p.BT * nt));
      int64_t max_split = p.K / (4 * BK);
      if (split > max_split) split = (int)max_split;
      // the partial products must stay small next to the operands, or small outright
      int64_t cap = out_elems > 0 ? (int64_t)((double)(p.M + p.N) * p.K * p.BT / (2.0 * out_elems)) : 1;
      if (out_elems * (int64_t)dtype_size(a->dtype) <= (1 << 20) && cap < 16) cap = 16;
      if (cap > 512) cap = 512;
      if (cap < 1) cap = 1;
      if (split > cap) split = (int)cap;
      if (split < 1) split = 1;
      // fewer tiles than CUs: two K halves per tile keep every CU busy, and the
      // second pass over the output costs less than the idle quarter of the device
      if (split == 1 && tl * p.BT * nt < ctx->num_cu && p.K >= 16 * BK) split = 2;
      // A few more chunks when they fill the last round of blocks: with `per_cu`
      // blocks resident on a CU, blocks run in rounds of num_cu * per_cu, and a
      // round that is three quarters empty costs as much as a full one.  (300 x 784
      // over K 5000 in 64 x 128 tiles: 11 chunks = 385 blocks take 82 us, 14 chunks
      // = 490 blocks 70 us, 15 chunks = 525 blocks 94 us.)
      if (split > 1) {
        int best_s = split;
        double best_fill = fill(split);
        const int hi = (int)std::min<int64_t>(max_split, split + (split * 3 + 9) / 10);
        for (int cand = split + 1; cand <= hi; ++cand)
          if (fill(cand) > best_fill + 0.1) { best_fill = fill(cand); best_s = cand; }
        // ... or a few less, when that makes whole rounds (28 products of 128 x 128 over
        // K 5000 in 64 x 64 tiles: 12 chunks each = 1344 blocks on 1024 places, 9 = 1008)
        const int lo = std::max(2, split - (split * 3 + 9) / 10);
        for (int cand = split - 1; cand >= lo; --cand)
          if (fill(cand) > best_fill + 0.1) { best_fill = fill(cand); best_s = cand; }
        split = best_s;
      }
    }
    if (fill_out) *fill_out = fill(split);
    return split;
  };
  // tile shape: least padded work per unit of efficiency and of device filled
  const bool f64 = a->dtype == HGPU_F64;
  int cfg = 0;
  double best = 1e300;
  double costs[kNumTiles];
  for (int c = 0; c < (a->dtype == HGPU_F32 ? kNumTiles : kFirstF32OnlyTile); ++c) {
    int64_t bm = kTiles[c].wgm * kTiles[c].tm * 16, bn = kTiles[c].wgn * kTiles[c].tn * 16;
    double padded = (double)((p.M + bm - 1) / bm * bm) * (double)((p.N + bn - 1) / bn * bn);
    // fp64: the instruction is slow next to LDS, so the operand reuse of a larger
    // tile buys little and three 64 x 64 blocks on a CU run it as well as two of
    // 64 x 128 (300 x 784 over K 5000: 64 against 74 us)
    const double eff = (f64 && bm == 64 && bn == 64) ? 0.85 : kTiles[c].eff;
    double cost = padded / eff;
    // a tile shape that cannot occupy the device even with K split pays for the idle CUs
    double blocks = (double)((p.M + bm - 1) / bm) * (double)((p.N + bn - 1) / bn) * (double)p.BT;
    double can_split = (double)(p.K / (4 * BK));
    double cap0 = (double)(p.M + p.N) * p.K / (2.0 * p.M * p.N);
    if (can_split > cap0) can_split = cap0;
    if (can_split > 512) can_split = 512;
    if (can_split < 1) can_split = 1;
    if (blocks * can_split < ctx->num_cu) cost *= ctx->num_cu / (blocks * can_split);
    costs[c] = cost;
    if (cost < best * 0.999) { best = cost; cfg = c; }
  }
  if (f64) {
    // among shapes within 15 % of the least, the one whose blocks fill their rounds
    // best (the fp32 choices were tuned without this step)
    double best2 = 1e300;
    for (int c = 0; c < kFirstF32OnlyTile; ++c) {
      if (costs[c] > best * 1.15) continue;
      double fl = 1;
      (void)plan_split(c, &fl);
      const double c2 = costs[c] / std::max(fl, 0.25);
      if (c2 < best2 * 0.999) { best2 = c2; cfg = c; }
    }
  }
  const int64_t BM = kTiles[cfg].wgm * kTiles[cfg].tm * 16, BN = kTiles[cfg].wgn * kTiles[cfg].tn * 16;
  int64_t tiles = ((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN);
  if (tiles > 0x7fffffff) return HGPU_OK;
  int split = plan_split(cfg, nullptr);
  if (const char* e = getenv("HORDEAD_GEMM_SPLIT")) {   // for measurements
    int v = atoi(e);
    if (v >= 1 && v <= p.K / BK) split = v;
  }
  p.kchunk = ((p.K + split - 1) / split + BK - 1) / BK * BK;
  p.term_split = (int)((p.K + p.kchunk - 1) / p.kchunk);
  p.split = (int)(p.term_split * nt);                // K chunks of all terms
  // terms that are one chunk each, under tiles that fill the device by
  // themselves: every block adds the terms up in its registers, no partials
  p.term_loop = (nt > 1 && p.term_split == 1 && tiles * p.BT >= ctx->num_cu / 2 &&
                 term_loop_tile(kTiles[cfg].wgm, kTiles[cfg].wgn, kTiles[cfg].tm, kTiles[cfg].tn)) ? 1 : 0;
  if (p.term_loop) p.split = 1;
  split = p.split;
  if (split > 65535) return HGPU_OK;

  size_t es = dtype_size(a->dtype);
  int64_t out_n = nelem(out);
  const void* zero_tab = nullptr;
  int rc = zero_block(ctx, &zero_tab);
  if (rc) return rc;
  hgpu_buffer* koff = nullptr;
  const int64_t Kp = p.K;
  rc = buffer_alloc(ctx, (size_t)Kp * 16, &koff);
  if (rc) return rc;
  hgpu_buffer* part = nullptr;
  if (split > 1) {
    rc = buffer_alloc(ctx, (size_t)out_n * split * es, &part);
    if (rc) { buffer_release(koff); return rc; }
  }
  p.c_split_stride = split > 1 ? out_n : 0;
  int64_t* ka = (int64_t*)koff->ptr;
  int64_t* kb = ka + p.K;
  // lanes run along k when the innermost K dim is contiguous and long enough to
  // fill a 16-lane group, or when running along m / n would be no better
  auto along_k = [](int64_t sk, int64_t ek, int64_t srow) {
    if (sk < 0) sk = -sk;
    if (srow < 0) srow = -srow;
    if (sk == 1 && (ek >= 16 || srow != 1)) return true;
    return srow != 1 && sk < srow;
  };
  bool akc = along_k(p.k.sa[p.k.nd - 1], p.k.shape[p.k.nd - 1], p.m.sa[p.m.nd - 1]);
  bool bkc = along_k(p.k.sb[p.k.nd - 1], p.k.shape[p.k.nd - 1], p.n.sb[p.n.nd - 1]);
  p.a_kc = akc ? 1 : 0;
  p.b_kc = bkc ? 1 : 0;
  p.c_rows_contig = (p.m.sc[p.m.nd - 1] == 1 && p.n.sc[p.n.nd - 1] != 1 && p.M >= 64) ? 1 : 0;
  bool va, vb;
  {
    va = vector_ok(es, akc ? p.k : p.m, (akc ? p.k.nd : p.m.nd) - 1, akc ? p.k.sa : p.m.sa);
    vb = vector_ok(es, bkc ? p.k : p.n, (bkc ? p.k.nd : p.n.nd) - 1, bkc ? p.k.sb : p.n.sb);
  }
  dim3 grid((unsigned)tiles, (unsigned)split, (unsigned)p.BT);
  {
    double flops = 2.0 * p.M * p.N * p.K * p.BT * nt;
    double bytes = (((double)p.M * p.K + (double)p.N * p.K) * nt + (double)p.M * p.N) * p.BT * es;
    const char* label = a->dtype == HGPU_F64 ? "gemm_f64" : "gemm_f32";
    if (ctx->profiling && ctx->profile_shapes) {
      char buf[128];
      char terms[24] = "";
      if (nt > 1) snprintf(terms, sizeof terms, ",terms%lld%s", (long long)nt, p.term_loop ? "loop" : "");
      snprintf(buf, sizeof buf, "%s[M%lldxN%lldxK%lldxB%lld,s%d,%s%s,t%lldx%lld%s]", label, (long long)p.M, (long long)p.N, (long long)p.K, (long long)p.BT, split, akc ? (va ? "K" : "k") : (va ? "M" : "m"), bkc ? (vb ? "K" : "k") : (vb ? "N" : "n"), (long long)BM, (long long)BN, terms);
      label = intern_label(ctx, buf);
    }
    // the helper launches are timed under their own names, the label times the MFMA kernel alone
    if (p.k.nd > 1) {
      const Reads none;
      LaunchGuard lk(ctx, "gemm_k_offsets", (double)Kp * 16, 0, &none);
      hipLaunchKernelGGL(k_koff, dim3((unsigned)((Kp + 255) / 256)), dim3(256), 0, ctx->stream, p.k, p.K, Kp, ka, kb);
      p.kmask = -1;
      p.ksa = p.ksb = 0;
    } else {   // single K dim: offsets are k * stride, the table a block of zeros
      ka = kb = (int64_t*)zero_tab;
      p.kmask = 0;
      p.ksa = p.k.sa[0];
      p.ksb = p.k.sb[0];
    }
    void* cdst = split > 1 ? part->ptr : data_ptr(out);
    LaunchArgs la{ctx->stream, cfg, 0, 0, va, vb, grid, data_ptr(a), data_ptr(b), cdst, ka, kb};
    {
      const Reads reads = product_reads(data_ptr(a), data_ptr(b), n_terms, p.a_term, p.b_term);
      LaunchGuard lg(ctx, label, bytes, flops, &reads);
      la.ev_start = lg.start_event();
      la.ev_stop = lg.stop_event();
      if (a->dtype == HGPU_F64) launch_f64(p, la);
      else launch_f32(p, la);
    }
    if (split > 1 && partials_out && split <= 3 && is_dense(out)) {
      int64_t sh[HGPU_MAX_RANK + 1], st[HGPU_MAX_RANK + 1];
      sh[0] = split;
      for (int d = 0; d < out->rank; ++d) sh[d + 1] = out->shape[d];
      dense_strides(out->rank + 1, sh, st);
      *partials_out = new_view(ctx, part, a->dtype, out->rank + 1, sh, st, 0);
    } else if (split > 1) {
      rc = sum_partials(ctx, a->dtype, out_n, (int)split, part, out);
    }
  }
  hipError_t e = hipGetLastError();
  buffer_release(koff);
  if (part) buffer_release(part);
  if (rc) return rc;
  if (e != hipSuccess) {
    if (partials_out && *partials_out) { hgpu_release(*partials_out); *partials_out = nullptr; }
    return check_hip(ctx, e, "gemm");
  }
  *handled = true;
  return HGPU_OK;
}

}  // namespace hg

// ---- the matrix cores' ceiling, measured -----------------------------------
// Loops of nothing but one MFMA instruction on independent accumulators: what
// a product kernel built on that instruction cannot exceed on this part.
namespace {
typedef __attribute__((ext_vector_type(4))) double probe_d4;
typedef __attribute__((ext_vector_type(4))) float probe_f4;
typedef __attribute__((ext_vector_type(16))) float probe_f16;

__global__ void __launch_bounds__(256) mfma_probe_f64_16x16x4(double* out, int iters) {
  probe_d4 acc[4];
  for (int i = 0; i < 4; ++i) acc[i] = probe_d4{0, 0, 0, 0};
  const double a = threadIdx.x * 0.001, b = threadIdx.x * 0.002;
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc[i], 0, 0, 0);
  }
  double s = 0;
  for (int i = 0; i < 4; ++i) s += acc[i][0] + acc[i][1] + acc[i][2] + acc[i][3];
  out[blockIdx.x * 256 + threadIdx.x] = s;
}
__global__ void __launch_bounds__(256) mfma_probe_f64_4x4x4(double* out, int iters) {
  double acc[8];
  for (int i = 0; i < 8; ++i) acc[i] = 0;
  const double a = threadIdx.x * 0.001, b = threadIdx.x * 0.002;
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, acc[i], 0, 0, 0);
  }
  double s = 0;
  for (int i = 0; i < 8; ++i) s += acc[i];
  out[blockIdx.x * 256 + threadIdx.x] = s;
}
__global__ void __launch_bounds__(256) mfma_probe_f32_16x16x4(float* out, int iters) {
  probe_f4 acc[4];
  for (int i = 0; i < 4; ++i) acc[i] = probe_f4{0, 0, 0, 0};
  const float a = threadIdx.x * 0.001f, b = threadIdx.x * 0.002f;
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc[i], 0, 0, 0);
  }
  float s = 0;
  for (int i = 0; i < 4; ++i) s += acc[i][0] + acc[i][1] + acc[i][2] + acc[i][3];
  out[blockIdx.x * 256 + threadIdx.x] = s;
}
__global__ void __launch_bounds__(256) mfma_probe_f32_32x32x2(float* out, int iters) {
  probe_f16 acc[2];
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 16; ++j) acc[i][j] = 0;
  const float a = threadIdx.x * 0.001f, b = threadIdx.x * 0.002f;
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int i = 0; i < 2; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc[i], 0, 0, 0);
  }
  float s = 0;
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 16; ++j) s += acc[i][j];
  out[blockIdx.x * 256 + threadIdx.x] = s;
}
// The same instruction fed the way a product kernel feeds it: four wavefronts
// hold a 64 x 64 tile (2 x 2 blocks each), every K step of 16 reads its
// fragments from LDS and ends with a barrier; nothing is loaded from memory.
__global__ void __launch_bounds__(256) mfma_probe_f64_16x16x4_lds(double* out, int iters) {
  __shared__ double As[16][65], Bs[16][65];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, wm = wave >> 1, wn = wave & 1;
  for (int i = t; i < 16 * 65; i += 256) { (&As[0][0])[i] = i * 1e-3; (&Bs[0][0])[i] = i * 2e-3; }
  __syncthreads();
  probe_d4 acc[2][2];
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j) acc[i][j] = probe_d4{0, 0, 0, 0};
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int kk = 0; kk < 16; kk += 4) {
      double fa[2], fb[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) fa[i] = As[kk + (lane >> 4)][wm * 32 + i * 16 + (lane & 15)];
#pragma unroll
      for (int j = 0; j < 2; ++j) fb[j] = Bs[kk + (lane >> 4)][wn * 32 + j * 16 + (lane & 15)];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[i], fb[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  double s = 0;
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j) s += acc[i][j][0] + acc[i][j][1] + acc[i][j][2] + acc[i][j][3];
  out[blockIdx.x * 256 + t] = s;
}
}  // namespace

extern "C" int hgpu_mfma_probe(hgpu_ctx* ctx, int variant, int iters, double* tflops) {
  if (!ctx || !tflops || iters < 1) return HGPU_ERR_INVALID;
  if (int rc = no_capture(ctx, "mfma_probe")) return rc;
  // 16 wavefronts per CU: every SIMD has four to pick from; the LDS-fed variants 4, 5, 6 run one, two, four per SIMD
  const int blocks = ctx->num_cu * (variant == 4 ? 1 : variant == 5 ? 2 : 4);
  hgpu_buffer* buf = nullptr;
  int rc = buffer_alloc(ctx, (size_t)blocks * 256 * 8, &buf);
  if (rc) return rc;
  double flops_per_wave_iter = 0;
  auto launch = [&]() {
    switch (variant) {
      case 0: hipLaunchKernelGGL(mfma_probe_f64_16x16x4, dim3(blocks), dim3(256), 0, ctx->stream, (double*)buf->ptr, iters); flops_per_wave_iter = 4 * 2.0 * 16 * 16 * 4; break;
      case 1: hipLaunchKernelGGL(mfma_probe_f64_4x4x4, dim3(blocks), dim3(256), 0, ctx->stream, (double*)buf->ptr, iters); flops_per_wave_iter = 8 * 2.0 * 4 * 4 * 4 * 4; break;
      case 2: hipLaunchKernelGGL(mfma_probe_f32_16x16x4, dim3(blocks), dim3(256), 0, ctx->stream, (float*)buf->ptr, iters); flops_per_wave_iter = 4 * 2.0 * 16 * 16 * 4; break;
      case 3: hipLaunchKernelGGL(mfma_probe_f32_32x32x2, dim3(blocks), dim3(256), 0, ctx->stream, (float*)buf->ptr, iters); flops_per_wave_iter = 2 * 2.0 * 32 * 32 * 2; break;
      case 4: case 5: case 6:
        hipLaunchKernelGGL(mfma_probe_f64_16x16x4_lds, dim3(blocks), dim3(256), 0, ctx->stream, (double*)buf->ptr, iters);
        flops_per_wave_iter = 16 * 2.0 * 16 * 16 * 4;
        break;
      default: break;
    }
  };
  if (variant < 0 || variant > 6) { buffer_release(buf); return fail(ctx, HGPU_ERR_INVALID, "mfma_probe: variant %d", variant); }
  hipEvent_t e0, e1;
  LaunchGuard lg(ctx);
  launch();   // warm-up
  hipError_t e = hipEventCreate(&e0);
  if (e == hipSuccess) e = hipEventCreate(&e1);
  if (e == hipSuccess) {
    (void)hipEventRecord(e0, ctx->stream);
    launch();
    (void)hipEventRecord(e1, ctx->stream);
    e = hipEventSynchronize(e1);
  }
  float ms = 0;
  if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  buffer_release(buf);
  if (e != hipSuccess || ms <= 0) return check_hip(ctx, e == hipSuccess ? hipErrorUnknown : e, "mfma_probe");
  *tflops = flops_per_wave_iter * (double)iters * (double)blocks * 4.0 / ((double)ms * 1e-3) / 1e12;
  return HGPU_OK;
}
