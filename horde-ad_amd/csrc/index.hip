// Indexing kernels: gather and scatter-add driven by index ARRAYS.
//
// horde-ad's gather/scatter take an index FUNCTION and the `Concrete` backend
// evaluates it once per position on the host (tgatherZSScalar / tscatterZSScalar,
// src/HordeAd/Core/OpsConcrete.hs:1581-1665).  Here the host layer evaluates
// the function once over all positions at a time and hands over one I64 array
// per indexed dimension; each array is a view over the position space shm, so
// an index that ignores some position variables costs no memory (stride 0).
//
// Out-of-bounds rule (OpsConcrete.hs:923-950): a position with any index
// outside [0, extent) reads zeros in gather and is skipped in scatter.
//
// Scatter-add adds colliding positions in ascending row-major order of the
// positions, the reference's own order (tscatterZSScalar walks `shsEnum shm`,
// OpsConcrete.hs:1581-1619), and without atomics on data: the positions are
// sorted by destination with a stable radix sort, or counted per destination and
// put in order there, and every destination's run is summed front to back by
// one lane per element.  Results do not depend on the run and,
// for floating point, carry the rounding of that very order as long as no
// destination is hit more than 256 times; a longer run is summed in segments
// of 256 entries (each front to back) whose sums are added in ascending order,
// so that the serial part of a scatter into a handful of cells stays bounded.
#include "common.hpp"

#include <rocprim/rocprim.hpp>

using namespace hg;

namespace {

constexpr int kBlock = 256;
constexpr int kMaxIx = 8;

struct IxSpace {
  int nd;                          // merged position dims
  int n_ix;
  int64_t shape[HG_KDIMS];
  int64_t st[kMaxIx][HG_KDIMS];    // strides of each index array over the position dims
  int64_t data_st[HG_KDIMS];       // strides of the data operand over the position dims (scatter)
  const int64_t* ix[kMaxIx];
  int64_t extent[kMaxIx];          // indexed extents of the table
  int64_t table_st[kMaxIx];        // strides of the table over the indexed dims
};

__device__ __forceinline__ bool resolve(const IxSpace& sp, int64_t m, int64_t* table_off, int64_t* data_off) {
  int64_t off[kMaxIx];
#pragma unroll
  for (int k = 0; k < kMaxIx; ++k) off[k] = 0;
  int64_t doff = 0;
  int64_t r = m;
  for (int i = sp.nd - 1; i >= 0; --i) {
    int64_t c;
    if (i > 0) {
      int64_t q = r / sp.shape[i];
      c = r - q * sp.shape[i];
      r = q;
    } else {
      c = r;
    }
    doff += c * sp.data_st[i];
#pragma unroll
    for (int k = 0; k < kMaxIx; ++k)
      if (k < sp.n_ix) off[k] += c * sp.st[k][i];
  }
  bool ok = true;
  int64_t t = 0;
#pragma unroll
  for (int k = 0; k < kMaxIx; ++k) {
    if (k < sp.n_ix) {
      int64_t v = sp.ix[k][off[k]];
      ok = ok && v >= 0 && v < sp.extent[k];
      t += v * sp.table_st[k];
    }
  }
  *table_off = t;
  *data_off = doff;
  return ok;
}

// out dense [M, N]; src inner part described by `inner` (operand 0 = src strides over shn).
template <typename T>
__global__ void __launch_bounds__(kBlock) k_gather(IxSpace sp, Dims inner, int64_t M, int64_t N, const T* __restrict__ src, T* __restrict__ out) {
  int64_t total = M * N;
  int64_t step = (int64_t)gridDim.x * kBlock;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < total; i += step) {
    int64_t m = N == 1 ? i : i / N;
    int64_t n = N == 1 ? 0 : i - m * N;
    int64_t toff, doff;
    bool ok = resolve(sp, m, &toff, &doff);
    T v = T(0);
    if (ok) {
      int64_t io[1];
      decompose<1>(inner, n, io);
      v = src[toff + io[0]];
    }
    out[i] = v;
  }
}

// Slices that are contiguous in the table and a whole number of V-sized units
// (16 bytes when sizes and strides allow): a lane moves one unit, so the lanes
// of a slice read consecutive units of one place in the table, and the position
// of a slice is resolved by each of its lanes from the same few index entries
// (one cache line).  `units` = units per slice; tbl_unit = table element size /
// sizeof(V) as a fraction num/den folded into the offsets by the caller:
// table offsets arrive in elements and are scaled by es_over_v (elements per unit
// inverted: unit offset = element offset / elems_per_unit, exact by the caller's checks).
template <typename V>
__global__ void __launch_bounds__(kBlock) k_gather_units(IxSpace sp, int64_t M, int64_t units, int64_t elems_per_unit, const V* __restrict__ src, V* __restrict__ out) {
  const int64_t total = M * units;
  const int64_t step = (int64_t)gridDim.x * kBlock;
  const bool small = total < (int64_t)0x7fffffff;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < total; i += step) {
    int64_t m, u;
    if (small) {
      const uint32_t q = (uint32_t)i / (uint32_t)units;
      m = q;
      u = (uint32_t)i - q * (uint32_t)units;
    } else {
      m = i / units;
      u = i - m * units;
    }
    int64_t toff, doff;
    const bool ok = resolve(sp, m, &toff, &doff);
    V v{};
    if (ok) v = src[toff / elems_per_unit + u];
    out[i] = v;
  }
}

// The sum of the products of gathered slices with an array b [M, N]: what a gather into memory and a contraction with b would
// leave, in one pass over b and the slices.  Products and sums in double; a position out of bounds multiplies zeros.
// Bound by b (and the slices, as far as the caches do not hold the table): eight groups of V elements in flight per lane.
// The blocks' sums are added by the one that finishes last (the counters as the fused sums' kernels use them).
// 100,000 rows of 512 bytes out of 20,000 (61 MB): 19.6 us; the gather into memory 18.7, the contraction after it 18.0 and
// its partial sums 3.9.  (Four groups, each waiting for its index before the next is asked for: 26.1.)
__device__ __forceinline__ bool draws_last(unsigned* ticket, unsigned n) {
  if (__hip_atomic_fetch_add(ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != n - 1) return false;
  __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // for the next launch
  return true;
}
__device__ __forceinline__ double wave_total(double v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off);
  return v;
}
constexpr int kDotGroups = 8;     // in flight per lane
template <typename T, int V, bool ONE>
__global__ void __launch_bounds__(kBlock) k_gather_dot(IxSpace sp, int64_t M, int64_t units, const T* __restrict__ src, const T* __restrict__ b, T* __restrict__ out,
                                                        unsigned long long* part, unsigned* tickets) {
  struct alignas(sizeof(T) * V) Group { T v[V]; };
  const int64_t total = M * units, step = (int64_t)gridDim.x * kBlock;
  const bool small = total < (int64_t)0x7fffffff;
  double acc = 0;
  constexpr int F = kDotGroups;
  for (int64_t i0 = (int64_t)blockIdx.x * kBlock + threadIdx.x; i0 < total; i0 += F * step) {
    Group x[F], y[F];
    int64_t at[F], m[F], u[F], v[F];
    bool ok[F];
#pragma unroll
    for (int q = 0; q < F; ++q) {
      at[q] = i0 + q * step < total ? i0 + q * step : total - 1;
      if (small) {
        const uint32_t d = (uint32_t)at[q] / (uint32_t)units;
        m[q] = d;
        u[q] = (uint32_t)at[q] - d * (uint32_t)units;
      } else {
        m[q] = at[q] / units;
        u[q] = at[q] - m[q] * units;
      }
    }
    // loads come back in the order they were issued: the indices, then b, then the slices that the indices name
    if (ONE) {
#pragma unroll
      for (int q = 0; q < F; ++q) v[q] = sp.ix[0][m[q] * sp.st[0][0]];
    }
#pragma unroll
    for (int q = 0; q < F; ++q) y[q] = *reinterpret_cast<const Group*>(b + at[q] * V);
#pragma unroll
    for (int q = 0; q < F; ++q) {
      int64_t toff, doff;
      if (ONE) {
        ok[q] = v[q] >= 0 && v[q] < sp.extent[0];
        toff = v[q] * sp.table_st[0];
      } else {
        ok[q] = resolve(sp, m[q], &toff, &doff);
      }
      x[q] = *reinterpret_cast<const Group*>(src + (ok[q] ? toff : 0) + u[q] * V);      // (the table has a slice)
    }
#pragma unroll
    for (int q = 0; q < F; ++q)
      if (i0 + q * step < total) {
#pragma unroll
        for (int e = 0; e < V; ++e) acc += (double)(ok[q] ? x[q].v[e] : T(0)) * (double)y[q].v[e];
      }
  }
  __shared__ double red[kBlock / 64];
  __shared__ bool last;
  const int w = threadIdx.x >> 6;
  acc = wave_total(acc);
  if ((threadIdx.x & 63) == 0) red[w] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    const double tot = (red[0] + red[1]) + (red[2] + red[3]);
    const unsigned long long old = __hip_atomic_exchange(part + blockIdx.x, __double_as_longlong(tot), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("" :: "v"(old) : "memory");    // a use of the returned value: the ticket is drawn once the sum has arrived
    const unsigned n = gridDim.x, c = blockIdx.x & 15;
    last = draws_last(tickets + 32 * (c + 1), (n - c + 15) / 16) && draws_last(tickets, n < 16 ? n : 16);
  }
  __syncthreads();
  if (!last) return;
  asm volatile("" ::: "memory");
  acc = 0;
  for (unsigned i = threadIdx.x; i < gridDim.x; i += kBlock) acc += __longlong_as_double((long long)__hip_atomic_load(part + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  acc = wave_total(acc);
  if ((threadIdx.x & 63) == 0) red[w] = acc;
  __syncthreads();
  if (threadIdx.x == 0) out[0] = (T)((red[0] + red[1]) + (red[2] + red[3]));
}

// src is a view [M (position dims), N (inner dims)]; out dense [P, N], zeroed.
// Distinct positions go to distinct places (the caller's promise): plain stores.
template <typename T>
__global__ void __launch_bounds__(kBlock) k_scatter_store(IxSpace sp, Dims inner, int64_t M, int64_t N, const T* __restrict__ src, T* __restrict__ out) {
  int64_t total = M * N;
  int64_t step = (int64_t)gridDim.x * kBlock;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < total; i += step) {
    int64_t m = N == 1 ? i : i / N;
    int64_t n = N == 1 ? 0 : i - m * N;
    int64_t toff, doff;
    bool ok = resolve(sp, m, &toff, &doff);
    if (ok) {
      int64_t io[1];
      decompose<1>(inner, n, io);
      out[toff + n] = src[doff + io[0]];
    }
  }
}

// Entries of one run that a lane adds front to back.  A destination hit by at most
// kSeg positions is summed in exactly the reference's order; a longer run is cut,
// from its first entry, into segments of kSeg entries that separate lanes add up,
// and the segment sums are then added in ascending order (k_scatter_combine).
constexpr int kSeg = 256;

// key[m] = where position m's slice starts in out (the same for colliding
// positions), or `skip` when an index is out of bounds; val[m] = m.  Also clears
// long_head, one entry per kSeg sorted entries (see k_scatter_runs).
template <typename K>
__global__ void __launch_bounds__(kBlock) k_scatter_keys(IxSpace sp, int64_t M, K skip, K* __restrict__ key, uint32_t* __restrict__ val,
                                                         uint32_t* __restrict__ long_head, int64_t n_buckets) {
  int64_t step = (int64_t)gridDim.x * kBlock;
  for (int64_t m = (int64_t)blockIdx.x * kBlock + threadIdx.x; m < M; m += step) {
    int64_t toff, doff;
    bool ok = resolve(sp, m, &toff, &doff);
    key[m] = ok ? (K)toff : skip;
    val[m] = (uint32_t)m;
    if (m < n_buckets) long_head[m] = 0;
  }
}

// the data operand's offset of position m (resolve() without the index arrays)
__device__ __forceinline__ int64_t data_offset(const IxSpace& sp, int64_t m) {
  int64_t doff = 0, r = m;
  for (int i = sp.nd - 1; i >= 0; --i) {
    int64_t c = r;
    if (i > 0) { int64_t q = r / sp.shape[i]; c = r - q * sp.shape[i]; r = q; }
    doff += c * sp.data_st[i];
  }
  return doff;
}

// key / val sorted by key, equal keys in ascending position order.  One lane per
// (sorted entry, inner element); a lane works when its entry starts a SEGMENT:
// the first entry of a run, or an entry a multiple of kSeg entries after it.
// It adds the segment's slices front to back, starting from zero.  A run of one
// segment is written to `out` at once.  The segment sums of a longer run go to
// `part`, two places per bucket of kSeg sorted entries -- a bucket holds at most
// one first segment of a long run (place 1) and one later segment (place 0),
// because segments of one run start kSeg entries apart and a long run is
// longer than a bucket -- and long_head[bucket] remembers where the run starts.
// Is sorted entry `at` (key k, not the first entry of its run) the start of a later segment of a long run?
template <typename K>
__device__ __forceinline__ bool later_segment_start(const K* __restrict__ key, int64_t at, K k) {
  if (at < kSeg || key[at - kSeg] != k) return false;   // fewer than kSeg entries of this run before this one
  int64_t lo = 0, hi = at - kSeg;                       // the run's first entry: the first key that is not smaller
  while (lo < hi) {
    const int64_t mid = (lo + hi) >> 1;
    if (key[mid] < k) lo = mid + 1; else hi = mid;
  }
  return (at - lo) % kSeg == 0;
}

// Adds entries j .. end - 1 of the run with key k to acc, front to back; stops at the first other key.
// Keys, positions and values of four entries are in flight together.  Returns the first entry not added.
template <typename T, typename K>
__device__ __forceinline__ int64_t add_run(const IxSpace& sp, const K* __restrict__ key, const uint32_t* __restrict__ val, const T* __restrict__ src, int64_t io,
                                           K k, int64_t j, int64_t end, int64_t M, T* acc) {
  while (j < end) {
    const int64_t j1 = j + 1 < M ? j + 1 : M - 1, j2 = j + 2 < M ? j + 2 : M - 1, j3 = j + 3 < M ? j + 3 : M - 1;
    const K k0 = key[j], k1 = key[j1], k2 = key[j2], k3 = key[j3];
    const uint32_t p0 = val[j], p1 = val[j1], p2 = val[j2], p3 = val[j3];
    if (k0 != k) return j;
    const bool m1 = j + 1 < end && k1 == k, m2 = m1 && j + 2 < end && k2 == k, m3 = m2 && j + 3 < end && k3 == k;
    const T v0 = src[data_offset(sp, (int64_t)p0) + io];
    const T v1 = src[data_offset(sp, (int64_t)(m1 ? p1 : p0)) + io];
    const T v2 = src[data_offset(sp, (int64_t)(m2 ? p2 : p0)) + io];
    const T v3 = src[data_offset(sp, (int64_t)(m3 ? p3 : p0)) + io];
    *acc = (T)(*acc + v0);
    if (!m1) return j + 1;
    *acc = (T)(*acc + v1);
    if (!m2) return j + 2;
    *acc = (T)(*acc + v2);
    if (!m3) return j + 3;
    *acc = (T)(*acc + v3);
    j += 4;
  }
  return j;
}

// key / val sorted by key, equal keys in ascending position order.  One lane per
// (sorted entry, inner element); a lane works when its entry starts a SEGMENT:
// the first entry of a run, or an entry a multiple of kSeg entries after it.
// It adds the segment's slices front to back, starting from zero.  A run of one
// segment is written to `out` at once.  The segment sums of a longer run go to
// `part`, two places per bucket of kSeg sorted entries -- a bucket holds at most
// one first segment of a long run (place 1) and one later segment (place 0),
// because segments of one run start kSeg entries apart and a long run is
// longer than a bucket -- and long_head[bucket] remembers where the run starts.
template <typename T, typename K>
__global__ void __launch_bounds__(kBlock) k_scatter_runs(IxSpace sp, Dims inner, int64_t M, int64_t N, K skip, const K* __restrict__ key,
                                                         const uint32_t* __restrict__ val, const T* __restrict__ src, T* __restrict__ out,
                                                         T* __restrict__ part, uint32_t* __restrict__ long_head) {
  int64_t total = M * N;
  int64_t step = (int64_t)gridDim.x * kBlock;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < total; i += step) {
    int64_t at = i / N;
    int64_t n = i - at * N;
    const K k = key[at];
    if (k == skip) continue;
    const bool head = at == 0 || key[at - 1] != k;
    if (!head && !later_segment_start(key, at, k)) continue;
    int64_t io[1];
    decompose<1>(inner, n, io);
    const int64_t end = at + kSeg < M ? at + kSeg : M;
    T acc = T(0);
    const int64_t j = add_run(sp, key, val, src, io[0], k, at, end, M, &acc);
    const bool more = j < M && key[j] == k;
    if (head && !more) {
      out[(int64_t)k + n] = acc;
    } else {
      const int64_t q = at / kSeg;
      part[(q * 2 + (head ? 1 : 0)) * N + n] = acc;
      if (head && n == 0) long_head[q] = (uint32_t)(at - q * kSeg) + 1;
    }
  }
}

// The same for single elements (N = 1), a wavefront per 64 sorted entries: EVERY
// lane fetches its entry's value (coalesced keys and positions, one gather), and
// the lane at a segment's start then collects the values of the lanes behind it
// through the wavefront, nearest first -- the same order, without a chain of
// dependent loads.  What lies beyond the wavefront's 64 entries it adds itself.
template <typename T, typename K>
__global__ void __launch_bounds__(kBlock) k_scatter_runs1(IxSpace sp, int64_t M, K skip, const K* __restrict__ key, const uint32_t* __restrict__ val,
                                                          const T* __restrict__ src, T* __restrict__ out, T* __restrict__ part, uint32_t* __restrict__ long_head) {
  const int lane = threadIdx.x & 63;
  const int64_t step = (int64_t)gridDim.x * kBlock;
  for (int64_t base = (int64_t)blockIdx.x * kBlock + (threadIdx.x & ~63); base < M; base += step) {   // the same trips for all lanes of a wavefront
    const int64_t at = base + lane;
    const bool valid = at < M;
    const K k = valid ? key[at] : skip;
    const bool live = valid && k != skip;
    const T v = live ? src[data_offset(sp, (int64_t)val[at])] : T(0);
    K before = (K)__shfl_up((unsigned long long)k, 1);
    if (lane == 0) before = at > 0 && valid ? key[at - 1] : (K)~k;
    const bool head = live && (at == 0 || before != k);
    const bool start = head || (live && later_segment_start(key, at, k));
    T acc = (T)(T(0) + v);
    bool open = start;                      // still inside the run
    int reach = 1;                          // entries of the segment this lane has added
    for (int d = 1; d < 64; ++d) {
      const K kd = (K)__shfl_down((unsigned long long)k, d);
      const T vd = __shfl_down(v, d);
      const bool take = open && lane + d < 64 && kd == k;      // (a segment is longer than a wavefront's share, so its end is not met here)
      if (open && lane + d < 64 && !take) open = false;
      if (take) { acc = (T)(acc + vd); reach = d + 1; }
      if (!__any(take)) break;
    }
    if (!start) continue;
    int64_t j = at + reach;
    if (open && lane + reach >= 64) {       // the run goes on behind the wavefront's entries
      const int64_t end = at + kSeg < M ? at + kSeg : M;
      j = add_run(sp, key, val, src, (int64_t)0, k, j, end, M, &acc);
    }
    const bool more = j < M && key[j] == k && j - at >= kSeg;
    if (head && !more) {
      out[(int64_t)k] = acc;
    } else {
      const int64_t q = at / kSeg;
      part[q * 2 + (head ? 1 : 0)] = acc;
      if (head) long_head[q] = (uint32_t)(at - q * kSeg) + 1;
    }
  }
}

// One lane per (bucket, inner element): where a long run starts in the bucket,
// its segment sums are added in ascending order and written to `out`.
template <typename T, typename K>
__global__ void __launch_bounds__(kBlock) k_scatter_combine(int64_t M, int64_t N, int64_t n_buckets, const K* __restrict__ key, const T* __restrict__ part,
                                                            const uint32_t* __restrict__ long_head, T* __restrict__ out) {
  int64_t total = n_buckets * N;
  int64_t step = (int64_t)gridDim.x * kBlock;
  for (int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x; i < total; i += step) {
    int64_t q = N == 1 ? i : i / N;
    int64_t n = N == 1 ? 0 : i - q * N;
    const uint32_t h = long_head[q];
    if (!h) continue;
    const int64_t at = q * kSeg + (int64_t)h - 1;
    const K k = key[at];
    T acc = part[(q * 2 + 1) * N + n];
    for (int64_t a = at + kSeg; a < M && key[a] == k; a += kSeg) acc = (T)(acc + part[(a / kSeg) * 2 * N + n]);
    out[(int64_t)k + n] = acc;
  }
}

// k_scatter_keys -> stable radix sort by key -> k_scatter_runs -> k_scatter_combine.
// bufs: keys (in, out), positions (in, out), sort workspace, segment sums, long_head.
template <typename K>
hipError_t scatter_sorted(hgpu_ctx* ctx, const IxSpace& sp, const Dims& inner, int64_t M, int64_t N, const hgpu_array* src, hgpu_array* o, int* rc_out) {
  const K skip = (K)nelem(o);   // larger than every slice start
  int end_bit = 1;
  while (end_bit < (int)(8 * sizeof(K)) && ((uint64_t)skip >> end_bit) != 0) ++end_bit;
  const int64_t n_buckets = (M + kSeg - 1) / kSeg;
  const size_t es = dtype_size(src->dtype);
  hgpu_buffer *kb = nullptr, *vb = nullptr, *tb = nullptr, *pb = nullptr, *hb = nullptr;
  auto drop = [&] { for (hgpu_buffer* b : {kb, vb, tb, pb, hb}) if (b) buffer_release(b); };
  int rc = buffer_alloc(ctx, (size_t)M * 2 * sizeof(K), &kb);
  if (!rc) rc = buffer_alloc(ctx, (size_t)M * 8, &vb);
  if (!rc) rc = buffer_alloc(ctx, (size_t)n_buckets * 2 * (size_t)N * es, &pb);
  if (!rc) rc = buffer_alloc(ctx, (size_t)n_buckets * 4, &hb);
  if (rc) { drop(); *rc_out = rc; return hipSuccess; }
  K* key_in = (K*)kb->ptr;
  K* key_out = key_in + M;
  uint32_t* val_in = (uint32_t*)vb->ptr;
  uint32_t* val_out = val_in + M;
  uint32_t* long_head = (uint32_t*)hb->ptr;
  size_t temp_bytes = 0;
  hipError_t e = rocprim::radix_sort_pairs(nullptr, temp_bytes, key_in, key_out, val_in, val_out, (size_t)M, 0, (unsigned)end_bit, ctx->stream);
  if (e == hipSuccess) {
    rc = buffer_alloc(ctx, temp_bytes > 0 ? temp_bytes : 1, &tb);
    if (rc) { drop(); *rc_out = rc; return hipSuccess; }
    hipLaunchKernelGGL(k_scatter_keys<K>, dim3(grid_for(M, kBlock, ctx->num_cu * 8)), dim3(kBlock), 0, ctx->stream, sp, M, skip, key_in, val_in, long_head, n_buckets);
    e = rocprim::radix_sort_pairs(tb->ptr, temp_bytes, key_in, key_out, val_in, val_out, (size_t)M, 0, (unsigned)end_bit, ctx->stream);
    if (e == hipSuccess) {
      unsigned g = grid_for(M * N, kBlock, ctx->num_cu * 8);
      if (N == 1) {
        HG_DISPATCH_DTYPE(src->dtype, T, hipLaunchKernelGGL((k_scatter_runs1<T, K>), dim3(g), dim3(kBlock), 0, ctx->stream, sp, M, skip, (const K*)key_out, (const uint32_t*)val_out,
                                                            (const T*)data_ptr(src), (T*)data_ptr(o), (T*)pb->ptr, long_head));
      } else {
        HG_DISPATCH_DTYPE(src->dtype, T, hipLaunchKernelGGL((k_scatter_runs<T, K>), dim3(g), dim3(kBlock), 0, ctx->stream, sp, inner, M, N, skip, (const K*)key_out, (const uint32_t*)val_out,
                                                            (const T*)data_ptr(src), (T*)data_ptr(o), (T*)pb->ptr, long_head));
      }
      e = hipGetLastError();
    }
    if (e == hipSuccess) {
      unsigned g = grid_for(n_buckets * N, kBlock, ctx->num_cu * 8);
      HG_DISPATCH_DTYPE(src->dtype, T, hipLaunchKernelGGL((k_scatter_combine<T, K>), dim3(g), dim3(kBlock), 0, ctx->stream, M, N, n_buckets, (const K*)key_out, (const T*)pb->ptr,
                                                          (const uint32_t*)long_head, (T*)data_ptr(o)));
      e = hipGetLastError();
    }
  }
  drop();
  *rc_out = HGPU_OK;
  return e;
}

// ---- scatter-add by counting -------------------------------------------------
// Up to 2^20 positions into a table whose cells are hit a few hundred times on average: instead of
// sorting all positions by destination, count the hits of every cell, hand every cell a stretch of `val`,
// drop the positions there in any order, and put each cell's few positions in ascending order where they are
// added up.  Short passes over 4-byte words (M positions, C cells) replace the ten launches
// of a radix or merge sort of (key, position) pairs, and the pass that adds up writes every cell, empty ones
// too, so that the result is not cleared beforehand.  100,000 rows of 512 bytes into 20,000 cells: 134 us with
// the sort, 34 us so.  The counters are the only atomics, on integers: which of its places in the stretch a
// position gets varies from run to run, the sums do not.
// A cell may be hit far more often than the average (a padding index): a run of several segments of kSeg entries is put in
// order by a block of its own, and its segments are added up wherever there is room, as after the sort.  Half of those 100,000 picks
// on one row: 1470 us with the sort, 4750 with one block per long run, 82 so.
constexpr int64_t kCountedPositions = (int64_t)1 << 20;   // (a bit for each fits the LDS of a CU: k_cell_order)
constexpr int64_t kCountedPerCell = 512;
constexpr int64_t kOrderedInPlace = (int64_t)1 << 17;     // up to here the runs of several segments are ordered in the launch that places the others (k_cell_place)
// ... and up to so many hits a cell on average: where most cells have a long run their passes over cell[] add up (131072
// positions in 300 cells: 237 us, with k_cell_order 85; 100,000 rows of 16 floats into 250: 217 and 71)
constexpr int64_t kOrderedInPlaceHits = 32;
constexpr int64_t kCountedLeast = 1024;   // up to here the library sorts in one launch: 18.8 us submitted one after another against 21.4 by counting; from 1025 on 27 against 21.4
constexpr int kSmallRun = 64;        // a cell's positions that its own group of lanes orders in LDS; up to kSeg a wavefront does

// cell[m] = position m's destination (or ~0: skipped), rank[m] = how many positions of that cell counted before it.
// A block counts its positions among themselves first, in a table of LDS (open addressing, twice as many slots
// as positions), and then adds each cell's count to the table of all with one atomic: addresses that many positions share are
// asked once a block (2^20 positions, all in 128 cells: 757 us with one atomic for a wavefront's equal cells, 95 us so).
// SPAN: most positions of a block; the small one leaves LDS for more blocks on a CU.
constexpr int kCountPositions = 4096, kCountThreads = 1024;
template <int SPAN>
__global__ void __launch_bounds__(SPAN / 4) k_cell_count(IxSpace sp, int64_t M, int span, uint32_t* __restrict__ counts, uint32_t* __restrict__ cell, uint32_t* __restrict__ rank) {
  constexpr int kSlots = 2 * SPAN, kPlaceBits = 13;
  static_assert(kSlots <= 1 << kPlaceBits && SPAN <= 1 << (32 - kPlaceBits), "a slot and a count in a word");
  __shared__ uint32_t key[kSlots], cnt[kSlots], place[SPAN];
  const int t = threadIdx.x, nt = blockDim.x, slots = 2 * span;        // (span: positions of a block, a power of two and a multiple of nt)
  for (int i = t; i < slots; i += nt) {
    key[i] = 0xffffffffu;
    cnt[i] = 0;
  }
  __syncthreads();
  const int64_t m0 = (int64_t)blockIdx.x * span;
  const int here = M - m0 < (int64_t)span ? (int)(M - m0) : span;
  for (int i = t; i < here; i += nt) {
    int64_t toff = 0, doff;
    const bool ok = resolve(sp, m0 + i, &toff, &doff);
    const uint32_t c = ok ? (uint32_t)toff : 0xffffffffu;
    cell[m0 + i] = c;
    place[i] = 0xffffffffu;
    if (!ok) continue;
    uint32_t q = (c * 0x9e3779b1u) >> 8 & (uint32_t)(slots - 1);
    for (;;) {                       // (at most half of the slots are taken: ends)
      const uint32_t was = atomicCAS(&key[q], 0xffffffffu, c);
      if (was == 0xffffffffu || was == c) break;
      q = (q + 1) & (uint32_t)(slots - 1);
    }
    place[i] = atomicAdd(&cnt[q], 1u) << kPlaceBits | q;
  }
  __syncthreads();
  for (int i0 = t; i0 < slots; i0 += 8 * nt) {       // (eight atomics in flight)
    uint32_t c[8], before[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) c[u] = i0 + u * nt < slots ? key[i0 + u * nt] : 0xffffffffu;
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (c[u] != 0xffffffffu) before[u] = atomicAdd(&counts[c[u]], cnt[i0 + u * nt]);
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (c[u] != 0xffffffffu) cnt[i0 + u * nt] = before[u];
  }
  __syncthreads();
  for (int i = t; i < here; i += nt)
    if (place[i] != 0xffffffffu) rank[m0 + i] = cnt[place[i] & (kSlots - 1)] + (place[i] >> kPlaceBits);
}

// Totals made on the way, cleared beforehand.
struct CellTotals {
  uint32_t placed;       // next free place of val
  uint32_t runs;         // runs of more than kSmallRun entries listed
  uint32_t parts;        // segments of kSeg entries of those that have several: rows of partial sums
  uint32_t unused;
};
// A run of more than kSmallRun entries: its cell, and the row of its first partial sum where it has several segments.
struct LongRun { uint32_t cell, part; };

// Where each cell's stretch of val starts (and, in the top bit, whether its run has several segments): the cells of a
// block side by side, the blocks in any order.  The totals are drawn from once a block.
constexpr uint32_t kSeveral = 0x80000000u;
constexpr int kCellsPerBlock = 1024;
__global__ void __launch_bounds__(kBlock) k_cell_starts(int64_t C, const uint32_t* __restrict__ counts, uint32_t* __restrict__ starts, CellTotals* __restrict__ totals, LongRun* __restrict__ runs, uint32_t* __restrict__ part_run) {
  __shared__ uint32_t sums[3][kBlock];
  __shared__ uint32_t base[3];
  const int t = threadIdx.x;
  const int64_t c0 = (int64_t)blockIdx.x * kCellsPerBlock + 4 * t;
  uint32_t n[4], own[3] = {0, 0, 0};        // as in CellTotals
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    n[i] = c0 + i < C ? counts[c0 + i] : 0;
    own[0] += n[i];
    own[1] += n[i] > kSmallRun ? 1 : 0;
    own[2] += n[i] > kSeg ? (n[i] + kSeg - 1) / kSeg : 0;
  }
  const int kinds = __syncthreads_or(own[1] != 0) ? 3 : 1;
  for (int k = 0; k < kinds; ++k) sums[k][t] = own[k];
  __syncthreads();
  for (int d = 1; d < kBlock; d <<= 1) {
    uint32_t v[3];
    for (int k = 0; k < kinds; ++k) v[k] = t >= d ? sums[k][t - d] : 0;
    __syncthreads();
    for (int k = 0; k < kinds; ++k) sums[k][t] += v[k];
    __syncthreads();
  }
  if (t < kinds) base[t] = atomicAdd(reinterpret_cast<uint32_t*>(totals) + t, sums[t][kBlock - 1]);
  __syncthreads();
  uint32_t at = base[0] + sums[0][t] - own[0];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (c0 + i < C) starts[c0 + i] = at | (n[i] > kSeg ? kSeveral : 0);
    at += n[i];
  }
  if (own[1] == 0) return;
  uint32_t run = base[1] + sums[1][t] - own[1], part = base[2] + sums[2][t] - own[2];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (n[i] <= kSmallRun) continue;
    const uint32_t segs = n[i] > kSeg ? (n[i] + kSeg - 1) / kSeg : 0;
    for (uint32_t k = 0; k < segs; ++k) part_run[part + k] = run;
    runs[run++] = LongRun{(uint32_t)(c0 + i), part};
    part += segs;
  }
}

// The positions of one run of several segments, in ascending order: the block goes through cell[] twice, counting and writing.
constexpr int kOrderThreads = 1024;
__device__ __forceinline__ void order_by_scan(int64_t M, uint32_t c0, const uint32_t* __restrict__ cell, uint32_t* at, uint32_t* sums) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int share = (int)((M + kOrderThreads - 1) / kOrderThreads) * 64;      // positions of a wavefront
  const int p0 = wave * share, p1 = (int64_t)p0 + share < M ? p0 + share : (int)M;
  uint32_t o = 0;
  for (int pass = 0; pass < 2; ++pass) {
    for (int p = p0; p < p1; p += 8 * 64) {
      uint32_t c[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) c[q] = p + 64 * q + lane < p1 ? cell[p + 64 * q + lane] : 0xffffffffu;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const unsigned long long hit = __ballot(c[q] == c0);
        if (pass == 1 && c[q] == c0) at[o + (uint32_t)__popcll(hit & ((1ull << lane) - 1))] = (uint32_t)(p + 64 * q + lane);
        o += (uint32_t)__popcll(hit);
      }
    }
    if (pass == 1) break;
    if (lane == 0) sums[wave] = o;
    __syncthreads();
    o = 0;
    for (int w = 0; w < wave; ++w) o += sums[w];
  }
  __syncthreads();
}

// Drops the positions into their cells' stretches.  With `order` the runs of several segments are left out and put in order
// here, a block for each, from cell[] alone, which this launch only reads: a launch less than with k_cell_order
// (2000 rows of 512 bytes submitted one after another: 21.3 -> 18.9 us), and up to 2^17 positions the passes over
// cell[] are short (50,000 of 100,000 positions: 20 us).
__global__ void __launch_bounds__(kOrderThreads) k_cell_place(int64_t M, bool order, const uint32_t* __restrict__ starts, const uint32_t* __restrict__ cell, const uint32_t* __restrict__ rank,
                                                              const CellTotals* __restrict__ totals, const LongRun* __restrict__ runs, uint32_t* val) {
  __shared__ uint32_t sums[kOrderThreads / 64];
  const uint32_t n_runs = order && totals->parts ? totals->runs : 0;
  const int64_t step = (int64_t)gridDim.x * kOrderThreads;
  for (int64_t m = (int64_t)blockIdx.x * kOrderThreads + threadIdx.x; m < M; m += step) {
    const uint32_t c = cell[m];
    if (c == 0xffffffffu) continue;
    const uint32_t at = starts[c];
    if (!(order && (at & kSeveral))) val[(at & ~kSeveral) + rank[m]] = (uint32_t)m;
  }
  for (uint32_t i = blockIdx.x; i < n_runs; i += gridDim.x) {
    const uint32_t c = runs[i].cell, at = starts[c];
    if (at & kSeveral) order_by_scan(M, c, cell, val + (at & ~kSeveral), sums);      // (the same for the whole block)
  }
}

// The same for more positions or hits, after they have been placed: runs of up to 1024 entries by their ranks, longer ones by a block with a bit of LDS per position, set for the
// run's and read off in order -- the work grows with n + M / 32, which beats sorting networks from a few hundred entries on
// and does not know a longest run; from a quarter of all positions on by order_by_scan.  The words of 32 bits stand 33
// to 32 so that lanes that read 32 of them each hit different banks.
__global__ void __launch_bounds__(kOrderThreads) k_cell_order(int64_t M, const uint32_t* __restrict__ counts, const uint32_t* __restrict__ starts, const CellTotals* __restrict__ totals,
                                                              const LongRun* __restrict__ runs, const uint32_t* __restrict__ cell, uint32_t* val) {
  __shared__ __attribute__((aligned(16))) uint32_t lds[kCountedPositions / 32 + kCountedPositions / 1024];
  __shared__ uint32_t sums[kOrderThreads / 64];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const uint32_t n_runs = totals->parts ? totals->runs : 0;
  const int words = (int)((M + 31) / 32), per = (words + kOrderThreads - 1) / kOrderThreads;
  auto word_at = [](int w) { return w + (w >> 5); };
  for (uint32_t i = blockIdx.x; i < n_runs; i += gridDim.x) {
    const uint32_t c = runs[i].cell, n = counts[c];
    if (n <= kSeg) continue;                                  // (the same for the whole block)
    uint32_t* at = val + (starts[c] & ~kSeveral);
    if ((int64_t)n * 4 >= M) {
      order_by_scan(M, c, cell, at, sums);
      continue;
    }
    if (n <= kOrderThreads) {
      const uint32_t p = (uint32_t)t < n ? at[t] : 0xffffffffu;
      lds[t] = p;
      __syncthreads();
      uint32_t r = 0;
      for (uint32_t d = 0; d < n; d += 8) {            // (up to the next eight: the places behind n hold what is never smaller)
        const uint4 x = *reinterpret_cast<const uint4*>(lds + d), y = *reinterpret_cast<const uint4*>(lds + d + 4);
        r += (x.x < p) + (x.y < p) + (x.z < p) + (x.w < p) + (y.x < p) + (y.y < p) + (y.z < p) + (y.w < p);
      }
      if ((uint32_t)t < n) at[r] = p;
      __syncthreads();
      continue;
    }
    for (int w = t; w < words; w += kOrderThreads) lds[word_at(w)] = 0;
    __syncthreads();
    for (uint32_t e = t; e < n; e += 4 * kOrderThreads) {
      uint32_t p[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) p[q] = e + q * kOrderThreads < n ? at[e + q * kOrderThreads] : at[e];
#pragma unroll
      for (int q = 0; q < 4; ++q) atomicOr(&lds[word_at((int)(p[q] >> 5))], 1u << (p[q] & 31));
    }
    __syncthreads();
    uint32_t total = 0;
    for (int w = t * per; w < (t + 1) * per && w < words; ++w) total += (uint32_t)__popc(lds[word_at(w)]);
    uint32_t scan = total;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t v = (uint32_t)__shfl_up(scan, d);
      if (lane >= d) scan += v;
    }
    if (lane == 63) sums[wave] = scan;
    __syncthreads();
    uint32_t o = scan - total;
    for (int w = 0; w < wave; ++w) o += sums[w];
    for (int w = t * per; w < (t + 1) * per && w < words; ++w)
      for (uint32_t bits = lds[word_at(w)]; bits; bits &= bits - 1) at[o++] = (uint32_t)(32 * w) + (uint32_t)(__ffs((int)bits) - 1);
    __syncthreads();
  }
}

template <typename T, int V> struct UnitOf { using type = T __attribute__((ext_vector_type(V), aligned(sizeof(T)))); };
template <typename T> struct UnitOf<T, 1> { using type = T; };

// Adds the slices of `n` positions, in the order of `list`, to acc, F loads in flight.
// LINEAR: the positions have one merged dim, a position's slice starts at a multiple of its number (divisions in front of
// every load otherwise: 100,000 rows of 16 floats into 400 cells 99 us, 73 without).
template <typename U, int F, bool LINEAR, typename T>
__device__ __forceinline__ U add_positions(const IxSpace& sp, U acc, const uint32_t* list, uint32_t n, const T* __restrict__ from) {
  auto slice = [&](uint32_t m) { return from + (LINEAR ? (int64_t)m * sp.data_st[0] : data_offset(sp, (int64_t)m)); };
  uint32_t j = 0;
  for (; j + F <= n; j += F) {
    U x[F];
#pragma unroll
    for (int q = 0; q < F; ++q) x[q] = *reinterpret_cast<const U*>(slice(list[j + q]));
#pragma unroll
    for (int q = 0; q < F; ++q) acc = (U)(acc + x[q]);
  }
  for (; j < n; ++j) acc = (U)(acc + *reinterpret_cast<const U*>(slice(list[j])));
  return acc;
}

// Everything the last pass reads besides its operands.
struct CellLists {
  const uint32_t *counts, *starts, *val;
  const CellTotals* totals;
  const LongRun* runs;
  const uint32_t* part_run;
  uint32_t* tickets;       // one per row of partial sums and piece of G units (those of a run's first row are used)
  void* parts;             // [rows][N]
};

// dst[0 .. n) = src[0 .. n), distinct numbers, in ascending order: every lane finds the ranks of its share, E numbers at a time.
template <int E>
__device__ __forceinline__ void order_few(const uint32_t* src, uint32_t n, uint32_t* dst, int lane, int lanes) {
  for (uint32_t e = lane; e < n; e += E * lanes) {
    uint32_t p[E], r[E];
#pragma unroll
    for (int q = 0; q < E; ++q) {
      p[q] = e + q * lanes < n ? src[e + q * lanes] : 0;
      r[q] = 0;
    }
    for (uint32_t d = 0; d < n; ++d) {
      const uint32_t x = src[d];
#pragma unroll
      for (int q = 0; q < E; ++q) r[q] += x < p[q] ? 1 : 0;
    }
#pragma unroll
    for (int q = 0; q < E; ++q)
      if (e + q * lanes < n) dst[r[q]] = p[q];
  }
}
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// First the segments of the runs that have several, a group of G lanes (8 to 64) for every G units of V elements of each:
// the positions come through LDS and the slices are added front to back, eight loads in flight (115 us for a segment of
// rows of 512 bytes when every round of loads waited for its positions, 60 so).  Whoever finishes a run's last segment
// adds the sums in ascending order (the sums are written, a fence, a ticket; such runs are rare enough for fences).
// Then the runs of one segment, a wavefront for every 64 units: their positions are put in order in LDS.
// Then the cells, each in `stretches` pieces (more than one where few cells with wide slices would leave the
// device idle), a group of lanes for each: the positions are put in order in LDS, and the lanes run along the
// piece and add the positions' slices in ascending order, four loads in flight.
template <typename T, int V, bool LINEAR>
__global__ void __launch_bounds__(kBlock, 6) k_cell_sum(IxSpace sp, Dims inner, int64_t C, int64_t N, int G, int64_t stretches, CellLists in, const T* __restrict__ src, T* __restrict__ out) {
  using U = typename UnitOf<T, V>::type;
  constexpr int kWaveWords = 64 / 8 * 2 * kSmallRun;         // two lists for each group of eight lanes, or two of a whole segment
  static_assert(kWaveWords >= 2 * kSeg, "a segment's positions twice");
  __shared__ uint32_t lists[kBlock / 64][kWaveWords];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t units = N / V;
  auto element = [&](int64_t u) {
    int64_t io[1] = {u * V};
    if constexpr (V == 1) decompose<1>(inner, u, io);
    return io[0];
  };
  const int g = threadIdx.x / G, l = threadIdx.x % G, groups = kBlock / G, in_wave = 64 / G;
  uint32_t* list = lists[wave] + lane / G * (2 * kSmallRun);
  const uint32_t n_parts = in.totals->parts, n_runs = in.totals->runs;
  // each kind of work starts at the block where the one before it ended: they go on side by side
  int64_t block = blockIdx.x;
  auto behind = [&](int64_t used) {
    block -= used % gridDim.x;
    if (block < 0) block += gridDim.x;
  };
  {
    const int64_t pieces = (units + G - 1) / G, items = (int64_t)n_parts * pieces;
    for (int64_t i0 = (block * (kBlock / 64) + wave) * in_wave; i0 < items; i0 += (int64_t)gridDim.x * groups) {
      const int64_t i = i0 + lane / G;
      const bool ok = i < items;
      const int64_t row = ok ? i / pieces : 0, piece = ok ? i - row * pieces : 0, u = piece * G + l;
      const LongRun run = in.runs[in.part_run[row]];
      const uint32_t n = in.counts[run.cell], segs = (n + kSeg - 1) / kSeg, at = (uint32_t)row - run.part;
      const uint32_t len = !ok ? 0 : n - at * kSeg < (uint32_t)kSeg ? n - at * kSeg : (uint32_t)kSeg;
      const uint32_t* mine = in.val + (in.starts[run.cell] & ~kSeveral) + at * kSeg;
      const bool live = ok && u < units;
      const T* from = src + (live ? element(u) : 0);
      U* part = reinterpret_cast<U*>((T*)in.parts + (int64_t)run.part * N + u * V);
      U acc{};
      for (uint32_t e0 = 0; e0 < (uint32_t)kSeg; e0 += 2 * kSmallRun) {
        const uint32_t m = len <= e0 ? 0 : len - e0 < 2 * kSmallRun ? len - e0 : 2 * kSmallRun;
        for (uint32_t e = l; e < m; e += G) list[e] = mine[e0 + e];
        wave_sync();
        if (live) acc = add_positions<U, 8, LINEAR>(sp, acc, list, m, from);
        wave_sync();
      }
      if (live) part[(int64_t)at * units] = acc;
      __threadfence();
      uint32_t before = 0;
      if (l == 0 && ok) before = atomicAdd(&in.tickets[(int64_t)run.part * pieces + piece], 1u);
      before = (uint32_t)__shfl(before, lane / G * G);
      if (live && before == segs - 1) {
        __threadfence();
        acc = part[0];
        uint32_t j = 1;
        for (; j + 8 <= segs; j += 8) {
          U x[8];
#pragma unroll
          for (int q = 0; q < 8; ++q) x[q] = part[(int64_t)(j + q) * units];
#pragma unroll
          for (int q = 0; q < 8; ++q) acc = (U)(acc + x[q]);
        }
        for (; j < segs; ++j) acc = (U)(acc + part[(int64_t)j * units]);
        *reinterpret_cast<U*>(out + (int64_t)run.cell * N + u * V) = acc;
      }
    }
  }
  if (n_runs > 0) {
    if (n_parts > 0) behind(((int64_t)n_parts * ((units + G - 1) / G) + groups - 1) / groups);
    const int64_t pieces = (units + 63) / 64, items = (int64_t)n_runs * pieces;
    uint32_t *raw = lists[wave], *sorted = raw + kSeg;
    for (int64_t i = block * (kBlock / 64) + wave; i < items; i += (int64_t)gridDim.x * (kBlock / 64)) {
      const int64_t r = i / pieces, u = (i - r * pieces) * 64 + lane;
      const uint32_t c = in.runs[r].cell, n = in.counts[c];
      if (n > (uint32_t)kSeg) continue;
      const uint32_t* mine = in.val + in.starts[c];
      for (uint32_t e = lane; e < n; e += 64) raw[e] = mine[e];
      wave_sync();
      order_few<4>(raw, n, sorted, lane, 64);
      wave_sync();
      if (u < units) *reinterpret_cast<U*>(out + (int64_t)c * N + u * V) = add_positions<U, 8, LINEAR>(sp, U{}, sorted, n, src + element(u));
      wave_sync();
    }
    behind((items + kBlock / 64 - 1) / (kBlock / 64));
  }
  uint32_t *raw = list, *sorted = list + kSmallRun;
  const int64_t step = (int64_t)gridDim.x * groups, len = (units + stretches - 1) / stretches;
  for (int64_t i = block * groups + g; i < C * stretches; i += step) {
    const int64_t c = stretches == 1 ? i : i / stretches, u0 = (i - c * stretches) * len, u1 = u0 + len < units ? u0 + len : units;
    const uint32_t n = in.counts[c];
    if (n > kSmallRun) continue;
    const uint32_t* mine = in.val + in.starts[c];
    for (uint32_t e = l; e < n; e += G) raw[e] = mine[e];
    wave_sync();
    order_few<1>(raw, n, sorted, l, G);
    wave_sync();
    for (int64_t u = u0 + l; u < u1; u += G)
      *reinterpret_cast<U*>(out + c * N + u * V) = add_positions<U, 4, LINEAR>(sp, U{}, sorted, n, src + element(u));
    wave_sync();
  }
}

// What a scatter reads (it writes new arrays only).
Reads scatter_reads(const IxSpace& sp, const hgpu_array* src) {
  Reads r{data_ptr(src)};
  for (int k = 0; k < sp.n_ix; ++k) r.push_back(sp.ix[k]);
  return r;
}

// k_cell_count -> k_cell_starts -> k_cell_place (-> k_cell_order) -> k_cell_sum.  sp's table strides are in slices; every
// element of o is written.
hipError_t scatter_counted(hgpu_ctx* ctx, const IxSpace& sp, const Dims& inner, int64_t M, int64_t N, int64_t C, const hgpu_array* src, hgpu_array* o, int* rc_out) {
  const size_t es = dtype_size(src->dtype);
  // 16-byte units when the slices are contiguous and every one starts on a boundary of its elements
  const bool contiguous = inner.nd == 1 && (inner.st[0][0] == 1 || N == 1);
  const int V = es >= 4 && (src->dtype == HGPU_F64 || src->dtype == HGPU_F32) && contiguous && N % (int64_t)(16 / es) == 0 ? (int)(16 / es) : 1;
  const int64_t units = N / V;
  int G = 8;
  while (G < 64 && G < units) G <<= 1;
  // Pieces of a cell: as many as leave every lane four units, until the lanes fill the device.  (1500 slices of 120 KB into
  // three cells: 434 us with the sort, 10.4 ms with a group of lanes per cell, 90 so.)
  const int64_t room = ((int64_t)ctx->num_cu * 2048 + C * G - 1) / (C * G), longest = (units + 4 * G - 1) / (4 * G);
  const int64_t stretches = std::max<int64_t>(1, std::min(room, longest));
  const int64_t max_runs = M / (kSmallRun + 1) + 1;
  const int64_t max_parts = M > kSeg ? M / kSeg + M / (kSeg + 1) + 1 : 0;       // (a run of several segments has more than kSeg entries)
  const int64_t pieces = (units + G - 1) / G, n_tickets = max_parts * pieces;
  const int64_t head = (C + 4 + n_tickets + 3) / 4 * 4;        // counters, totals, tickets: cleared together
  const int64_t words = (head + C + 3 * M + 2 * max_runs + max_parts + 3) / 4 * 4;
  hgpu_buffer* wb = nullptr;
  *rc_out = buffer_alloc(ctx, (size_t)words * 4 + (size_t)(max_parts * N) * es, &wb);
  if (*rc_out) return hipSuccess;
  uint32_t* counts = (uint32_t*)wb->ptr;
  CellTotals* totals = (CellTotals*)(counts + C);
  uint32_t* starts = counts + head;
  uint32_t* cell = starts + C;
  uint32_t* rank = cell + M;
  uint32_t* val = rank + M;
  LongRun* runs = (LongRun*)(val + M);
  uint32_t* part_run = val + M + 2 * max_runs;
  *rc_out = zero_fill(ctx, counts, (size_t)head * 4, true);
  if (*rc_out) { buffer_release(wb); return hipSuccess; }
  const Reads reads = scatter_reads(sp, src);
  LaunchGuard lg(ctx, "scatter_counted", 2.0 * M * N * es + 8.0 * M * sp.n_ix, (double)M * N, &reads);
  // Positions of a block: few while latency counts, then as many as leave every CU a block; and where cells are hit more
  // than 64 times, no more than 64 blocks if that can be had, since one address takes their atomics one after
  // another (100,000 positions in 400 cells: 390 blocks 44 us).
  int span = kBlock;
  while (span < kCountPositions && ((int64_t)span * ctx->num_cu * (M <= kOrderedInPlace ? 2 : 1) < M || (M > 64 * C && M > (int64_t)64 * span))) span <<= 1;
  const int nt = std::clamp(span / 4, kBlock, kCountThreads);
  const dim3 gk((unsigned)((M + span - 1) / span));
  if (span <= 4 * kBlock) hipLaunchKernelGGL(k_cell_count<4 * kBlock>, gk, dim3((unsigned)nt), 0, ctx->stream, sp, M, span, counts, cell, rank);
  else hipLaunchKernelGGL(k_cell_count<kCountPositions>, gk, dim3((unsigned)nt), 0, ctx->stream, sp, M, span, counts, cell, rank);
  hipLaunchKernelGGL(k_cell_starts, dim3((unsigned)((C + kCellsPerBlock - 1) / kCellsPerBlock)), dim3(kBlock), 0, ctx->stream, C, (const uint32_t*)counts, starts, totals, runs, part_run);
  const bool in_place = M <= kOrderedInPlace && M <= kOrderedInPlaceHits * C;
  hipLaunchKernelGGL(k_cell_place, dim3(grid_for(M, kOrderThreads, ctx->num_cu * 2)), dim3(kOrderThreads), 0, ctx->stream, M, in_place, (const uint32_t*)starts, (const uint32_t*)cell,
                     (const uint32_t*)rank, (const CellTotals*)totals, (const LongRun*)runs, val);
  if (!in_place)
    hipLaunchKernelGGL(k_cell_order, dim3((unsigned)ctx->num_cu), dim3(kOrderThreads), 0, ctx->stream, M, (const uint32_t*)counts, (const uint32_t*)starts, (const CellTotals*)totals, (const LongRun*)runs,
                       (const uint32_t*)cell, val);
  const CellLists in{counts, starts, val, totals, runs, part_run, counts + C + 4, (char*)wb->ptr + words * 4};
  // lanes for the cells' pieces, and for the segments and the runs of one segment that a mean number of hits lets expect
  const int64_t hits = M / C, long_lanes = hits <= kSmallRun / 2 ? 0 : (M / kSeg + 1) * pieces * G + std::min(C, max_runs) * ((units + 63) / 64) * 64;
  const unsigned gc = grid_for(C * stretches * G + std::max(long_lanes, (M / kSeg + 1) * pieces * G), kBlock, ctx->num_cu * 16);
  auto sum = [&](auto kernel, auto* from, auto* to) { hipLaunchKernelGGL(kernel, dim3(gc), dim3(kBlock), 0, ctx->stream, sp, inner, C, N, G, stretches, in, from, to); };
  auto sum_as = [&](auto linear) {
    constexpr bool L = decltype(linear)::value;
    if (V == 2) sum(k_cell_sum<double, 2, L>, (const double*)data_ptr(src), (double*)data_ptr(o));
    else if (V == 4) sum(k_cell_sum<float, 4, L>, (const float*)data_ptr(src), (float*)data_ptr(o));
    else HG_DISPATCH_DTYPE(src->dtype, T, sum(k_cell_sum<T, 1, L>, (const T*)data_ptr(src), (T*)data_ptr(o)));
  };
  if (sp.nd == 1) sum_as(std::true_type{});
  else sum_as(std::false_type{});
  const hipError_t e = hipGetLastError();
  buffer_release(wb);
  return e;
}

int build_space(hgpu_ctx* ctx, const char* who, int n_ix, const hgpu_array* const* ix, int rank_m, const int64_t* shm,
                const int64_t* data_st, IxSpace* sp) {
  if (n_ix < 0 || n_ix > kMaxIx) return fail(ctx, HGPU_ERR_UNSUPPORTED, "%s: %d index arrays (at most %d)", who, n_ix, kMaxIx);
  int64_t zero[HGPU_MAX_RANK] = {0};
  // merge position dims jointly over all index arrays and the data operand
  const int64_t* sts[kMaxIx + 1];
  for (int k = 0; k < n_ix; ++k) {
    const hgpu_array* a = ix[k];
    if (!a || a->dtype != HGPU_I64) return fail(ctx, HGPU_ERR_INVALID, "%s: index array %d is not I64", who, k);
    if (a->rank != rank_m) return fail(ctx, HGPU_ERR_INVALID, "%s: index array %d has rank %d, positions have rank %d", who, k, a->rank, rank_m);
    for (int i = 0; i < rank_m; ++i)
      if (a->shape[i] != shm[i]) return fail(ctx, HGPU_ERR_INVALID, "%s: index array %d differs from shm in dim %d", who, k, i);
    sts[k] = a->strides;
  }
  sts[n_ix] = data_st ? data_st : zero;
  // collapse() handles 4 operands; do the merge here for up to kMaxIx + 1.
  int nops = n_ix + 1;
  sp->nd = 0;
  sp->n_ix = n_ix;
  for (int i = 0; i < rank_m; ++i) {
    if (shm[i] == 1) continue;
    bool merged = false;
    if (sp->nd > 0) {
      int p = sp->nd - 1;
      bool ok = true;
      for (int k = 0; k < nops; ++k) {
        int64_t prev = k < n_ix ? sp->st[k][p] : sp->data_st[p];
        if (prev != sts[k][i] * shm[i]) { ok = false; break; }
      }
      if (ok) {
        sp->shape[p] *= shm[i];
        for (int k = 0; k < n_ix; ++k) sp->st[k][p] = sts[k][i];
        sp->data_st[p] = sts[n_ix][i];
        merged = true;
      }
    }
    if (!merged) {
      if (sp->nd == HG_KDIMS) return fail(ctx, HGPU_ERR_UNSUPPORTED, "%s: more than %d merged position dims", who, HG_KDIMS);
      sp->shape[sp->nd] = shm[i];
      for (int k = 0; k < n_ix; ++k) sp->st[k][sp->nd] = sts[k][i];
      sp->data_st[sp->nd] = sts[n_ix][i];
      sp->nd++;
    }
  }
  if (sp->nd == 0) {
    sp->nd = 1;
    sp->shape[0] = 1;
    for (int k = 0; k < n_ix; ++k) sp->st[k][0] = 0;
    sp->data_st[0] = 0;
  }
  for (int k = 0; k < kMaxIx; ++k) {
    sp->ix[k] = k < n_ix ? (const int64_t*)data_ptr(ix[k]) : nullptr;
    sp->extent[k] = 0;
    sp->table_st[k] = 0;
  }
  return HGPU_OK;
}

}  // namespace

namespace hg {

struct GatherJob : HeldJob {
  IxSpace sp;
  int64_t M, N, units, epu;     // positions, elements of a slice; of `unit` bytes each: units of a slice, elements of a unit
  int unit;                     // 0: element by element
  int dtype;
  const void* src;
  void* out;
  hipError_t launch(hgpu_ctx* ctx, hipEvent_t start, hipEvent_t stop) override {
    const dim3 g(grid_for(M * units, kBlock, ctx->num_cu * 16));
    auto go = [&](auto* u) {
      using U = std::remove_pointer_t<decltype(u)>;
      if (start || stop) hipExtLaunchKernelGGL(k_gather_units<U>, g, dim3(kBlock), 0, ctx->stream, start, stop, 0, sp, M, units, epu, (const U*)src, (U*)out);
      else hipLaunchKernelGGL(k_gather_units<U>, g, dim3(kBlock), 0, ctx->stream, sp, M, units, epu, (const U*)src, (U*)out);
    };
    if (unit == 16) go((uint4*)nullptr);
    else if (unit == 8) go((uint64_t*)nullptr);
    else go((uint32_t*)nullptr);
    return hipGetLastError();
  }
};
std::shared_ptr<GatherJob> gather_into_locked(hgpu_ctx* ctx, const hgpu_buffer* b) { return std::dynamic_pointer_cast<GatherJob>(held_writer_locked(ctx, b)); }

// The held gather's result must be all of a or b, side by side, and the other operand dense too: then both run along the same
// linear index.  The gather stays held; it is dropped if nobody else has its result.
int try_gather_dot(hgpu_ctx* ctx, const hgpu_array* a, const hgpu_array* b, const hgpu_array* o, bool* handled) {
  *handled = false;
  if (!dtype_is_float(a->dtype) || !a->buf || !b->buf || !is_dense(a) || !is_dense(b)) return HGPU_OK;
  std::shared_ptr<GatherJob> job;
  const hgpu_array *g = a, *y = b;
  {
    std::lock_guard<LaunchMutex> lk(ctx->launch_mu);
    job = gather_into_locked(ctx, a->buf);
    if (!job && (job = gather_into_locked(ctx, b->buf))) std::swap(g, y);
  }
  if (!job || job->dtype != g->dtype || job->out != data_ptr(g) || job->M * job->N != nelem(g)) return HGPU_OK;
  const size_t es = dtype_size(g->dtype);
  const int V = std::max(1, job->unit / (int)es) > 1 && ((uintptr_t)data_ptr(y) % (uintptr_t)job->unit) == 0 ? job->unit / (int)es : 1;
  const int64_t units = job->N / V;
  const unsigned grid = grid_for((job->M * units + kDotGroups - 1) / kDotGroups, kBlock, ctx->num_cu * 8);
  void* tickets = nullptr;
  hgpu_buffer* part = nullptr;
  int rc = ticket_block(ctx, &tickets);
  if (!rc) rc = buffer_alloc(ctx, (size_t)grid * 8, &part);
  if (rc) return rc;
  hipError_t e = hipSuccess;
  {
    Reads reads{data_ptr(y)};
    LaunchGuard lg(ctx, "gather_dot", (2.0 * job->M * job->N + 1) * es + 8.0 * job->M * job->sp.n_ix, 2.0 * job->M * job->N, &reads);
    if (gather_into_locked(ctx, g->buf) == job) {      // (else it has gone out meanwhile: y reads it too, the memory was needed, another thread)
      auto go = [&](auto* t, auto v) {
        using T = std::remove_pointer_t<decltype(t)>;
        auto launch = [&](auto kernel) {
          hipLaunchKernelGGL(kernel, dim3(grid), dim3(kBlock), 0, ctx->stream, job->sp, job->M, units, (const T*)job->src, (const T*)data_ptr(y), (T*)data_ptr(o),
                             (unsigned long long*)part->ptr, (unsigned*)tickets);
        };
        if (job->sp.nd == 1 && job->sp.n_ix == 1) launch(k_gather_dot<T, decltype(v)::value, true>);
        else launch(k_gather_dot<T, decltype(v)::value, false>);
      };
      if (g->dtype == HGPU_F64) {
        if (V == 2) go((double*)nullptr, std::integral_constant<int, 2>{});
        else go((double*)nullptr, std::integral_constant<int, 1>{});
      } else {
        if (V == 4) go((float*)nullptr, std::integral_constant<int, 4>{});
        else if (V == 2) go((float*)nullptr, std::integral_constant<int, 2>{});
        else go((float*)nullptr, std::integral_constant<int, 1>{});
      }
      e = hipGetLastError();
      *handled = true;
    }
  }
  buffer_release(part);
  return e == hipSuccess ? HGPU_OK : check_hip(ctx, e, "gather_dot");
}

}  // namespace hg

extern "C" {

int hgpu_gather(hgpu_ctx* ctx, const hgpu_array* src, int n_ix, const hgpu_array* const* ix, int rank_m, const int64_t* shm, hgpu_array** out) {
  if (!ctx || !src || !out || rank_m < 0) return HGPU_ERR_INVALID;
  if (n_ix > src->rank) return fail(ctx, HGPU_ERR_INVALID, "gather: %d indices into rank %d", n_ix, src->rank);
  int rank_n = src->rank - n_ix;
  if (rank_m + rank_n > HGPU_MAX_RANK) return fail(ctx, HGPU_ERR_INVALID, "gather: result rank too large");
  int64_t osh[HGPU_MAX_RANK];
  int64_t M = 1, N = 1;
  for (int i = 0; i < rank_m; ++i) { osh[i] = shm[i]; M *= shm[i]; }
  for (int i = 0; i < rank_n; ++i) { osh[rank_m + i] = src->shape[n_ix + i]; N *= src->shape[n_ix + i]; }
  IxSpace sp;
  int rc = build_space(ctx, "gather", n_ix, ix, rank_m, shm, nullptr, &sp);
  if (rc) return rc;
  bool empty_table = false;
  for (int k = 0; k < n_ix; ++k) {
    sp.extent[k] = src->shape[k];
    sp.table_st[k] = src->strides[k];
    if (src->shape[k] == 0) empty_table = true;
  }
  hgpu_array* o = nullptr;
  if (M * N == 0 || empty_table) {
    rc = new_zeros(ctx, src->dtype, rank_m + rank_n, osh, &o);
    if (rc) return rc;
    *out = o;
    return HGPU_OK;
  }
  rc = new_dense(ctx, src->dtype, rank_m + rank_n, osh, &o);
  if (rc) return rc;
  const int64_t* is[1] = {src->strides + n_ix};
  Dims inner;
  if (!collapse(rank_n, src->shape + n_ix, 1, is, &inner)) { hgpu_release(o); return fail(ctx, HGPU_ERR_UNSUPPORTED, "gather: too many inner dims"); }
  {
    const char* label = "gather";
    if (ctx->profiling && ctx->profile_shapes) {
      char buf[120];
      snprintf(buf, sizeof buf, "gather[es%d,M%lld,N%lld,ix%d]", (int)dtype_size(src->dtype), (long long)M, (long long)N, n_ix);
      label = intern_label(ctx, buf);
    }
    const double bytes = 2.0 * M * N * dtype_size(src->dtype) + 8.0 * M * n_ix;
    // contiguous slices of whole 16-byte (or 8-byte) units: one unit per lane
    const int64_t es = (int64_t)dtype_size(src->dtype);
    const bool contiguous = N == 1 || (inner.nd == 1 && inner.st[0][0] == 1), floats = dtype_is_float(src->dtype);
    int unit = 0;
    if (contiguous) {
      for (int cand : {16, 8, 4}) {
        // (the element as a unit: floats, whose gathers can wait to be multiplied and summed instead of written)
        if ((cand <= es && !(floats && cand == es)) || (N * es) % cand != 0 || ((uintptr_t)data_ptr(src)) % (uintptr_t)cand != 0) continue;
        bool ok = true;
        for (int k = 0; k < n_ix && ok; ++k) ok = (src->strides[k] * es) % cand == 0;
        if (ok) { unit = cand; break; }
      }
    }
    if (unit) {
      auto job = std::make_shared<GatherJob>();
      job->label = label;
      job->bytes = bytes;
      job->sp = sp;
      job->M = M;
      job->N = N;
      job->units = N * es / unit;
      job->epu = unit / es;
      job->unit = unit;
      job->dtype = src->dtype;
      job->src = data_ptr(src);
      job->out = data_ptr(o);
      std::vector<hgpu_buffer*> read{src->buf};
      for (int k = 0; k < n_ix; ++k) read.push_back(ix[k]->buf);
      if (floats && hold_job(ctx, job, read, {o->buf}, true)) { *out = o; return HGPU_OK; }
      LaunchGuard lg(ctx, label, bytes, 0);      // (integers, or a gather that reads held results)
      const hipError_t e = job->launch(ctx, lg.start_event(), lg.stop_event());
      if (e != hipSuccess) { hgpu_release(o); return check_hip(ctx, e, "gather"); }
      *out = o;
      return HGPU_OK;
    }
    LaunchGuard lg(ctx, label, bytes, 0);
    unsigned g = grid_for(M * N, kBlock, ctx->num_cu * 8);
    switch (dtype_size(src->dtype)) {
      case 8: hipLaunchKernelGGL(k_gather<uint64_t>, dim3(g), dim3(kBlock), 0, ctx->stream, sp, inner, M, N, (const uint64_t*)data_ptr(src), (uint64_t*)data_ptr(o)); break;
      case 4: hipLaunchKernelGGL(k_gather<uint32_t>, dim3(g), dim3(kBlock), 0, ctx->stream, sp, inner, M, N, (const uint32_t*)data_ptr(src), (uint32_t*)data_ptr(o)); break;
      case 2: hipLaunchKernelGGL(k_gather<uint16_t>, dim3(g), dim3(kBlock), 0, ctx->stream, sp, inner, M, N, (const uint16_t*)data_ptr(src), (uint16_t*)data_ptr(o)); break;
      default: hipLaunchKernelGGL(k_gather<uint8_t>, dim3(g), dim3(kBlock), 0, ctx->stream, sp, inner, M, N, (const uint8_t*)data_ptr(src), (uint8_t*)data_ptr(o)); break;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) { hgpu_release(o); return check_hip(ctx, e, "gather"); }
  }
  *out = o;
  return HGPU_OK;
}

int hgpu_scatter_add(hgpu_ctx* ctx, const hgpu_array* src, int n_ix, const hgpu_array* const* ix, int rank_m, const int64_t* shp, int flags, hgpu_array** out) {
  if (!ctx || !src || !out || rank_m < 0 || n_ix < 0) return HGPU_ERR_INVALID;
  if (rank_m > src->rank) return fail(ctx, HGPU_ERR_INVALID, "scatter: %d position dims in rank %d", rank_m, src->rank);
  int rank_n = src->rank - rank_m;
  if (n_ix + rank_n > HGPU_MAX_RANK) return fail(ctx, HGPU_ERR_INVALID, "scatter: result rank too large");
  if (src->dtype == HGPU_BOOL) return fail(ctx, HGPU_ERR_INVALID, "scatter: Bool arrays have no sum");
  int64_t osh[HGPU_MAX_RANK];
  int64_t M = 1, N = 1;
  for (int i = 0; i < n_ix; ++i) osh[i] = shp[i];
  for (int i = 0; i < rank_m; ++i) M *= src->shape[i];
  for (int i = 0; i < rank_n; ++i) { osh[n_ix + i] = src->shape[rank_m + i]; N *= src->shape[rank_m + i]; }
  int64_t C = 1;
  for (int i = 0; i < n_ix; ++i) C *= shp[i];
  // (more cells than eight to a position: passes over the cells would outweigh those over the positions)
  const bool counted = (flags & 1) == 0 && N > 0 && C > 0 && M > kCountedLeast && M <= kCountedPositions && M <= kCountedPerCell * C && C <= 8 * M + 4096;
  hgpu_array* o = nullptr;
  int rc = counted ? new_dense(ctx, src->dtype, n_ix + rank_n, osh, &o) : new_zeros(ctx, src->dtype, n_ix + rank_n, osh, &o);
  if (rc) return rc;
  if (M * N == 0 || nelem(o) == 0) { *out = o; return HGPU_OK; }
  IxSpace sp;
  rc = build_space(ctx, "scatter", n_ix, ix, rank_m, src->shape, src->strides, &sp);
  if (rc) { hgpu_release(o); return rc; }
  for (int k = 0; k < n_ix; ++k) {
    sp.extent[k] = shp[k];
    sp.table_st[k] = counted ? o->strides[k] / N : o->strides[k];
  }
  const int64_t* is[1] = {src->strides + rank_m};
  Dims inner;
  if (!collapse(rank_n, src->shape + rank_m, 1, is, &inner)) { hgpu_release(o); return fail(ctx, HGPU_ERR_UNSUPPORTED, "scatter: too many inner dims"); }
  bool inj = (flags & 1) != 0;
  if (inj) {
    LaunchGuard lg(ctx, "scatter_store", 2.0 * M * N * dtype_size(src->dtype) + 8.0 * M * n_ix, 0);
    unsigned g = grid_for(M * N, kBlock, ctx->num_cu * 8);
    HG_DISPATCH_DTYPE(src->dtype, T, hipLaunchKernelGGL((k_scatter_store<T>), dim3(g), dim3(kBlock), 0, ctx->stream, sp, inner, M, N, (const T*)data_ptr(src), (T*)data_ptr(o)));
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) { hgpu_release(o); return check_hip(ctx, e, "scatter"); }
    *out = o;
    return HGPU_OK;
  }
  // sort the positions by destination (stable: colliding positions stay in ascending order), then sum every run in that order
  if (M >= (int64_t)1 << 32) { hgpu_release(o); return fail(ctx, HGPU_ERR_UNSUPPORTED, "scatter: %lld positions", (long long)M); }
  hipError_t e;
  if (counted) {
    e = scatter_counted(ctx, sp, inner, M, N, C, src, o, &rc);
  } else {
    const Reads reads = scatter_reads(sp, src);
    LaunchGuard lg(ctx, "scatter_sorted", 2.0 * M * N * dtype_size(src->dtype) + 8.0 * M * n_ix, (double)M * N, &reads);
    // destinations that fit 32 bits sort as 32-bit keys: half the bytes per sorting pass
    e = nelem(o) < (int64_t)0xffffffff ? scatter_sorted<uint32_t>(ctx, sp, inner, M, N, src, o, &rc) : scatter_sorted<uint64_t>(ctx, sp, inner, M, N, src, o, &rc);
  }
  if (rc) { hgpu_release(o); return rc; }
  if (e != hipSuccess) { hgpu_release(o); return check_hip(ctx, e, "scatter"); }
  *out = o;
  return HGPU_OK;
}

}  // extern "C"
