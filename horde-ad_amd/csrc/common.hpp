// Shared host-side definitions of the gfx950 backend: context, buffer, array
// view, dimension collapsing and launch helpers.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <atomic>
#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <initializer_list>
#include <map>
#include <memory>
#include <mutex>
#include <set>
#include <string>
#include <thread>
#include <vector>

#include "hordead_gpu.h"

// Largest number of dimensions a kernel sees after adjacent dimensions that
// are contiguous in every operand have been merged.
#define HG_KDIMS 10

// Blocks handed out while a graph is being captured belong to the capture's
// pool: replays of the graph write them again, so they may be reused by the
// capture itself but never by other work while the graph lives.
struct hgpu_cap_pool {
  std::multimap<size_t, void*> cache;   // guarded by the context's allocator mutex
  bool alive = true;                    // false once the graph is destroyed: blocks return to the context's cache
  int refs = 1;                         // the graph (or the open capture) + every live buffer
};

struct hgpu_buffer {
  hgpu_ctx* ctx;
  void* ptr;
  size_t bytes;      // size of the block handed out by the allocator
  std::atomic<int> refs;
  hgpu_cap_pool* pool = nullptr;
  // What the library knows about the block's contents without reading them (arrays are written
  // once): element i is the I64 value i (hgpu_iota), or the block holds a single element of all
  // zero bits.  A kernel chosen because of that knowledge marks the block, and the two entry points
  // that write into existing arrays (hgpu_overwrite, hgpu_assign) refuse a marked block.
  enum { kUnknown = 0, kIotaI64 = 1, kZeroScalar = 2 };
  int known = kUnknown;
  bool known_relied_on = false;
  int held = 0;      // how often launches that are held back read or write it (guarded by the context's launch_mu)
  int level = 0;     // among the levels of what goes out at one time (launch_held_locked in smallk.hip; guarded likewise)
};

struct hgpu_array {
  hgpu_ctx* ctx;
  std::atomic<int> refs;
  hgpu_buffer* buf;  // nullptr for zero-size arrays
  int dtype;
  int rank;
  int64_t shape[HGPU_MAX_RANK];
  int64_t strides[HGPU_MAX_RANK];  // in elements
  int64_t offset;                  // in elements, from buf->ptr
  // Arrays (views included) come and go by the thousand in a training step, most of them freed together
  // when the step's tape goes: their blocks are kept on a list per thread instead of going back to the
  // allocator, whose per-thread cache holds only a few blocks of one size.
  static void* operator new(size_t n);
  static void operator delete(void* p);
};

namespace hg {
// The addresses of what a launch reads: a few of them, in place (every launch has such a list).
class Reads {
  const void* few_[20];
  std::vector<const void*> many_;
  size_t n_ = 0;
 public:
  Reads() {}
  Reads(std::initializer_list<const void*> l) { add(l.begin(), l.end()); }
  explicit Reads(const std::vector<const void*>& v) { add(v.begin(), v.end()); }
  void push_back(const void* p) {
    if (n_ < sizeof few_ / sizeof few_[0]) few_[n_] = p;
    else {
      if (many_.empty()) many_.assign(few_, few_ + n_);
      many_.push_back(p);
    }
    ++n_;
  }
  template <typename I> void add(I from, I to) { for (; from != to; ++from) push_back(*from); }
  const void* const* begin() const { return many_.empty() ? few_ : many_.data(); }
  const void* const* end() const { return begin() + n_; }
};
struct DeferredQueue;                         // launches held back to be grouped (smallk.hip)
void flush_deferred_locked(hgpu_ctx* ctx);    // the caller holds launch_mu
void flush_deferred(hgpu_ctx* ctx);
// Before a launch that reads the blocks of `reads` and writes new arrays only: launches what it needs of the held-back work (the caller holds launch_mu).
void make_way_locked(hgpu_ctx* ctx, const Reads& reads);
void drop_deferred(hgpu_ctx* ctx);            // flush, then free the queue
void forget_remembered_sums(hgpu_ctx* ctx);   // results kept for a later call, and the arrays held for them (footprint.hip)
}  // namespace hg

// A mutex that knows whether the calling thread has it: what is held back may have to go out for an allocation, which some
// callers make under it and most do not.
class LaunchMutex {
  std::mutex m_;
  std::atomic<std::thread::id> owner_{std::thread::id()};
 public:
  void lock() { m_.lock(); owner_.store(std::this_thread::get_id(), std::memory_order_relaxed); }
  void unlock() { owner_.store(std::thread::id(), std::memory_order_relaxed); m_.unlock(); }
  bool mine() const { return owner_.load(std::memory_order_relaxed) == std::this_thread::get_id(); }
};

struct hgpu_ctx {
  int device;
  hipStream_t stream;
  std::mutex mu;                 // guards allocator state and `err`
  std::multimap<size_t, void*> cache;
  uint64_t in_use = 0, reserved = 0, n_device_allocs = 0;
  int64_t fail_after = -1;
  std::string err;
  void* staging = nullptr;       // pinned host memory: kReadBytes read back, then the number of the last read-back (read_back_locked)
  uint64_t reads_back = 0;       // guarded by launch_mu, like the staging block
  LaunchMutex launch_mu;         // serialises enqueue order across host threads
  uint64_t write_epoch = 0;      // counts the writes into existing arrays (hgpu_overwrite, hgpu_assign): results remembered for given inputs end with it
  int num_cu = 256;
  // JIT cache of fused elementwise kernels, keyed by generated source.
  std::map<std::string, void*> jit_cache;
  // Optional per-launch timing (hgpu_profile_enable): one event pair per launch.
  struct ProfRec { const char* name; hipEvent_t a, b; double bytes, flops; };
  bool profiling = false;
  bool profile_shapes = false;           // hgpu_profile_enable(ctx, 2): labels carry the problem shape
  std::set<std::string> label_pool;
  std::mutex label_mu;                    // guards label_pool: labels are made on any calling thread
  std::vector<ProfRec> prof;
  // A launch that goes into a recording is counted by its label; nothing is timed there.
  void count_recorded(const char* name, double bytes, double flops) {
    if (profiling && cap && name) prof.push_back({name, nullptr, nullptr, bytes, flops});
  }
  hgpu_buffer* zero_block = nullptr;     // 256 zero bytes, for kernels that want a dummy table
  hgpu_buffer* ticket_block = nullptr;   // counters (zero between launches) for kernels whose last block finishes a reduction
  hgpu_cap_pool* cap = nullptr;          // non-null while the stream is capturing into a graph
  std::vector<const void*> recorded_functions;   // the run-time compiled kernels of the open recording (guarded by launch_mu)
  // Small products whose launch is held back until something else needs the
  // stream: those that do not depend on one another then go out as one kernel.
  hg::DeferredQueue* dq = nullptr;
  bool dq_pending = false;
  int deferred_rc = 0;                   // first error of a held-back launch, reported by the next call that hands results to the host
};

struct hgpu_graph {
  hgpu_ctx* ctx;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  hgpu_cap_pool* pool = nullptr;
  struct Kernel { hipKernelNodeParams params; bool module; };   // the arguments are the graph's; module: compiled at run time
  std::vector<Kernel> direct;                                   // a short recording's kernels (direct_kernels in runtime.hip)
};

namespace hg {

inline size_t dtype_size(int dt) {
  switch (dt) {
    case HGPU_F64: case HGPU_I64: return 8;
    case HGPU_F32: case HGPU_I32: return 4;
    case HGPU_I16: return 2;
    case HGPU_I8: case HGPU_BOOL: return 1;
  }
  return 0;
}
inline bool dtype_is_float(int dt) { return dt == HGPU_F64 || dt == HGPU_F32; }
inline bool dtype_is_int(int dt) { return dt >= HGPU_I64 && dt <= HGPU_I8; }

int fail(hgpu_ctx* ctx, int code, const char* fmt, ...);
int check_hip(hgpu_ctx* ctx, hipError_t e, const char* what);

// Allocator (runtime.hip).  A request that the device cannot serve sends out what is held back, whose memory then comes back.
int buffer_alloc(hgpu_ctx* ctx, size_t bytes, hgpu_buffer** out);
int zero_block(hgpu_ctx* ctx, const void** out);   // a context-lifetime block of 256 zero bytes
// Context-lifetime counters (1024 of 32 bits, zero between launches) for kernels whose blocks draw tickets: the
// last one finishes the reduction and sets its counter back to zero.  Launches on the context's stream follow one
// another, so the same counters serve them all.
int ticket_block(hgpu_ctx* ctx, void** out);
// At most this many bytes go to the host, or to the device, by a kernel instead of a copy of the runtime's (runtime.hip).
constexpr size_t kReadBytes = 4096, kStoreBytes = 256;
// The `bytes` bytes at the device address p, once everything enqueued before has written them (runtime.hip; the caller holds launch_mu).
hipError_t read_back_locked(hgpu_ctx* ctx, const void* p, size_t bytes, void* host);
// Fails (HGPU_ERR_UNSUPPORTED) when the stream is capturing: for entry points that must talk to the host.
int no_capture(hgpu_ctx* ctx, const char* what);
void buffer_retain(hgpu_buffer* b);
void buffer_release(hgpu_buffer* b);

// Array construction helpers (runtime.hip).
hgpu_array* new_view(hgpu_ctx* ctx, hgpu_buffer* buf, int dtype, int rank, const int64_t* shape,
                     const int64_t* strides, int64_t offset);
int new_dense(hgpu_ctx* ctx, int dtype, int rank, const int64_t* shape, hgpu_array** out);
int new_zeros(hgpu_ctx* ctx, int dtype, int rank, const int64_t* shape, hgpu_array** out);
inline int64_t nelem(const hgpu_array* a) {
  int64_t n = 1;
  for (int i = 0; i < a->rank; ++i) n *= a->shape[i];
  return n;
}
inline void* data_ptr(const hgpu_array* a) {
  if (!a->buf) return nullptr;
  return (char*)a->buf->ptr + a->offset * (int64_t)dtype_size(a->dtype);
}
bool is_dense(const hgpu_array* a);
bool same_shape(const hgpu_array* a, const hgpu_array* b);

// Up to four operands viewed over one iteration space.  `nd` dimensions of
// extent `shape`, operand k advancing by `st[k][d]` elements along dim d.
struct Dims {
  int nd;
  int64_t shape[HG_KDIMS];
  int64_t st[4][HG_KDIMS];
};

// The same with two operands, as a grouped reduction's arguments hold it.
struct Dims2 {
  int nd;
  int64_t shape[HG_KDIMS];
  int64_t st[2][HG_KDIMS];
};

// One single-launch reduction of hgpu_contract (contract.hip) with every argument of its kernel: such a launch
// can be held back like a small product, and reductions that do not read one another's results then go out as
// one kernel (the bias and readout gradients at the end of a reverse pass).
struct RedJob {
  int dtype = 0;              // element type of operands and result
  int variant = 0;            // 0: a block per output, 1: a wavefront per output, 2: a lane per output, kSumRows and up: sums of partial results
  int hasb = 0;
  Dims keep, red;
  int64_t n_out = 0, R = 0, Q = 0, Lin = 0, sa = 0, sb = 0, chunk = 0;
  unsigned grid = 0;
  const void* a = nullptr;
  const void* b = nullptr;
  void* out = nullptr;
  const char* label = nullptr;
  double bytes = 0, flops = 0;
  // Sums of partial results: out[i] = sum over R partials s of a[s * sa + i] (kSumRows: of the doubles a[i * R + s]); outputs from n1 on go to out2.
  int64_t n1 = 0;
  void* out2 = nullptr;
  bool is_sum() const { return variant >= kSumRows; }
  enum { kSumRows = 3, kSumLane, kSum32, kSum8, kSumPair, kSumTiny };      // kSumPair: a[i] + b[i]; kSumTiny: R instructions, coded in sa
};
constexpr int kMaxGroupReductions = 4, kMaxGroupSums = 12;
// One dense copy between two arrays that do not overlap (hgpu_assign): `bytes` bytes in units of 2^unit bytes, to which both sides are aligned.
struct CopyJob {
  const void* src;
  void* dst;
  int64_t bytes;
  int unit;
};
constexpr int kMaxCopyJobs = 48;
// ewise.hip: launches up to kMaxCopyJobs independent copies as one kernel (the caller holds launch_mu)
hipError_t launch_copy_group(hgpu_ctx* ctx, const CopyJob* const* jobs, int n);
// One elementwise pass over dense arrays (fused.hip): its kernel, the kernel that runs up to kMaxMapJobs of them, and the
// arguments (element count, inputs, outputs) of 8 bytes each.
constexpr int kMaxMapJobs = 16;
struct MapJob {
  hipFunction_t fn, group;
  unsigned grid;
  std::vector<uint64_t> args;
  const char* label;
  double bytes, flops;
  int n_in = 0;
  std::vector<char> dense;           // per input: an array, not one element
  std::vector<uint64_t> depends;     // per output: inputs that must have been loaded for it to be stored, a bit for each
  std::vector<int> out_size;         // bytes of an output's element
  // Copies of whole results into existing arrays that came while the pass waited (hold_copy): where nobody else has the result by the time
  // the pass goes out, it is written to the copy's destination instead.
  struct Copy { int out; CopyJob job; hgpu_buffer *src, *dst; };
  std::vector<Copy> copies;
};
// smallk.hip: holds an elementwise pass back (retaining the buffers) to be launched with those of the same kernel that follow it; the caller holds launch_mu
void hold_map_locked(hgpu_ctx* ctx, MapJob&& job, const std::vector<hgpu_buffer*>& reads, const std::vector<hgpu_buffer*>& writes);
// smallk.hip: holds a copy back (retaining both buffers) to be launched with the copies that follow it
void hold_copy(hgpu_ctx* ctx, const CopyJob& job, hgpu_buffer* src, hgpu_buffer* dst);
// contract.hip: launches up to kMaxGroupReductions such reductions and kMaxGroupSums sums of partial results, all of one element type, as one kernel (the caller holds launch_mu)
hipError_t launch_reduction_group(hgpu_ctx* ctx, const RedJob* const* jobs, int n);
// One product that a recording may hold back (gemm.hip): its kernel, its arguments, and how such products are launched together.
struct WideJob;
// gemm.hip: launches up to kMaxWideJobs products of one kernel (the caller holds launch_mu)
hipError_t launch_wide_group(hgpu_ctx* ctx, const WideJob* const* jobs, int n);
bool longer_wide_shares(hgpu_ctx* ctx, const WideJob* const* jobs, int n, int* shares);
void set_wide_shares(WideJob& job, int shares);      // of a term's K
int wide_shares(const WideJob& job);                 // of all terms: as many partial results
const void* wide_partials(const WideJob& job);
const void* wide_row_partials(const WideJob& job);   // null: none
constexpr int kMaxWideJobs = 4;
// gemm.hip: row sums that a held product hands out beside its result (see join_wide_rows)
int wide_row_shares(const WideJob& job, int dtype, int n, const void* const* as, int64_t M, int64_t K, int64_t row_stride);
void wide_take_rows(WideJob& job, void* part, const void* factor);
bool wide_takes_rows(const WideJob& job);
// smallk.hip: the sums over K of n terms of M rows of floats of `dtype`, each term times the one element `factor` (null: 1), as
// *part (rows x *shares, doubles) by a held product that reads the same rows; false: there is none
bool join_wide_rows(hgpu_ctx* ctx, int dtype, int n, const void* const* as, int64_t M, int64_t K, int64_t row_stride, hgpu_buffer* factor_buf, const void* factor, hgpu_buffer** part, int* shares);
// One launch that is held back by itself (a gather of whole slices, index.hip; a small objective's reductions, fused.hip).
struct HeldJob {
  const char* label = nullptr;
  double bytes = 0, flops = 0;
  virtual ~HeldJob() {}
  virtual hipError_t launch(hgpu_ctx* ctx, hipEvent_t start, hipEvent_t stop) = 0;       // the caller holds launch_mu; events: null, or carried by the launch
};
// smallk.hip: holds the launch back (retaining the buffers) until something reads its results or writes to an array that exists;
// it never runs if nobody has any of the results any more by then.  What it reads of held results goes out first, or, with
// ready_only, it is not held (false: the caller launches it now).
bool hold_job(hgpu_ctx* ctx, const std::shared_ptr<HeldJob>& job, const std::vector<hgpu_buffer*>& reads, const std::vector<hgpu_buffer*>& writes, bool ready_only);
// smallk.hip, the caller holds launch_mu: the held launch that will write this block, if there is one; a held launch reads and writes more
std::shared_ptr<HeldJob> held_writer_locked(hgpu_ctx* ctx, const hgpu_buffer* b);
bool extend_job_locked(hgpu_ctx* ctx, const std::shared_ptr<HeldJob>& job, const std::vector<hgpu_buffer*>& reads, const std::vector<hgpu_buffer*>& writes);
// ... goes out now
void end_job_locked(hgpu_ctx* ctx, const std::shared_ptr<HeldJob>& job);
// A zero-extension (ewise.hip) that waits until something reads its result: a kernel that copies its operand to LDS reads the
// array that is extended instead (footprint.hip).  Dims as they lie in the dense result, from dst on.
struct PadJob : HeldJob {
  int dtype, nd;
  int64_t shape[HG_KDIMS], lo[HG_KDIMS], ext[HG_KDIMS], sst[HG_KDIMS];      // of the result; zeros in front; of the source, and its strides
  int64_t n;                   // elements of the result
  hgpu_buffer* src_buf;        // (kept by the queue as long as the job waits)
  const void* src;
  void* dst;
  hipError_t launch(hgpu_ctx* ctx, hipEvent_t start, hipEvent_t stop) override;
};
// fused.hip: holds the extremum of one dense row back, to be one launch with the sums over the same elements that follow; false: left to the caller
bool try_hold_extremum(hgpu_ctx* ctx, const hgpu_array* a, int want_max, const hgpu_array* index, const hgpu_array* value);
// contract.hip: the extremum of one row by a block (the caller holds launch_mu)
hipError_t launch_extremum_row(hgpu_ctx* ctx, int dtype, int64_t n, int want_max, const void* a, void* index, void* value);
// index.hip: *o (one element) = sum of a * b, where a held gather is to write a or b and need not for this; *handled: taken
int try_gather_dot(hgpu_ctx* ctx, const hgpu_array* a, const hgpu_array* b, const hgpu_array* o, bool* handled);
// smallk.hip: holds the product back (retaining the buffers) to be launched with those of the same kernel that do not depend on it
void hold_wide(hgpu_ctx* ctx, std::shared_ptr<WideJob> job, int kernel, const char* label, double bytes, double flops, const std::vector<hgpu_buffer*>& reads, hgpu_buffer* write);
// contract.hip: a program over a few elements (its last instruction's result is `out`), in a recording launched with held sums; false: left to the caller
bool try_tiny_map(hgpu_ctx* ctx, int n_in, const hgpu_array* const* in, int n_instr, const hgpu_fused_instr* prog, const hgpu_array* out);
// contract.hip: *acc += x, taking over x (the first term becomes the accumulator); the addition is held back where it can share a launch
int add_into(hgpu_ctx* ctx, hgpu_array** acc, hgpu_array* x);
// smallk.hip: holds the launch back (retaining the buffers it reads and writes); false: the caller launches it now
bool hold_reduction(hgpu_ctx* ctx, const RedJob& job, hgpu_buffer* const* reads, int n_reads, hgpu_buffer* write, hgpu_buffer* write2 = nullptr);
// contract.hip: the `parts` partial results of n elements in `part` are added up in `out` (dense), or the first n1 in out1 and the other n - n1 in out2.
// Held back where it can share a launch; launched alone it counts under `label`, where that is given, as a part of the product that left the partials.
int sum_partials(hgpu_ctx* ctx, int dtype, int64_t n, int parts, hgpu_buffer* part, const hgpu_array* out1, int64_t n1 = -1, const hgpu_array* out2 = nullptr, const char* label = nullptr);

// Builds the merged iteration space of `nops` operands that share `shape`.
// Size-1 dims vanish; adjacent dims merge when every operand's strides allow.
// Returns false when more than HG_KDIMS dims remain.
bool collapse(int rank, const int64_t* shape, int nops, const int64_t* const* strides, Dims* out);

inline void dense_strides(int rank, const int64_t* shape, int64_t* st) {
  int64_t s = 1;
  for (int i = rank - 1; i >= 0; --i) { st[i] = s; s *= shape[i]; }
}

inline unsigned grid_for(int64_t n, int block, int max_blocks) {
  int64_t g = (n + block - 1) / block;
  if (g < 1) g = 1;
  if (g > max_blocks) g = max_blocks;
  return (unsigned)g;
}

// Compiles `src` for gfx950 at run time (runtime.hip) and hands back the code
// object.  Code objects are kept on disk between processes, keyed by the
// source, the options and the compiler's version: a kernel that was compiled
// once (a second or so for the larger ones) is read back in under a
// millisecond.  The directory is $HORDEAD_GPU_CACHE, else
// $XDG_CACHE_HOME/hordead_gpu, else $HOME/.cache/hordead_gpu; HORDEAD_GPU_CACHE=off
// (or an unwritable directory) means no files.  `what` names the caller in errors.
int rtc_compile(hgpu_ctx* ctx, const std::string& src, const char* what, std::vector<char>* code);

// Zeroes `bytes` bytes (rounded up to 16) with a fill kernel (ewise.hip); fresh: of a block that nothing has been enqueued for.
int zero_fill(hgpu_ctx* ctx, void* p, size_t bytes, bool fresh = false);
// Strided copy between two views of equal shape (ewise.hip).
int copy_view(hgpu_ctx* ctx, int dtype, int rank, const int64_t* shape, const void* src,
              const int64_t* sst, void* dst, const int64_t* dst_st);

// Serialises enqueueing and, when profiling is on, brackets the launches made
// while it lives with an event pair labelled `name`; `bytes` / `flops` are the
// ALGORITHMIC traffic and work of those launches.
//
// `reads`: the launches write new arrays only, and these addresses lie in every block they read.  Held-back work whose
// results they do not read then stays held back (arrays are written once, and held work keeps its blocks, so
// reads-after-writes are the only order there is); without it everything held back goes first.
struct LaunchGuard {
  hgpu_ctx* ctx;
  bool timed = false;
  explicit LaunchGuard(hgpu_ctx* c, const char* name = nullptr, double bytes = 0, double flops = 0, const Reads* reads = nullptr) : ctx(c) {
    c->launch_mu.lock();
    (void)hipSetDevice(c->device);
    if (c->dq_pending && reads) make_way_locked(c, *reads);
    else if (c->dq_pending) flush_deferred_locked(c);   // stream order is program order
    static const bool trace = getenv("HORDEAD_GPU_TRACE_LAUNCHES") != nullptr;   // one line per launch, in program order
    if (trace && name) fprintf(stderr, "hordead_gpu: launch %s\n", name);
    c->count_recorded(name, bytes, flops);
    if (c->profiling && name && !c->cap) {
      hgpu_ctx::ProfRec r{name, nullptr, nullptr, bytes, flops};
      if (hipEventCreate(&r.a) == hipSuccess && hipEventCreate(&r.b) == hipSuccess) {
        (void)hipEventRecord(r.a, c->stream);
        c->prof.push_back(r);
        timed = true;
      }
    }
  }
  ~LaunchGuard() {
    if (timed && !stop_carried) (void)hipEventRecord(ctx->prof.back().b, ctx->stream);
    ctx->launch_mu.unlock();
  }
  // The guard's events for a launch that carries them itself (hipExtModuleLaunchKernel, hipExtLaunchKernel): they
  // then hold the kernel's own begin and end, which is what a profiler's kernel trace reports.  Events recorded
  // around a launch also time its dispatch and the cache write-back after it, 3-4 us more on this device.  The
  // first launch under the guard takes start_event(), the last one stop_event(); both are null while nothing is timed.
  bool stop_carried = false;
  hipEvent_t start_event() { return timed ? ctx->prof.back().a : nullptr; }
  hipEvent_t stop_event() {
    if (!timed) return nullptr;
    stop_carried = true;
    return ctx->prof.back().b;
  }
};

// What launches over these arrays read (see LaunchGuard).
inline Reads reads_of(int n, const hgpu_array* const* in) {
  Reads r;
  for (int i = 0; i < n; ++i) r.push_back(data_ptr(in[i]));
  return r;
}

// A recording's launches of run-time compiled kernels, which its graph names by their handles (the caller holds launch_mu).
inline void note_recorded(hgpu_ctx* c, hipFunction_t fn) {
  if (c->cap) c->recorded_functions.push_back((const void*)fn);
}

// Launch of a run-time compiled kernel under a guard: `first` / `last` say whether this is the first / last
// launch the guard's record is to cover.
inline hipError_t launch_module(LaunchGuard& lg, hipFunction_t fn, unsigned grid, unsigned block, void** args, bool first = true, bool last = true) {
  note_recorded(lg.ctx, fn);
  if (!lg.timed || (uint64_t)grid * block > 0xffffffffull) return hipModuleLaunchKernel(fn, grid, 1, 1, block, 1, 1, 0, lg.ctx->stream, args, nullptr);
  return hipExtModuleLaunchKernel(fn, grid * block, 1, 1, block, 1, 1, 0, lg.ctx->stream, args, nullptr, first ? lg.start_event() : nullptr,
                                  last ? lg.stop_event() : nullptr, 0);
}

// A label with the lifetime of the context (profiling records keep the pointer).
inline const char* intern_label(hgpu_ctx* c, const std::string& s) {
  std::lock_guard<std::mutex> g(c->label_mu);
  return c->label_pool.insert(s).first->c_str();
}

// The first error of a launch that had been held back and failed after its own
// call returned; cleared once handed out.  Every entry point that hands data or
// a finished recording to the host reports it, since the caller would otherwise
// read a result that was never written.  Call with launch_mu held.
inline int take_deferred_rc(hgpu_ctx* c) {
  const int rc = c->deferred_rc;
  c->deferred_rc = 0;
  return rc;
}

}  // namespace hg

#define HG_DISPATCH_DTYPE(dt, T, ...)                                   \
  switch (dt) {                                                         \
    case HGPU_F64: { using T = double; __VA_ARGS__; break; }            \
    case HGPU_F32: { using T = float; __VA_ARGS__; break; }             \
    case HGPU_I64: { using T = int64_t; __VA_ARGS__; break; }           \
    case HGPU_I32: { using T = int32_t; __VA_ARGS__; break; }           \
    case HGPU_I16: { using T = int16_t; __VA_ARGS__; break; }           \
    case HGPU_I8: { using T = int8_t; __VA_ARGS__; break; }             \
    case HGPU_BOOL: { using T = uint8_t; __VA_ARGS__; break; }          \
    default: break;                                                     \
  }

#define HG_CHECK_LAUNCH(ctx, what)                                      \
  do {                                                                  \
    hipError_t e__ = hipGetLastError();                                 \
    if (e__ != hipSuccess) return hg::check_hip(ctx, e__, what);        \
  } while (0)

// Device-side decomposition of a linear index over a merged iteration space.
#ifdef __HIPCC__
namespace hg {
template <int NOPS, typename D>
__device__ __forceinline__ void decompose(const D& d, int64_t lin, int64_t* off) {
#pragma unroll
  for (int k = 0; k < NOPS; ++k) off[k] = 0;
  if (lin < (int64_t)0x7fffffff) {
    uint32_t r = (uint32_t)lin;
    for (int i = d.nd - 1; i > 0; --i) {
      uint32_t s = (uint32_t)d.shape[i];
      uint32_t q = r / s;
      uint32_t c = r - q * s;
      r = q;
#pragma unroll
      for (int k = 0; k < NOPS; ++k) off[k] += (int64_t)c * d.st[k][i];
    }
#pragma unroll
    for (int k = 0; k < NOPS; ++k) off[k] += (int64_t)r * d.st[k][0];
  } else {
    int64_t r = lin;
    for (int i = d.nd - 1; i > 0; --i) {
      int64_t s = d.shape[i];
      int64_t q = r / s;
      int64_t c = r - q * s;
      r = q;
#pragma unroll
      for (int k = 0; k < NOPS; ++k) off[k] += c * d.st[k][i];
    }
#pragma unroll
    for (int k = 0; k < NOPS; ++k) off[k] += r * d.st[k][0];
  }
}
}  // namespace hg
#endif
