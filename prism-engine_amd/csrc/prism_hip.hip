// prism_hip.hip -- C ABI of the MI355X palettized-LUT contraction
// (declarations and contract: include/prism_hip.h).
//
// Host side: argument validation, device staging for host-pointer calls,
// kernel selection per shape, and the keyed HipBackend that mirrors the
// reference's MetalBackend (src/lut/engine_impl.rs:31-490).  There is no
// CPU fallback: every failure is returned as a negative code with text.
#include "prism_hip.h"

#include <cxxabi.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <vector>
#include <unordered_map>
#include <unordered_set>

#include "gemm_kernels.hpp"
#include "gemm_lookup.hpp"
#include "gemv_kernels.hpp"
#include "gemv_tile.hpp"
#include "gemv_lpr.hpp"
#include "gemv_mfma.hpp"
#include "host_io_kernels.hpp"
#include "measure_kernels.hpp"
#include "palette_kernels.hpp"
#include "step_kernels.hpp"

#define PRISM_HIP_VERSION "prism_hip 0.1 gfx950"

// Device memory of weights: one hipMalloc per chunk instead of one per
// tensor.  A context carves its uploads, 256-byte aligned and in upload
// order, out of its current chunk (8 MB first, doubling up to 64 MB);
// tensors over 16 MB get a chunk of their own.  A chunk is freed when the
// last weight in it is freed and no context carves from it any more, so
// weights outlive their context as before and a freed weight's bytes are
// reused only with its whole chunk.  MI355X: the 168 per-layer hipMallocs of
// a Qwen2.5-0.5B model take 2.3-5.4 ms and their hipFrees 17-20 ms.
struct WeightChunk {
  uint8_t* base = nullptr;
  size_t size = 0, used = 0;
  int device = 0;
  std::atomic<int> refs{0};  // weights in the chunk, plus one while a context carves from it
};

struct prism_hip_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  int num_cu = 256;
  size_t lds_max = 65536;  // dynamic + static LDS bytes one workgroup may use
  void* d_stage = nullptr;
  size_t stage_bytes = 0;
  // Pinned memory of the small host-pointer calls: operands in, results out,
  // and the sequence number of the last call (host_io_kernels.hpp).
  uint8_t* h_io = nullptr;
  uint8_t* h_io_dev = nullptr;  // its device address
  uint64_t io_seq = 0;
  // Stream-ordered pool for per-call device scratch of GEMMs on the caller's
  // streams, created on first use; it keeps what it has allocated, so a call after
  // the first reuses memory instead of allocating.
  hipMemPool_t pool = nullptr;
  // GEMM scratch (packed X, split-K partials) of the calls on the context's
  // own stream, which use it in stream order.
  void* d_gemm = nullptr;
  size_t gemm_bytes = 0;
  // This device's address of the static split-K scratch (looked up on the
  // first prism_hip_gemm_dev_noalloc).
  float* scratch = nullptr;
  // Host uploads: a ring of pinned staging buffers (created on first use),
  // each with the event of the last copy out of it, and a device buffer for
  // split-block payloads on their way to the GI layout.
  static constexpr int kRingSlots = 4;
  static constexpr size_t kRingSlotBytes = (size_t)16 << 20;
  void* ring[kRingSlots] = {};
  hipEvent_t ring_done[kRingSlots] = {};
  int ring_next = 0;
  void* d_upload = nullptr;
  size_t upload_bytes = 0;
  // The chunk uploads are carved from (holds one reference) and the size of
  // the next one.
  WeightChunk* carve = nullptr;
  size_t next_chunk = (size_t)8 << 20;
  std::string err;
  // Weights uploaded through this context; destroying the context orphans
  // them (w->ctx = nullptr) so a later prism_hip_weight_free stays valid.
  std::unordered_set<prism_hip_weight*> weights;
  // Decode-step models created on this context, orphaned the same way.
  std::unordered_set<prism_hip_model*> models;
  // Host functions of the kernels the last compute call launched, in
  // order, and their names once asked for (prism_hip_last_kernels).
  std::vector<const void*> launched;
  std::string kernels;
};

namespace prism {

// The launch log of the compute call running on this thread (NULL outside
// one): every dispatch site appends the kernel it launches.
thread_local std::vector<const void*>* g_launch_log = nullptr;

void note_launch(const void* fn) {
  if (g_launch_log) g_launch_log->push_back(fn);
}

}  // namespace prism

// hipLaunchKernelGGL that records the kernel (KERNEL as for
// hipLaunchKernelGGL: a template-id in parentheses).
#define PRISM_LAUNCH(KERNEL, ...)                                 \
  do {                                                            \
    prism::note_launch(reinterpret_cast<const void*>(&KERNEL));   \
    hipLaunchKernelGGL(KERNEL, __VA_ARGS__);                      \
  } while (0)

// hipLaunchKernel that records the kernel.
static hipError_t launch_fn(const void* fn, dim3 grid, dim3 block, void** args, size_t lds, hipStream_t st) {
  prism::note_launch(fn);
  return hipLaunchKernel(fn, grid, block, args, lds, st);
}

// For the length of one compute call: clears the context's launch log and
// makes it the thread's.
struct LaunchLog {
  std::vector<const void*>* prev;
  explicit LaunchLog(prism_hip_ctx* ctx) : prev(prism::g_launch_log) {
    ctx->launched.clear();
    ctx->kernels.clear();
    prism::g_launch_log = &ctx->launched;
  }
  ~LaunchLog() { prism::g_launch_log = prev; }
};

// Defined with prism_hip_model (model_step.hpp): forget the context.
static void model_detach(prism_hip_model* m);

// A weight's device copy is either the split-block payload as uploaded or,
// for 4-bit matrices the lane-per-row GEMV covers in one round of row groups,
// the GI layout (gemv_lpr.hpp: the same bytes regrouped per group of gi
// rows, each group's LUTs before its index chunks).  Kernels over GI take
// the base pointer as both their LUT and their index pointer.
struct prism_hip_weight {
  prism_hip_ctx* ctx = nullptr;
  int device = 0;
  uint32_t dim_m = 0, dim_n = 0, bits = 0, layout = 0;
  size_t bytes = 0;  // payload bytes as uploaded (split-block)
  uint32_t gi = 0;  // GI layout: rows per group; 0: split-block
  uint8_t* d = nullptr;
  WeightChunk* chunk = nullptr;  // the device memory d lies in
  const uint8_t* lut() const { return d; }
  const uint8_t* idx() const { return gi ? d : d + (size_t)dim_m * (2u << bits); }
};

// Packed X and split-K partials of prism_hip_gemm_dev_noalloc, the GEMM entry
// point that allocates nothing: one array on each GPU, held until the
// process ends.  The GEMM plan keeps every launch within it (plan_gemm).  In host code `scratch` is a
// host-side stand-in, never a device address: device_scratch() looks up each
// device's copy once, with that device current, and only that address is
// passed to kernels.
constexpr size_t kGemmScratchBytes = (size_t)64 << 20;
static __device__ __align__(256) float scratch[kGemmScratchBytes / sizeof(float)];

namespace {

thread_local std::string g_create_err;

// This device's address of `scratch` (the device is current), looked up
// once per device on the first no-alloc call that needs it.
hipError_t device_scratch(int device, float** out) {
  static std::mutex mu;
  static float* addr[64] = {};
  if (device < 0 || device >= 64) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[device]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    addr[device] = static_cast<float*>(p);
  }
  *out = addr[device];
  return hipSuccess;
}

int fail(prism_hip_ctx* ctx, int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  if (ctx) ctx->err = buf;
  return code;
}

#define HIP_TRY(ctx, expr)                                                                          \
  do {                                                                                              \
    hipError_t e_ = (expr);                                                                         \
    if (e_ != hipSuccess)                                                                           \
      return fail((ctx), PRISM_HIP_ERR_DEVICE, "%s failed: %s", #expr, hipGetErrorString(e_));     \
  } while (0)

size_t expected_bytes(uint32_t dm, uint32_t dn, uint32_t bits) {
  const size_t lut = (size_t)dm * (2u << bits);
  const size_t idx = (bits == 4) ? (size_t)dm * (dn / 2) : (size_t)dm * dn;
  return lut + idx;
}

int check_shape(prism_hip_ctx* ctx, uint32_t dm, uint32_t dn, uint32_t bits, uint32_t layout, size_t bytes) {
  if (bits != 4 && bits != 8) return fail(ctx, PRISM_HIP_ERR_BITS, "bits must be 4 or 8, got %u", bits);
  if (layout != PRISM_HIP_LAYOUT_SPLIT_BLOCK) return fail(ctx, PRISM_HIP_ERR_LAYOUT, "unknown layout %u", layout);
  if (dm == 0 || dn == 0) return fail(ctx, PRISM_HIP_ERR_SHAPE, "empty shape %ux%u", dm, dn);
  const size_t want = expected_bytes(dm, dn, bits);
  if (bytes != want)
    return fail(ctx, PRISM_HIP_ERR_SIZE, "payload is %zu bytes, %u-bit %ux%u needs %zu", bytes, bits, dm, dn, want);
  return PRISM_HIP_OK;
}

int ensure_stage(prism_hip_ctx* ctx, size_t bytes) {
  if (bytes <= ctx->stage_bytes) return PRISM_HIP_OK;
  if (ctx->d_stage) {
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    HIP_TRY(ctx, hipFree(ctx->d_stage));
    ctx->d_stage = nullptr;
    ctx->stage_bytes = 0;
  }
  size_t sz = 1 << 20;
  while (sz < bytes) sz <<= 1;
  HIP_TRY(ctx, hipMalloc(&ctx->d_stage, sz));
  ctx->stage_bytes = sz;
  return PRISM_HIP_OK;
}

// The context's pinned memory (0.4 ms, so at creation and not in the first
// call); without any left the runtime's copies serve instead.
void alloc_host_io(prism_hip_ctx* ctx) {
  const size_t bytes = 2 * prism::kHostIoBytes + prism::kHostIoBlocks * sizeof(uint64_t);
  void *h = nullptr, *d = nullptr;
  hipError_t e = hipHostMalloc(&h, bytes, hipHostMallocMapped | hipHostMallocCoherent);
  if (e == hipSuccess && (e = hipHostGetDevicePointer(&d, h, 0)) != hipSuccess) (void)hipHostFree(h);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return;
  }
  std::memset(h, 0, bytes);
  ctx->h_io = static_cast<uint8_t*>(h);
  ctx->h_io_dev = static_cast<uint8_t*>(d);
}

// The operands of one host-pointer call: `in` bytes of x on the device at
// d_in(), results written there at d_out(), and after the compute kernels
// finish() brings them to the host and waits.  Up to kHostIoBytes each way
// go through the context's pinned memory (host_io_kernels.hpp), more by the
// runtime's copies.
class HostCall {
 public:
  HostCall(prism_hip_ctx* ctx, size_t in, size_t out) : ctx_(ctx), in_(in), out_(out) {}
  int begin(const void* x) {
    off_ = (in_ + 255) & ~(size_t)255;
    const int rc = ensure_stage(ctx_, off_ + ((out_ + 255) & ~(size_t)255));
    if (rc) return rc;
    small_ = ctx_->h_io && in_ <= prism::kHostIoBytes && out_ <= prism::kHostIoBytes;
    if (!in_) return PRISM_HIP_OK;
    if (!small_) {
      HIP_TRY(ctx_, hipMemcpyAsync(ctx_->d_stage, x, in_, hipMemcpyHostToDevice, ctx_->stream));
      return PRISM_HIP_OK;
    }
    std::memcpy(ctx_->h_io, x, in_);
    hipLaunchKernelGGL(prism::k_host_in, dim3(prism::host_io_blocks(in_)), dim3(prism::kHostIoThreads), 0, ctx_->stream,
                       reinterpret_cast<const uint4*>(ctx_->h_io_dev), reinterpret_cast<uint4*>(ctx_->d_stage),
                       (uint32_t)((in_ + 15) / 16));
    HIP_TRY(ctx_, hipGetLastError());
    return PRISM_HIP_OK;
  }
  uint8_t* d_in() const { return static_cast<uint8_t*>(ctx_->d_stage); }
  uint8_t* d_out() const { return static_cast<uint8_t*>(ctx_->d_stage) + off_; }
  // Results, back to back from d_out() on, into y (the first y_bytes) and y2.
  int finish(void* y, size_t y_bytes, void* y2 = nullptr, size_t y2_off = 0) {
    if (!small_) {
      HIP_TRY(ctx_, hipMemcpyAsync(y, d_out(), y_bytes, hipMemcpyDeviceToHost, ctx_->stream));
      if (y2) HIP_TRY(ctx_, hipMemcpyAsync(y2, d_out() + y2_off, out_ - y2_off, hipMemcpyDeviceToHost, ctx_->stream));
      HIP_TRY(ctx_, hipStreamSynchronize(ctx_->stream));
      return PRISM_HIP_OK;
    }
    constexpr size_t kOut = prism::kHostIoBytes, kFlag = 2 * kOut;
    const uint64_t seq = ++ctx_->io_seq;
    const uint32_t blocks = prism::host_io_blocks(out_);
    hipLaunchKernelGGL(prism::k_host_out, dim3(blocks), dim3(prism::kHostIoThreads), 0, ctx_->stream,
                       reinterpret_cast<const uint4*>(d_out()), reinterpret_cast<uint4*>(ctx_->h_io_dev + kOut),
                       (uint32_t)((out_ + 15) / 16), reinterpret_cast<uint64_t*>(ctx_->h_io_dev + kFlag), seq);
    HIP_TRY(ctx_, hipGetLastError());
    // Poll for a while; then (a long kernel, or one that failed) wait for the
    // stream, which also reports errors.
    const uint64_t* flags = reinterpret_cast<const uint64_t*>(ctx_->h_io + kFlag);
    uint32_t ready = 0;  // workgroups that have finished
    for (int spin = 0; spin < 20000 && ready < blocks; spin++) {
      while (ready < blocks && __atomic_load_n(flags + ready, __ATOMIC_ACQUIRE) == seq) ready++;
#if defined(__x86_64__)
      if (ready < blocks) __builtin_ia32_pause();
#endif
    }
    if (ready < blocks) HIP_TRY(ctx_, hipStreamSynchronize(ctx_->stream));
    std::memcpy(y, ctx_->h_io + kOut, y_bytes);
    if (y2) std::memcpy(y2, ctx_->h_io + kOut + y2_off, out_ - y2_off);
    return PRISM_HIP_OK;
  }

 private:
  prism_hip_ctx* ctx_;
  size_t in_, out_, off_ = 0;
  bool small_ = false;
};

int ensure_upload_stage(prism_hip_ctx* ctx, size_t bytes) {
  if (bytes <= ctx->upload_bytes) return PRISM_HIP_OK;
  if (ctx->d_upload) {
    HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
    HIP_TRY(ctx, hipFree(ctx->d_upload));
    ctx->d_upload = nullptr;
    ctx->upload_bytes = 0;
  }
  size_t sz = 1 << 20;
  while (sz < bytes) sz <<= 1;
  HIP_TRY(ctx, hipMalloc(&ctx->d_upload, sz));
  ctx->upload_bytes = sz;
  return PRISM_HIP_OK;
}

// Host memcpy workers for the staging ring: copies of 512 KB and more are
// split into 256 KB parts that a few threads living for the whole process
// take in turn with the caller (one thread copies about 10-15 GB/s out of
// the page cache, the PCIe link takes several times that, and spawning
// threads per copy cost more than copying a 2 MB tensor).  One copy at a
// time; callers on several threads queue on `call_mu`.  The pool is never
// destroyed: its threads only ever run memcpy and end with the process.
class CopyPool {
 public:
  static CopyPool& get() {
    static CopyPool* p = new CopyPool();
    return *p;
  }
  void copy(void* dst, const void* src, size_t n) {
    constexpr size_t kPart = (size_t)256 << 10;
    if (n < 2 * kPart || workers_ == 0) {
      std::memcpy(dst, src, n);
      return;
    }
    std::lock_guard<std::mutex> call(call_mu_);
    {
      std::lock_guard<std::mutex> g(mu_);
      dst_ = static_cast<char*>(dst);
      src_ = static_cast<const char*>(src);
      n_ = n;
      finished_ = 0;
      total_ = (n + kPart - 1) / kPart;
      nparts_.store(total_);
      next_.store(0);
      gen_++;
    }
    cv_.notify_all();
    const size_t mine = work(kPart);
    std::unique_lock<std::mutex> g(mu_);
    finished_ += mine;
    // every part copied and every worker that took this job out of work()
    // (one still in it could otherwise claim a part of the next job)
    done_cv_.wait(g, [&] { return finished_ == total_ && active_ == 0; });
    nparts_.store(0);  // workers that wake late find no parts
  }

 private:
  CopyPool() {
    const unsigned hw = std::thread::hardware_concurrency();
    workers_ = std::min(7u, hw > 2 ? hw / 2 - 1 : 0u);
    for (unsigned i = 0; i < workers_; i++) std::thread([this] { loop(); }).detach();
  }
  // parts taken by this thread; the caller holds no lock
  size_t work(size_t part) {
    size_t done = 0;
    for (size_t i; (i = next_.fetch_add(1)) < nparts_.load();) {
      const size_t o = i * part, len = std::min(part, n_ - o);
      std::memcpy(dst_ + o, src_ + o, len);
      done++;
    }
    return done;
  }
  void loop() {
    uint64_t seen = 0;
    for (;;) {
      size_t part_bytes;
      {
        std::unique_lock<std::mutex> g(mu_);
        cv_.wait(g, [&] { return gen_ != seen; });
        seen = gen_;
        if (nparts_.load() == 0) continue;
        part_bytes = (size_t)256 << 10;
        active_++;
      }
      const size_t mine = work(part_bytes);
      std::lock_guard<std::mutex> g(mu_);
      finished_ += mine;
      active_--;
      if (finished_ == total_ && active_ == 0) done_cv_.notify_one();
    }
  }
  unsigned workers_ = 0;
  std::mutex call_mu_, mu_;
  std::condition_variable cv_, done_cv_;
  char* dst_ = nullptr;
  const char* src_ = nullptr;
  size_t n_ = 0, total_ = 0, finished_ = 0;
  unsigned active_ = 0;  // workers inside work() for the current job
  std::atomic<size_t> nparts_{0}, next_{0};
  uint64_t gen_ = 0;
};

void host_copy(void* dst, const void* src, size_t n) { CopyPool::get().copy(dst, src, n); }

// Host -> device copy of `bytes` through the pinned ring, in pieces of one
// slot: each piece waits for the last copy out of its slot, is copied into
// it on the host, and its device copy is enqueued on the context stream.
// `src` is consumed before the call returns; the device copies complete in
// stream order.
int stage_h2d(prism_hip_ctx* ctx, void* dst, const void* src, size_t bytes) {
  if (!ctx->ring[0]) {
    for (int i = 0; i < prism_hip_ctx::kRingSlots; i++) {
      HIP_TRY(ctx, hipHostMalloc(&ctx->ring[i], prism_hip_ctx::kRingSlotBytes, hipHostMallocDefault));
      HIP_TRY(ctx, hipEventCreateWithFlags(&ctx->ring_done[i], hipEventDisableTiming));
    }
  }
  for (size_t off = 0; off < bytes; off += prism_hip_ctx::kRingSlotBytes) {
    const size_t n = std::min(prism_hip_ctx::kRingSlotBytes, bytes - off);
    const int slot = ctx->ring_next;
    ctx->ring_next = (slot + 1) % prism_hip_ctx::kRingSlots;
    HIP_TRY(ctx, hipEventSynchronize(ctx->ring_done[slot]));
    host_copy(ctx->ring[slot], static_cast<const char*>(src) + off, n);
    HIP_TRY(ctx, hipMemcpyAsync(static_cast<char*>(dst) + off, ctx->ring[slot], n, hipMemcpyHostToDevice, ctx->stream));
    HIP_TRY(ctx, hipEventRecord(ctx->ring_done[slot], ctx->stream));
  }
  return PRISM_HIP_OK;
}

struct DeviceGuard {
  int prev = -1;
  explicit DeviceGuard(int dev) {
    if (hipGetDevice(&prev) != hipSuccess) prev = -1;
    if (prev != dev) (void)hipSetDevice(dev);
  }
  ~DeviceGuard() {
    int cur = -1;
    if (prev >= 0 && hipGetDevice(&cur) == hipSuccess && cur != prev) (void)hipSetDevice(prev);
  }
};

// Drop one reference; the last one frees the chunk (hipFree waits for work
// still using it).
void chunk_release(WeightChunk* c) {
  if (!c || c->refs.fetch_sub(1) != 1) return;
  DeviceGuard g(c->device);
  (void)hipFree(c->base);
  delete c;
}

// `bytes` of device memory for a weight: *chunk gets a reference on the
// chunk it lies in.
int weight_alloc(prism_hip_ctx* ctx, size_t bytes, uint8_t** d, WeightChunk** chunk) {
  constexpr size_t kAlign = 256, kOwn = (size_t)16 << 20, kMaxChunk = (size_t)64 << 20;
  const size_t need = (bytes + kAlign - 1) / kAlign * kAlign;
  auto fresh = [&](size_t size, WeightChunk** out) -> int {
    auto* c = new WeightChunk;
    c->size = size;
    c->device = ctx->device;
    const hipError_t e = hipMalloc(&c->base, size);
    if (e != hipSuccess) {
      delete c;
      return fail(ctx, PRISM_HIP_ERR_DEVICE, "weight memory (%zu bytes): hipMalloc: %s", size, hipGetErrorString(e));
    }
    *out = c;
    return PRISM_HIP_OK;
  };
  if (need > kOwn) {
    WeightChunk* c = nullptr;
    const int rc = fresh(need, &c);
    if (rc) return rc;
    c->used = need;
    c->refs = 1;
    *d = c->base;
    *chunk = c;
    return PRISM_HIP_OK;
  }
  if (!ctx->carve || ctx->carve->used + need > ctx->carve->size) {
    // at least `need`: a weight of up to kOwn bytes may exceed the next size
    WeightChunk* c = nullptr;
    const int rc = fresh(std::max(ctx->next_chunk, need), &c);
    if (rc) return rc;
    c->refs = 1;  // the context's
    chunk_release(ctx->carve);
    ctx->carve = c;
    ctx->next_chunk = std::min(kMaxChunk, ctx->next_chunk * 2);
  }
  WeightChunk* c = ctx->carve;
  *d = c->base + c->used;
  c->used += need;
  c->refs.fetch_add(1);
  *chunk = c;
  return PRISM_HIP_OK;
}

int ensure_pool(prism_hip_ctx* ctx) {
  if (ctx->pool) return PRISM_HIP_OK;
  hipMemPoolProps props;
  std::memset(&props, 0, sizeof props);
  props.allocType = hipMemAllocationTypePinned;
  props.handleTypes = hipMemHandleTypeNone;
  props.location.type = hipMemLocationTypeDevice;
  props.location.id = ctx->device;
  hipMemPool_t pool = nullptr;
  HIP_TRY(ctx, hipMemPoolCreate(&pool, &props));
  uint64_t keep = UINT64_MAX;  // never trim at synchronisation points
  const hipError_t e = hipMemPoolSetAttribute(pool, hipMemPoolAttrReleaseThreshold, &keep);
  if (e != hipSuccess) {
    (void)hipMemPoolDestroy(pool);
    return fail(ctx, PRISM_HIP_ERR_DEVICE, "hipMemPoolSetAttribute: %s", hipGetErrorString(e));
  }
  ctx->pool = pool;
  return PRISM_HIP_OK;
}

int check_weight(prism_hip_ctx* ctx, const prism_hip_weight* w) {
  if (!w) return fail(ctx, PRISM_HIP_ERR_NULL, "weight is NULL");
  if (w->ctx != ctx) return fail(ctx, PRISM_HIP_ERR_CONTEXT, "weight was uploaded through another context");
  return PRISM_HIP_OK;
}

hipStream_t pick_stream(prism_hip_ctx* ctx, void* stream) {
  return stream ? reinterpret_cast<hipStream_t>(stream) : ctx->stream;
}

// GI device layout (gemv_lpr.hpp) for 4-bit matrices with rows of at least
// 2048 elements whose rows fill every CU in one round of groups of 32..64
// rows (one group per workgroup; the gate/up form holds two 64 KB table
// sets, one workgroup per CU): G = ceil(N / num_cu) rounded up to a
// multiple of 8, so N = 14336 takes 56-row groups on 256 CUs.  Returns G, or
// 0 for split-block.  MI355X, against k_gemv_tile on split-block weights:
// 14336 x 4096 6.7 (64-row groups, 224 of them) against 8.4 us, gate + up
// 2 x 14336 x 4096 12.3 us; 4864 x 896 3.5 against 3.05 us and 896 x 4864
// 6.3 against 3.2 us (too few rows).
// 4-bit matrices with more than 64 rows per CU, up to 128 (N <= 32768 on 256
// CUs), take 32-row groups and the half-group kernels (gemv_lpr.hpp, HG): a
// workgroup's 64 lanes hold two 32-row groups, two workgroups per CU.
// MI355X, 2 x 18944 x 3584 gate + up (592 workgroups of 32 + 32 rows):
// 13.8 us against 16.2-17.1 on split-block weights and 18.8 with 64-row
// groups (one gate + up workgroup per CU: 296 of them, two rounds); the
// one-matrix 18944 x 3584 GEMV 8.7 against 9.4 us.
// 8-bit matrices take the same groups when K % 512 == 0 (k_gemv_lpr8's
// eight waves split a row into whole blocks of four 16-byte chunks):
// 14336 x 4096 at 1 / 2 / 4 / 8 vectors 11.8 / 12.1 / 13.6 / 18.2 us
// against 14.3 / 15.5 / 18.2 / 19.8 on split-block weights; more than 64
// rows per CU stay split-block.
uint32_t gi_rows(const prism_hip_ctx* ctx, uint32_t dm, uint32_t dn, uint32_t bits) {
  if (dn < 2048 || (bits == 4 && dn % 64 != 0) || (bits == 8 && dn % 512 != 0) || (bits != 4 && bits != 8))
    return 0;
  const uint32_t ncu = (uint32_t)ctx->num_cu;
  uint32_t G = ((dm + ncu - 1) / ncu + 7) / 8 * 8;
  if (bits == 4 && G > (uint32_t)prism::kGiMaxRows && (dm + 63) / 64 <= 2 * ncu) G = 32;
  if (G < 32 || G > (uint32_t)prism::kGiMaxRows || prism::gi_bytes(G, dm, dn, bits) >= (1ull << 31)) return 0;
  return G;
}

// 4-bit GI weights run by the half-group kernels: 32-row groups, more of
// them than CUs (the 32-row groups of N <= 8192 run one group per
// workgroup, lanes 32..63 idle, so that every CU has one).
bool gi_half_groups(const prism_hip_ctx* ctx, const prism_hip_weight* w) {
  return w->bits == 4 && w->gi == 32 && (w->dim_m + 31) / 32 > (uint32_t)ctx->num_cu;
}

// ---------------------------------------------------------------- GEMV plan
// k_gemv_tile (gemv_tile.hpp) for K % 8 == 0 with 16-byte aligned x, in
// passes of up to 8 batch vectors (the matrix-core kernel of gemv_mfma.hpp
// takes several vectors over many rows, up to 16 a pass); k_gemv_generic
// otherwise.

struct TilePlan {
  const void* fn = nullptr;
  int threads = 0;
  int R = 1;
  size_t lds = 0;
};

// WI > 1: WI independent one-wave tiles per workgroup (threads == 64).
template <int BITS, int UPL, int R, bool DUAL, int NB, int EPI, int WI>
TilePlan tile_entry(int threads) {
  TilePlan p;
  p.fn = reinterpret_cast<const void*>(&prism::k_gemv_tile<BITS, UPL, R, DUAL, NB, EPI, WI>);
  if constexpr (WI > 1) {
    p.threads = 64 * WI;
    p.R = R * WI;
    p.lds = WI * prism::gemv_tile_wave_lds_bytes<BITS, R, DUAL, NB>();
  } else {
    p.threads = threads;
    p.R = R;
    p.lds = prism::gemv_tile_lds_bytes<BITS, R, DUAL, NB>(threads);
  }
  return p;
}

// Units per thread of the attention-combine prologue (kEpiAttnIn): at 6..8
// the unrolled combines spilled 8..148 VGPRs, so longer rows take more waves.
constexpr int kAttnInUplMax = 4;

// x units held in VGPRs: NB * UPL * 4 registers, at most 64.
template <int BITS, int R, bool DUAL, int NB, int EPI = 0, int WI = 1>
TilePlan tile_pick_upl(int upl, int threads) {
  switch (upl) {
#define PRISM_TU(u) \
  case u:           \
    if constexpr (NB * (u) <= 16 && ((EPI & prism::kEpiAttnIn) == 0 || (u) <= kAttnInUplMax)) \
      return tile_entry<BITS, u, R, DUAL, NB, EPI, WI>(threads);                                  \
    else                                                                                             \
      return TilePlan{};
    PRISM_TU(1) PRISM_TU(2) PRISM_TU(3) PRISM_TU(4) PRISM_TU(5) PRISM_TU(6) PRISM_TU(7) PRISM_TU(8)
#undef PRISM_TU
  }
  return TilePlan{};
}

// Rows per workgroup: 2 (4 tables for gate+up), 4 for 4+ batch vectors and
// for 8-bit weights (whose LUT loads are spread over >= 256 threads).
// `epi` (prism::kEpiNorm, kEpiResid, kEpiAttnIn | kEpiResid; decode step
// only) is 4-bit, batch 1.
TilePlan plan_tile(uint32_t bits, uint32_t N, uint32_t K, uint32_t nb, bool dual, uintptr_t xaddr, int epi = 0) {
  if (K % 8 != 0 || K == 0 || xaddr % 16 != 0) return TilePlan{};
  // buffer descriptors address the index block and x with 32-bit ranges
  if ((uint64_t)N * K * bits / 8 >= (1ull << 31) || (uint64_t)K * 2 >= (1ull << 31)) return TilePlan{};
  const uint32_t U = K / 8;
  const int NB = nb <= 1 ? 1 : nb <= 2 ? 2 : nb <= 4 ? 4 : 8;
  if (dual && NB != 1) return TilePlan{};
  if (epi == prism::kEpiPair ? !dual : epi && (NB != 1 || bits != 4)) return TilePlan{};
  const uint32_t uplmax = (epi & prism::kEpiAttnIn) ? (uint32_t)kAttnInUplMax : (uint32_t)(16 / NB < 8 ? 16 / NB : 8);
  // Very tall single-vector 4-bit matrices (an LM head: N >= 32768) take 4
  // rows per wave: at 2 rows, dispatching N/2 workgroups costs more than
  // their bytes (measured on 151936 x 896: 47 us at R=2, 26 us at R=4), and
  // one-wave tiles go four to a workgroup (below).
  const bool tall = bits == 4 && NB == 1 && !dual && N >= 32768;
  // 4-bit single-vector rows of 65..128 units (K <= 1024, the decode step's
  // and cfg1's shapes): two independent one-wave tiles per workgroup.
  // MI355X: 4864x896 3.04 against 3.22 us with one two-wave tile (K split
  // over the waves), the Qwen2.5-0.5B decode step 540 against 553 us/token;
  // four tiles: 3.06 / 543.  Longer rows (cfg2's gate_up, K = 3584) lost
  // with two or four (17.2 against 16.4 us).
  const bool pair = bits == 4 && NB == 1 && !tall && U > 64 && U <= 128;
  // waves per workgroup: the fewest that keep UPL <= uplmax; 8-bit rows at
  // least 4
  uint32_t W = 0;
  const uint32_t wmin = bits == 8 ? 4u : 1u;
  for (uint32_t w = wmin; w <= 8; w *= 2)
    if ((U + 64 * w - 1) / (64 * w) <= uplmax) {
      W = w;
      break;
    }
  if (!W) return TilePlan{};
  const int upl = (int)((U + 64 * W - 1) / (64 * W));
  const int threads = (int)(64 * W);
  if (bits == 4) {
    if (pair) {
      if (dual) {
        if (epi == prism::kEpiNorm) return tile_pick_upl<4, 2, true, 1, prism::kEpiNorm, 2>(upl, threads);
        if (epi == prism::kEpiPair) return tile_pick_upl<4, 2, true, 1, prism::kEpiPair, 2>(upl, threads);
        if (epi) return TilePlan{};
        return tile_pick_upl<4, 2, true, 1, 0, 2>(upl, threads);
      }
      if (epi == prism::kEpiNorm) return tile_pick_upl<4, 2, false, 1, prism::kEpiNorm, 2>(upl, threads);
      if (epi == prism::kEpiResid) return tile_pick_upl<4, 2, false, 1, prism::kEpiResid, 2>(upl, threads);
      if (epi == (prism::kEpiAttnIn | prism::kEpiResid))
        return tile_pick_upl<4, 2, false, 1, prism::kEpiAttnIn | prism::kEpiResid, 2>(upl, threads);
      if (epi) return TilePlan{};
      return tile_pick_upl<4, 2, false, 1, 0, 2>(upl, threads);
    }
    if (dual) {
      if (epi == prism::kEpiNorm) return tile_pick_upl<4, 2, true, 1, prism::kEpiNorm>(upl, threads);
      if (epi == prism::kEpiPair) return tile_pick_upl<4, 2, true, 1, prism::kEpiPair>(upl, threads);
      if (epi) return TilePlan{};
      return tile_pick_upl<4, 2, true, 1>(upl, threads);
    }
    if (tall) {
      // one-wave tiles, four to a workgroup: 151936 x 896 in 20.0 us against
      // 24.8 with one tile per workgroup (38 K workgroups to dispatch)
      if (W == 1) {
        if (epi == prism::kEpiNorm) return tile_pick_upl<4, 4, false, 1, prism::kEpiNorm, 4>(upl, threads);
        if (epi == prism::kEpiResid) return tile_pick_upl<4, 4, false, 1, prism::kEpiResid, 4>(upl, threads);
        if (epi) return TilePlan{};
        return tile_pick_upl<4, 4, false, 1, 0, 4>(upl, threads);
      }
      if (epi == prism::kEpiNorm) return tile_pick_upl<4, 4, false, 1, prism::kEpiNorm>(upl, threads);
      if (epi == prism::kEpiResid) return tile_pick_upl<4, 4, false, 1, prism::kEpiResid>(upl, threads);
      if (epi) return TilePlan{};
      return tile_pick_upl<4, 4, false, 1>(upl, threads);
    }
    if (epi == prism::kEpiNorm) return tile_pick_upl<4, 2, false, 1, prism::kEpiNorm>(upl, threads);
    if (epi == prism::kEpiResid) return tile_pick_upl<4, 2, false, 1, prism::kEpiResid>(upl, threads);
    if (epi == (prism::kEpiAttnIn | prism::kEpiResid))
      return tile_pick_upl<4, 2, false, 1, prism::kEpiAttnIn | prism::kEpiResid>(upl, threads);
    if (epi) return TilePlan{};
    switch (NB) {
      case 1: return tile_pick_upl<4, 2, false, 1>(upl, threads);
      case 2: return tile_pick_upl<4, 2, false, 2>(upl, threads);
      case 4: return tile_pick_upl<4, 4, false, 4>(upl, threads);
      default: return tile_pick_upl<4, 4, false, 8>(upl, threads);
    }
  }
  if (dual) {
    if (epi == prism::kEpiPair) return tile_pick_upl<8, 2, true, 1, prism::kEpiPair>(upl, threads);
    return tile_pick_upl<8, 2, true, 1>(upl, threads);
  }
  switch (NB) {
    case 1: return tile_pick_upl<8, 4, false, 1>(upl, threads);
    case 2: return tile_pick_upl<8, 4, false, 2>(upl, threads);
    case 4: return tile_pick_upl<8, 4, false, 4>(upl, threads);
    default: return tile_pick_upl<8, 4, false, 8>(upl, threads);
  }
}

// GEMV over raw split-block device pointers (lut2/idx2 non-null: gate+up
// with the SwiGLU epilogue, or with d_y2 non-null the two raw outputs).
// `epi` selects the decode step's fused norm / residual forms, which have no
// generic fallback.
int launch_gemv_raw(prism_hip_ctx* ctx, uint32_t bits, uint32_t N, uint32_t K, const uint8_t* lut,
                    const uint8_t* idx, const uint8_t* lut2, const uint8_t* idx2, const void* d_x, uint32_t nb,
                    void* d_y, hipStream_t st, int epi = 0, float eps = 0.0f, const float* xpart = nullptr,
                    void* d_y2 = nullptr) {
  const bool dual = (lut2 != nullptr);
  const bool pair = dual && d_y2 != nullptr;
  if (pair) epi = prism::kEpiPair;
  prism::GemvArgs a;
  a.lut = lut;
  a.idx = idx;
  a.lut2 = lut2;
  a.idx2 = idx2;
  a.y2 = reinterpret_cast<uint16_t*>(d_y2);
  a.N = N;
  a.K = K;
  a.eps = eps;
  a.xpart = xpart;
  for (uint32_t b0 = 0; b0 < nb;) {
    uint32_t chunk = (nb - b0 < 8) ? nb - b0 : 8;
    const uint32_t wide = (nb - b0 < (uint32_t)prism::kGmMaxNb) ? nb - b0 : (uint32_t)prism::kGmMaxNb;
    a.x = reinterpret_cast<const uint16_t*>(d_x) + (size_t)b0 * K;
    a.y = reinterpret_cast<uint16_t*>(d_y) + (size_t)b0 * N;
    void* args[] = {&a};
    // Several batch vectors over 4096 rows or more: the matrix-core kernel
    // (gemv_mfma.hpp), from 5 vectors, and for 4-bit rows up to 8192 long
    // from 3 (from 2 over 8192 rows or more).  Against the tile kernel on
    // MI355X: 4-bit 14336x4096 at 8 / 4 / 3 / 2 vectors 11.2 / 10.0 / 9.9 /
    // 9.6 vs 21.8 / 13.3 / 12.9 / 10.2 us; 8-bit at 8 vectors 19.6 vs 26.0
    // us, 29.8 vs 2 x 20 at 4096x14336, 6.1 vs 7.8 at 4864x896.  Slower with
    // fewer rows (2048: 64 workgroups), at one vector (9.5 vs 8.6), for 4-bit
    // at 2 vectors over 4864 rows (4.1 vs 3.6), for 8-bit at 3..4 vectors and
    // for long 4-bit rows at 3..4 (4096x14336: 16.5 vs 14.8).
    // It takes up to 16 vectors a pass, the tile kernel 8.
    const bool mfma_batch =
        wide >= 5 || (bits == 4 && K <= 8192 && (wide >= 3 || (wide == 2 && N >= 8192)));
    if (!dual && !epi && mfma_batch && N >= 4096 && K % prism::kGmGroup == 0 &&
        (uint64_t)N * K * bits / 8 < (1ull << 31) && reinterpret_cast<uintptr_t>(a.x) % 16 == 0) {
      chunk = wide;
      a.nb = chunk;
      const void* fn = bits == 8 ? reinterpret_cast<const void*>(&prism::k_gemv_mfma<8>)
                                 : reinterpret_cast<const void*>(&prism::k_gemv_mfma<4>);
      HIP_TRY(ctx, launch_fn(fn, dim3((N + prism::kGmRows - 1) / prism::kGmRows), dim3(64 * prism::kGmWaves),
                                   args, 0, st));
      b0 += chunk;
      continue;
    }
    TilePlan p = plan_tile(bits, N, K, chunk, dual, reinterpret_cast<uintptr_t>(a.x), epi);
    // rows too long for the tile kernel's registers at this many vectors:
    // fewer vectors per pass (each pass streams the weights again, still far
    // cheaper than the generic kernel: 2 x 20 us against 830 us for 8
    // vectors on 4096x14336 8-bit)
    for (uint32_t c = chunk; !p.fn && c > 1 && !epi && !dual;) {
      c = c > 4 ? 4 : c > 2 ? 2 : 1;
      const TilePlan q = plan_tile(bits, N, K, c, dual, reinterpret_cast<uintptr_t>(a.x), epi);
      if (q.fn) {
        p = q;
        chunk = c;
      }
    }
    a.nb = chunk;
    if (p.fn) {
      const uint32_t grid = (N + (uint32_t)p.R - 1) / (uint32_t)p.R;
      HIP_TRY(ctx, launch_fn(p.fn, dim3(grid), dim3(p.threads), args, p.lds, st));
    } else {
      if (epi && !pair) return fail(ctx, PRISM_HIP_ERR_SHAPE, "no fused kernel for %u-bit %ux%u", bits, N, K);
      const void* fn;
      if (pair)
        fn = bits == 4 ? reinterpret_cast<const void*>(&prism::k_gemv_generic<4, prism::kGenPair>)
                       : reinterpret_cast<const void*>(&prism::k_gemv_generic<8, prism::kGenPair>);
      else if (dual)
        fn = bits == 4 ? reinterpret_cast<const void*>(&prism::k_gemv_generic<4, prism::kGenSwiglu>)
                       : reinterpret_cast<const void*>(&prism::k_gemv_generic<8, prism::kGenSwiglu>);
      else
        fn = bits == 4 ? reinterpret_cast<const void*>(&prism::k_gemv_generic<4, prism::kGenSingle>)
                       : reinterpret_cast<const void*>(&prism::k_gemv_generic<8, prism::kGenSingle>);
      HIP_TRY(ctx, launch_fn(fn, dim3(N), dim3(64), args, 0, st));
    }
    b0 += chunk;
  }
  return PRISM_HIP_OK;
}

// GEMV over GI weights (w2: gate + up, SwiGLU or with d_y2 the pair).
// One or two vectors a pass: k_gemv_lpr; three to eight over groups of more
// than 32 rows, K % 256 == 0 and x within its LDS: k_gemv_lpr4m; otherwise
// three or more: the matrix-core kernel (K % 128 == 0) in passes of up to
// 16, else lane-per-row passes of two.  x not 16-byte aligned: the generic
// kernel.
// k_gemv_lpr with the wave's chunk count as a compile-time constant when
// every wave has the same count (K/32 a multiple of S) and it is 8 or 16,
// else the run-time loop.
template <int S, int NM, int NB, int EPI>
void launch_lpr(dim3 groups, hipStream_t st, const prism::LprArgs& a) {
  const uint32_t NC = a.K / 32;
  const uint32_t nch = NC % S == 0 ? NC / S : 0;
  if (nch == 16)
    PRISM_LAUNCH((prism::k_gemv_lpr<S, NM, NB, EPI, 16>), groups, dim3(64 * S), 0, st, a.w, a.w2, a.x, a.y, a.y2, a.N, a.K, a.nb, a.G);
  else if (nch == 8)
    PRISM_LAUNCH((prism::k_gemv_lpr<S, NM, NB, EPI, 8>), groups, dim3(64 * S), 0, st, a.w, a.w2, a.x, a.y, a.y2, a.N, a.K, a.nb, a.G);
  else
    PRISM_LAUNCH((prism::k_gemv_lpr<S, NM, NB, EPI>), groups, dim3(64 * S), 0, st, a.w, a.w2, a.x, a.y, a.y2, a.N, a.K, a.nb, a.G);
}

// The half-group form (G = 32), with a compile-time chunk count as above,
// and also for 14 chunks per wave (K = 3584 at 8 waves, config 2's rows:
// gate + up 13.8 against 14.55 us for the run-time loop, MI355X; 16 waves
// 16.6, and 15.3-15.4 with 7 compile-time chunks each).
template <int S, int NM, int NB, int EPI>
void launch_lpr_hg(dim3 grid, hipStream_t st, const prism::LprArgs& a) {
  const uint32_t NC = a.K / 32;
  const uint32_t nch = NC % S == 0 ? NC / S : 0;
  if (nch == 16)
    PRISM_LAUNCH((prism::k_gemv_lpr_hg<S, NM, NB, EPI, 16>), grid, dim3(64 * S), 0, st, a.w, a.w2, a.x, a.y, a.y2, a.N, a.K, a.nb, a.G);
  else if (nch == 14)
    PRISM_LAUNCH((prism::k_gemv_lpr_hg<S, NM, NB, EPI, 14>), grid, dim3(64 * S), 0, st, a.w, a.w2, a.x, a.y, a.y2, a.N, a.K, a.nb, a.G);
  else if (nch == 8)
    PRISM_LAUNCH((prism::k_gemv_lpr_hg<S, NM, NB, EPI, 8>), grid, dim3(64 * S), 0, st, a.w, a.w2, a.x, a.y, a.y2, a.N, a.K, a.nb, a.G);
  else
    PRISM_LAUNCH((prism::k_gemv_lpr_hg<S, NM, NB, EPI>), grid, dim3(64 * S), 0, st, a.w, a.w2, a.x, a.y, a.y2, a.N, a.K, a.nb, a.G);
}

// 8-bit GI weights: k_gemv_lpr8 with the wave's chunk count as a
// compile-time constant when it is 16, 32 or 64 (K = 2048 / 4096 / 8192),
// else the loop over 4-chunk blocks.  Eight vectors a pass only with a
// compile-time count (the loop form runs out of SGPRs for their x).
bool lpr8_static(uint32_t K) {
  const uint32_t nch = K / 16 / 8;
  return nch == 16 || nch == 32 || nch == 64;
}
// Eight vectors with a run-time chunk count have no kernel: that returns an
// error (the dispatch below never asks for it) instead of launching nothing.
template <int NM, int NB, int EPI>
int launch_lpr8(prism_hip_ctx* ctx, dim3 groups, hipStream_t st, const prism::LprArgs& a) {
  const uint32_t nch = a.K / 16 / 8;
  if (nch == 32)
    PRISM_LAUNCH((prism::k_gemv_lpr8<8, NM, NB, EPI, 32>), groups, dim3(512), 0, st, a.w, a.w2, a.x, a.y, a.y2, a.N, a.K, a.nb, a.G);
  else if (nch == 16)
    PRISM_LAUNCH((prism::k_gemv_lpr8<8, NM, NB, EPI, 16>), groups, dim3(512), 0, st, a.w, a.w2, a.x, a.y, a.y2, a.N, a.K, a.nb, a.G);
  else if (nch == 64)
    PRISM_LAUNCH((prism::k_gemv_lpr8<8, NM, NB, EPI, 64>), groups, dim3(512), 0, st, a.w, a.w2, a.x, a.y, a.y2, a.N, a.K, a.nb, a.G);
  else if constexpr (NB < 8)
    PRISM_LAUNCH((prism::k_gemv_lpr8<8, NM, NB, EPI>), groups, dim3(512), 0, st, a.w, a.w2, a.x, a.y, a.y2, a.N, a.K, a.nb, a.G);
  else
    return fail(ctx, PRISM_HIP_ERR_SHAPE, "k_gemv_lpr8: %d vectors need a compile-time chunk count (K = %u)", NB,
                a.K);
  return PRISM_HIP_OK;
}

// GEMV over 8-bit GI weights: gate + up (SwiGLU, or the pair with d_y2) in
// one k_gemv_lpr8 pass; one matrix in passes of 1 / 2 vectors (k_gemv_lpr8),
// of 3..8 with the lane-per-row lookups feeding the matrix cores when x fits
// their LDS (k_gemv_lpr8m: nb * (K / 2 + 4) <= 16512), else of 4 or 8
// (k_gemv_lpr8; 3..4 vectors then have K > 8248, so the run-time chunk loop),
// or of up to 16 on the matrix cores from 9 vectors on (from 5 when the
// chunk count is not a compile-time one and x does not fit k_gemv_lpr8m)
// (k_gemv_mfma<8, GI>).  x not 16-byte aligned: the generic kernel.
// Config 4 (14336 x 4096), MI355X, alternating on one box: 3 / 4 vectors
// 12.77-12.81 / 12.95-13.05 us on k_gemv_lpr8m against 13.37-13.50 /
// 13.27-13.39 on k_gemv_lpr8; 2 vectors 12.73-12.80 against 11.92-11.96, so
// 2 stay with k_gemv_lpr8.
int launch_gemv_gi8(prism_hip_ctx* ctx, const prism_hip_weight* w, const prism_hip_weight* w2, const void* d_x,
                    uint32_t nb, void* d_y, void* d_y2, hipStream_t st) {
  const uint32_t N = w->dim_m, K = w->dim_n;
  const bool aligned = reinterpret_cast<uintptr_t>(d_x) % 16 == 0;
  const uint32_t G = w->gi;
  const dim3 groups((N + G - 1) / G);
  prism::GemvArgs ga{};
  ga.gi = G;
  ga.lut = ga.idx = w->d;
  ga.N = N;
  ga.K = K;
  if (w2) {
    ga.lut2 = ga.idx2 = w2->d;
    ga.x = reinterpret_cast<const uint16_t*>(d_x);
    ga.y = reinterpret_cast<uint16_t*>(d_y);
    ga.y2 = reinterpret_cast<uint16_t*>(d_y2);
    ga.nb = 1;
    if (aligned) {
      prism::LprArgs a{};
      a.G = G;
      a.w = w->d;
      a.w2 = w2->d;
      a.x = ga.x;
      a.y = ga.y;
      a.y2 = ga.y2;
      a.N = N;
      a.K = K;
      a.nb = 1;
      const int rc = d_y2 ? launch_lpr8<2, 1, prism::kLprPair>(ctx, groups, st, a)
                          : launch_lpr8<2, 1, prism::kLprSwiglu>(ctx, groups, st, a);
      if (rc) return rc;
    } else if (d_y2) {
      PRISM_LAUNCH((prism::k_gemv_generic<8, prism::kGenPair, true>), dim3(N), dim3(64), 0, st, ga);
    } else {
      PRISM_LAUNCH((prism::k_gemv_generic<8, prism::kGenSwiglu, true>), dim3(N), dim3(64), 0, st, ga);
    }
    HIP_TRY(ctx, hipGetLastError());
    return PRISM_HIP_OK;
  }
  for (uint32_t b0 = 0; b0 < nb;) {
    const uint16_t* x = reinterpret_cast<const uint16_t*>(d_x) + (size_t)b0 * K;
    uint16_t* y = reinterpret_cast<uint16_t*>(d_y) + (size_t)b0 * N;
    const uint32_t left = nb - b0;
    uint32_t chunk;
    if (!aligned) {
      ga.x = x;
      ga.y = y;
      ga.nb = chunk = left;
      PRISM_LAUNCH((prism::k_gemv_generic<8, prism::kGenSingle, true>), dim3(N), dim3(64), 0, st, ga);
    } else if (left >= 3 && left <= 8 && left * (K / 2 + prism::kLpr8mXPad) <= (uint32_t)prism::kLpr8mXDw) {
      prism::LprArgs a{};
      a.G = G;
      a.w = w->d;
      a.x = x;
      a.y = y;
      a.N = N;
      a.K = K;
      a.nb = chunk = left;
      HIP_TRY(ctx, prism::launch_gemv_lpr8m(groups, st, a));
    } else if (left >= 9 || (left >= 5 && !lpr8_static(K))) {
      ga.x = x;
      ga.y = y;
      ga.nb = chunk = left < (uint32_t)prism::kGmMaxNb ? left : (uint32_t)prism::kGmMaxNb;
      PRISM_LAUNCH((prism::k_gemv_mfma<8, true>), dim3((N + prism::kGmRows - 1) / prism::kGmRows),
                   dim3(64 * prism::kGmWaves), 0, st, ga);
    } else {
      prism::LprArgs a{};
      a.G = G;
      a.w = w->d;
      a.x = x;
      a.y = y;
      a.N = N;
      a.K = K;
      a.nb = chunk = left;
      const int rc = left == 1   ? launch_lpr8<1, 1, prism::kLprPlain>(ctx, groups, st, a)
                     : left == 2 ? launch_lpr8<1, 2, prism::kLprPlain>(ctx, groups, st, a)
                     : left <= 4 ? launch_lpr8<1, 4, prism::kLprPlain>(ctx, groups, st, a)
                                 : launch_lpr8<1, 8, prism::kLprPlain>(ctx, groups, st, a);
      if (rc) return rc;
    }
    HIP_TRY(ctx, hipGetLastError());
    b0 += chunk;
  }
  return PRISM_HIP_OK;
}

int launch_gemv_gi(prism_hip_ctx* ctx, const prism_hip_weight* w, const prism_hip_weight* w2, const void* d_x,
                   uint32_t nb, void* d_y, void* d_y2, hipStream_t st) {
  if (w->bits == 8) return launch_gemv_gi8(ctx, w, w2, d_x, nb, d_y, d_y2, st);
  const uint32_t N = w->dim_m, K = w->dim_n;
  const bool aligned = reinterpret_cast<uintptr_t>(d_x) % 16 == 0;
  const uint32_t G = w->gi;
  const dim3 groups((N + G - 1) / G);
  const bool hg = gi_half_groups(ctx, w);
  if (w2) {
    if (aligned) {
      prism::LprArgs a{};
      a.G = G;
      a.w = w->d;
      a.w2 = w2->d;
      a.x = reinterpret_cast<const uint16_t*>(d_x);
      a.y = reinterpret_cast<uint16_t*>(d_y);
      a.y2 = reinterpret_cast<uint16_t*>(d_y2);
      a.N = N;
      a.K = K;
      a.nb = 1;
      // the pair form splits K over the waves as the one-matrix GEMV does
      // (8 waves), so each output is that GEMV's bit for bit
      if (hg) {
        if (d_y2)
          launch_lpr_hg<8, 2, 1, prism::kLprPair>(groups, st, a);
        else
          launch_lpr_hg<8, 2, 1, prism::kLprSwiglu>(groups, st, a);
      } else if (d_y2)
        launch_lpr<8, 2, 1, prism::kLprPair>(groups, st, a);
      else
        launch_lpr<16, 2, 1, prism::kLprSwiglu>(groups, st, a);
    } else {
      prism::GemvArgs a{};
      a.gi = G;
      a.lut = a.idx = w->d;
      a.lut2 = a.idx2 = w2->d;
      a.x = reinterpret_cast<const uint16_t*>(d_x);
      a.y = reinterpret_cast<uint16_t*>(d_y);
      a.y2 = reinterpret_cast<uint16_t*>(d_y2);
      a.N = N;
      a.K = K;
      a.nb = 1;
      if (d_y2)
        PRISM_LAUNCH((prism::k_gemv_generic<4, prism::kGenPair, true>), dim3(N), dim3(64), 0, st, a);
      else
        PRISM_LAUNCH((prism::k_gemv_generic<4, prism::kGenSwiglu, true>), dim3(N), dim3(64), 0, st, a);
    }
    HIP_TRY(ctx, hipGetLastError());
    return PRISM_HIP_OK;
  }
  for (uint32_t b0 = 0; b0 < nb;) {
    const uint16_t* x = reinterpret_cast<const uint16_t*>(d_x) + (size_t)b0 * K;
    uint16_t* y = reinterpret_cast<uint16_t*>(d_y) + (size_t)b0 * N;
    const uint32_t left = nb - b0;
    uint32_t chunk;
    if (!aligned) {
      prism::GemvArgs a{};
      a.gi = G;
      a.lut = a.idx = w->d;
      a.x = x;
      a.y = y;
      a.N = N;
      a.K = K;
      a.nb = chunk = left;
      PRISM_LAUNCH((prism::k_gemv_generic<4, prism::kGenSingle, true>), dim3(N), dim3(64), 0, st, a);
    } else if (!hg && G > 32 && (left == 3 || left == 4) && K % 256 == 0 &&
               left * (K / 2 + prism::kLpr8mXPad) <= (uint32_t)prism::kLpr8mXDw) {
      // 3..4 vectors over groups of 33..64 rows: k_gemv_lpr4q, the lane-per-row
      // lookups feeding 4 x 4 x 4 matrix-core blocks.  MI355X, 14336 x 4096,
      // bench.py alternating on one box: 3 / 4 vectors 8.04-8.21 /
      // 8.10-8.25 us against 8.39-8.50 / 8.43-8.61 for k_gemv_lpr4m.
      prism::LprArgs a{};
      a.G = G;
      a.w = w->d;
      a.x = x;
      a.y = y;
      a.N = N;
      a.K = K;
      a.nb = chunk = left;
      HIP_TRY(ctx, prism::launch_gemv_lpr4q(groups, st, a));
    } else if (!hg && G > 32 && left >= 3 && left <= 8 && K % 256 == 0 &&
               left * (K / 2 + prism::kLpr8mXPad) <= (uint32_t)prism::kLpr8mXDw) {
      // 3..8 vectors over groups of 33..64 rows (both row tiles of
      // k_gemv_lpr4m busy) when x fits its LDS.  MI355X, 14336 x 4096,
      // alternating on one box: 3 / 4 / 8 vectors 8.16-8.24 / 8.26-8.29 /
      // 9.02 us against 9.40-9.42 / 9.48-9.51 / 10.07-10.22 for
      // k_gemv_mfma<4, GI>; 1 / 2 vectors 7.97 / 8.07-8.13 against
      // 6.36-6.38 / 7.59-7.91 for k_gemv_lpr, which keeps them.
      prism::LprArgs a{};
      a.G = G;
      a.w = w->d;
      a.x = x;
      a.y = y;
      a.N = N;
      a.K = K;
      a.nb = chunk = left;
      HIP_TRY(ctx, prism::launch_gemv_lpr4m(groups, st, a));
    } else if (left >= 3 && K % prism::kGmGroup == 0) {
      prism::GemvArgs a{};
      a.gi = G;
      a.lut = a.idx = w->d;
      a.x = x;
      a.y = y;
      a.N = N;
      a.K = K;
      a.nb = chunk = left < (uint32_t)prism::kGmMaxNb ? left : (uint32_t)prism::kGmMaxNb;
      PRISM_LAUNCH((prism::k_gemv_mfma<4, true>), dim3((N + prism::kGmRows - 1) / prism::kGmRows),
                   dim3(64 * prism::kGmWaves), 0, st, a);
    } else {
      prism::LprArgs a{};
      a.G = G;
      a.w = w->d;
      a.x = x;
      a.y = y;
      a.N = N;
      a.K = K;
      a.nb = chunk = left >= 2 ? 2u : 1u;
      if (hg) {
        const dim3 pairs((groups.x + 1) / 2);
        if (chunk == 2)
          launch_lpr_hg<8, 1, 2, prism::kLprPlain>(pairs, st, a);
        else
          launch_lpr_hg<8, 1, 1, prism::kLprPlain>(pairs, st, a);
      } else if (chunk == 2)
        launch_lpr<8, 1, 2, prism::kLprPlain>(groups, st, a);
      else
        launch_lpr<8, 1, 1, prism::kLprPlain>(groups, st, a);
    }
    HIP_TRY(ctx, hipGetLastError());
    b0 += chunk;
  }
  return PRISM_HIP_OK;
}

// GEMVs in passes over the weights.
int launch_gemv_passes(prism_hip_ctx* ctx, const prism_hip_weight* w, const prism_hip_weight* w2, const void* d_x,
                       uint32_t nb, void* d_y, hipStream_t st, void* d_y2 = nullptr) {
  if (w->gi) return launch_gemv_gi(ctx, w, w2, d_x, nb, d_y, d_y2, st);
  return launch_gemv_raw(ctx, w->bits, w->dim_m, w->dim_n, w->lut(), w->idx(), w2 ? w2->lut() : nullptr,
                         w2 ? w2->idx() : nullptr, d_x, nb, d_y, st, 0, 0.0f, nullptr, d_y2);
}

// ---------------------------------------------------------------- GEMM plan
// k_gemm_lookup_x (X as it is, tt x 32 tokens a workgroup) or k_gemm_lookup
// (X packed first; rt x 32 rows and tt x 32 tokens a wave, ks waves sharing a
// token group's K range), over `split` ranges of K whose fp32 partials
// k_gemm_split_sum adds in order, `tokens` of X at a time; or, w4 = 2, 4 or 8,
// k_gemm_w4 with 32 * w4 tokens a block, or, w8, k_gemm8.
struct GemmPlan {
  int w4 = 0;
  bool w8 = false;
  bool packed = false;
  int rt = 2, tt = 1;
  uint32_t ks = prism::kLkWaves, split = 1, per_split = 0, tokens = 0;
  size_t x_bytes = 0, p_bytes = 0;  // scratch of one launch: packed X, partials
  float us = 3.4e38f;               // its estimated time
};

// Grows the context stream's GEMM scratch.
hipError_t ensure_gemm_scratch(prism_hip_ctx* ctx, size_t bytes) {
  if (bytes <= ctx->gemm_bytes) return hipSuccess;
  hipError_t e;
  if (ctx->d_gemm) {
    if ((e = hipStreamSynchronize(ctx->stream)) != hipSuccess) return e;
    if ((e = hipFree(ctx->d_gemm)) != hipSuccess) return e;
    ctx->d_gemm = nullptr;
    ctx->gemm_bytes = 0;
  }
  size_t size = (size_t)1 << 20;
  while (size < bytes) size <<= 1;
  if ((e = hipMalloc(&ctx->d_gemm, size)) == hipSuccess) ctx->gemm_bytes = size;
  return e;
}

// The plan's scratch sizes and the tokens one launch takes (all of M, or with
// a large M as many as keep packed X within the scratch and the launch below 2^32
// threads); false when the partials do not fit.
bool plan_sizes(GemmPlan* p, uint32_t bits, uint32_t M, uint32_t N, uint32_t K) {
  const uint32_t step = prism::lk_step(bits);
  const uint32_t units = p->packed ? (K + 2 * step - 1) / (2 * step) : (K + step - 1) / step;
  p->per_split = (units + p->split - 1) / p->split;
  p->split = (units + p->per_split - 1) / p->per_split;
  p->tokens = M;
  p->x_bytes = p->p_bytes = 0;
  // in tiles of 32 tokens: a workgroup's, what launch and scratch hold
  const uint32_t rows = p->packed ? 32u * p->rt : 64u;
  const uint32_t group = (uint32_t)p->tt * (p->packed ? prism::kLkWaves / p->ks : 1);
  const size_t tile = p->packed ? (size_t)units * 2 * step * 64 : 0;
  size_t fit = std::max<size_t>(1, 0xFFFFFFFFu / (64 * prism::kLkWaves) / ((N + rows - 1) / rows)) * group;
  if (p->packed) fit = std::min(fit, kGemmScratchBytes / tile);
  if (fit < (M + 31) / 32) {
    if (fit > group) fit = fit / group * group;
    if (fit == 0 || p->split > 1) return false;
    p->tokens = (uint32_t)fit * 32;
  }
  if (p->packed) p->x_bytes = (p->tokens + 31) / 32 * tile;
  if (p->split > 1) p->p_bytes = (size_t)p->split * M * N * 4;
  return p->x_bytes + p->p_bytes <= kGemmScratchBytes;
}

// Index (or LUT) bytes one launch addresses with 31-bit buffer offsets.
constexpr size_t kMaxIndexBytes = 0x7F000000;

int run_gemm_blocks(prism_hip_ctx* ctx, const prism_hip_weight* w, const GemmPlan& p, const void* d_X, uint32_t M,
                    void* d_Y, hipStream_t st) {
  const uint8_t *lut = w->lut(), *idx = w->idx();
  const uint16_t* X = static_cast<const uint16_t*>(d_X);
  uint16_t* Y = static_cast<uint16_t*>(d_Y);
  uint32_t N = w->dim_m, K = w->dim_n, G = w->gi;
  const void* fn;
#define PRISM_GI(K_, ...) \
  (G ? reinterpret_cast<const void*>(&prism::K_<__VA_ARGS__ true>) : reinterpret_cast<const void*>(&prism::K_<__VA_ARGS__ false>))
  if (p.w8)
    fn = PRISM_GI(k_gemm8, );
  else
    fn = p.w4 == 2 ? PRISM_GI(k_gemm_w4, 2, ) : p.w4 == 4 ? PRISM_GI(k_gemm_w4, 4, ) : PRISM_GI(k_gemm_w4, 8, );
#undef PRISM_GI
  const uint32_t bm = p.w8 ? prism::GM8_BM : 32u * p.w4, bn = p.w8 ? prism::GM8_BN : prism::GW4_BN;
  void* args[] = {&lut, &idx, &X, &Y, &M, &N, &K, &G};
  HIP_TRY(ctx, launch_fn(fn, dim3((M + bm - 1) / bm * ((N + bn - 1) / bn)), dim3(256), args, 0, st));
  return PRISM_HIP_OK;
}

int run_gemm(prism_hip_ctx* ctx, const prism_hip_weight* w, GemmPlan p, const void* d_X, uint32_t M, void* d_Y,
             hipStream_t st, float* fixed) {
  if (p.w4 || p.w8) return run_gemm_blocks(ctx, w, p, d_X, M, d_Y, st);
  const uint32_t N = w->dim_m, K = w->dim_n, bits = w->bits, step = prism::lk_step(bits);
  const size_t need = p.x_bytes + p.p_bytes;
  // scratch: the caller's, the context stream's kept one, or on another
  // stream one of the call's own from the pool
  void* scratch_mem = fixed;
  bool temp = false;
  if (need && !fixed) {
    hipError_t e = hipSuccess;
    if (st == ctx->stream) {
      e = ensure_gemm_scratch(ctx, need);
      scratch_mem = ctx->d_gemm;
    } else {
      int rc = ensure_pool(ctx);
      if (rc) return rc;
      e = hipMallocFromPoolAsync(&scratch_mem, need, ctx->pool, st);
      temp = e == hipSuccess;
    }
    if (e != hipSuccess) {
      if (e != hipErrorOutOfMemory) return fail(ctx, PRISM_HIP_ERR_DEVICE, "GEMM scratch: %s", hipGetErrorString(e));
      (void)hipGetLastError();  // no memory for scratch: the kernel that needs none
      p = GemmPlan{};
      p.tt = 2;
      plan_sizes(&p, bits, M, N, K);
    }
  }
  prism::LkArgs a{};
  a.P = p.split > 1 ? reinterpret_cast<float*>(static_cast<uint8_t*>(scratch_mem) + p.x_bytes) : nullptr;
  a.K = K;
  a.ldy = N;
  a.G = w->gi;
  a.per_split = p.per_split;
  a.KS = p.ks;
  const uint32_t unit = p.packed ? 2 * step : step;
  const void* fn = p.packed ? prism::lk_kernel(bits, p.rt, p.tt, K % unit != 0)
                            : prism::lkx_kernel(bits, p.tt, K % unit != 0);
  const uint32_t rows = p.packed ? 32u * p.rt : 64u;
  const uint32_t group = 32u * p.tt * (p.packed ? prism::kLkWaves / p.ks : 1u);
  // index and LUT offsets are 31-bit: split-block weights past 2 GiB of either go in row slabs.
  // GI weights are below 2 GiB whole (gi_rows), and their rows lie in groups: never cut.
  const size_t row_bytes = (size_t)K * bits / 8;
  const uint32_t slab = w->gi ? N
                              : (uint32_t)std::min<size_t>(
                                    N, kMaxIndexBytes / std::max<size_t>(row_bytes, 2u << bits) / rows * rows);
  hipError_t e = hipSuccess;
  for (uint32_t m = 0; m < M && e == hipSuccess; m += p.tokens) {
    const uint16_t* X = static_cast<const uint16_t*>(d_X) + (size_t)m * K;
    a.M = std::min(p.tokens, M - m);
    a.X = X;
    if (p.packed) {
      uint16_t* Xp = static_cast<uint16_t*>(scratch_mem);
      uint32_t steps = (K + unit - 1) / unit * 2, tiles = (a.M + 31) / 32, k = K;
      void* pa[] = {&X, &Xp, &a.M, &k, &steps, &tiles};
      const size_t pieces = (size_t)tiles * 32 * steps * (step / 8);
      e = launch_fn(prism::lk_pack_kernel(bits), dim3((unsigned)((pieces + 255) / 256)), dim3(256), pa, 0, st);
      a.X = Xp;
    }
    for (uint32_t n = 0; n < N && e == hipSuccess; n += slab) {
      a.N = std::min(slab, N - n);
      a.lut = w->lut() + (size_t)n * (2u << bits);
      a.idx = w->idx() + (size_t)n * row_bytes;
      a.Y = static_cast<uint16_t*>(d_Y) + (size_t)m * N + n;
      void* args[] = {&a};
      e = launch_fn(fn, dim3((a.N + rows - 1) / rows * ((a.M + group - 1) / group), p.split), dim3(64 * prism::kLkWaves),
                    args, 0, st);
    }
  }
  if (e == hipSuccess && a.P) {
    const uint64_t mn = (uint64_t)M * N;
    PRISM_LAUNCH(prism::k_gemm_split_sum, dim3((unsigned)((mn + 1023) / 1024)), dim3(256), 0, st, a.P,
                 static_cast<uint16_t*>(d_Y), mn, p.split);
    e = hipGetLastError();
  }
  if (temp) {
    const hipError_t f = hipFreeAsync(scratch_mem, st);
    if (e == hipSuccess) e = f;
  }
  if (e != hipSuccess) return fail(ctx, PRISM_HIP_ERR_DEVICE, "GEMM launch: %s", hipGetErrorString(e));
  return PRISM_HIP_OK;
}

// Estimated time of a plan in us on MI355X.  Fitted to every plan of 730 shapes
// (64 .. 151936 rows of 768 .. 16384, odd ones among them) at 5 to 17 numbers of
// tokens each from 5 to 2048, over weights in the Infinity Cache and over as many
// that they are not, for the least time lost by the plan it picks: with scratch 0.5 %
// over the fastest plan on average, one in twenty over 4 %, at most 26; without, 0.1 %
// and at most 20.  (Shapes left out of the fit: 0.7 and 0.1 %, at most 19 and 14.)
float gemm_plan_us(const GemmPlan& p, uint32_t bits, uint32_t gi, uint32_t M, uint32_t N, uint32_t K,
                   uint32_t num_cu) {
  const float mn = (float)M * (float)N * 1e-6f;
  auto rounds = [&](uint64_t groups) { return (float)((groups + num_cu - 1) / num_cu); };  // over the CUs
  if (p.w4 || p.w8) {
    // k_gemm_w4 of 64, 128 and 256 tokens, k_gemm8: fixed us, us per step, more with all CUs busy; the
    // same for each round after the first, of which a last one that is not full counts a quarter for
    // its share of the CUs; us per million outputs
    static const float kBlocks[4][6] = {{4.09f, 0.728f, 0.0129f, 2.68f, 0.594f, 0.0484f},
                                        {8.49f, 0.685f, 0.212f, 10.6f, 0.846f, 0.0242f},
                                        {12.8f, 1.1f, 0.344f, 13.6f, 1.5f, 0.0559f},
                                        {10.1f, 1.54f, 0.0145f, 12.6f, 1.67f, 0.0112f}};
    static_assert(prism::GM8_BK == prism::GW4_BK, "one K step for both");
    const float* f = kBlocks[p.w8 ? 3 : p.w4 == 8 ? 2 : p.w4 / 4];
    const uint32_t bm = p.w8 ? prism::GM8_BM : 32u * p.w4, bn = p.w8 ? prism::GM8_BN : prism::GW4_BN;
    const uint64_t tiles = (uint64_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn);
    const float steps = (float)(K / prism::GW4_BK), fill = (float)tiles / (float)num_cu;
    const float more = 0.25f * std::max(1.0f, fill) + 0.75f * rounds(tiles) - 1.0f;
    return f[0] + steps * (f[1] + f[2] * std::min(1.0f, fill)) + more * (f[3] + steps * f[4]) + f[5] * mn;
  }
  const uint32_t rows = p.packed ? 32u * p.rt : 64u, blocks = (N + rows - 1) / rows;
  const uint32_t group = 32u * p.tt * (p.packed ? prism::kLkWaves / p.ks : 1u);
  const float r = rounds((uint64_t)blocks * ((M + group - 1) / group) * p.split);
  const float steps = (float)((p.packed ? 2u : 1u) * ((p.per_split + p.ks - 1) / p.ks));
  // MB of x that the row blocks read; stores of single values, where N does not allow whole ones
  const float x_mb = (float)blocks * (float)M * (float)K * 2e-6f;
  const float odd = N % (p.packed && p.ks == 1 && p.split == 1 ? 8 : 4) ? (float)p.split * mn : 0.0f;
  const float sum = p.split > 1 ? 1.0f : 0.0f, partials = sum * (float)p.split * mn;
  const float astray = (uint64_t)K * bits / 8 % 16 ? r * steps : 0.0f;  // steps over index rows that are not aligned
  const float apart = gi ? 0.0f : r * steps;  // steps whose lanes read index rows apart, not GI groups
  const float unaligned = (uint64_t)M * N % 4 ? sum * (float)p.split : 0.0f;  // partials the sum reads one by one
  if (!p.packed) {
    // 32 and 64 tokens: fixed us (LUT loads, tables, sum, store), us per step; the same for each
    // round after the first; us per MB of x; the sum's launch and its us per million partials; us per
    // million single stores, per split whose partials are not aligned, per step over unaligned rows
    // and over rows that are not GI
    static const float kX[2][2][11] = {
        {{3.81f, 0.57f, 2.5f, 0.752f, 0.0172f, 2.12f, 1.35f, 0.202f, 0.568f, 0.0894f, 0.296f},
         {5.59f, 0.914f, 3.1f, 1.23f, 0.0213f, 2.16f, 2.29f, 0.189f, 0.438f, 0.469f, 0.13f}},
        {{3.56f, 0.509f, 3.81f, 0.461f, 0.033f, 2.83f, 0.127f, 0.0018f, 0.626f, 0.0f, 0.364f},
         {6.07f, 0.747f, 3.52f, 0.664f, 0.0284f, 2.16f, 1.76f, 1.01f, 0.444f, 0.148f, 0.19f}}};
    const float* f = kX[bits == 8][p.tt - 1];
    return f[0] + steps * f[1] + (r - 1.0f) * (f[2] + steps * f[3]) + f[4] * x_mb + f[5] * sum + f[6] * partials +
           f[7] * odd + f[8] * unaligned + f[9] * astray +
           f[10] * apart;
  }
  // 64 x 64 and 128 x 64 (4 bits) or 64 x 128 (8 bits) a wave: per round fixed us and us per step, more
  // with all waves at work (not past M) and with each doubling of the waves on one token group; us per
  // MB of x; k_pack_x, a launch and its us per million elements; the sum and the stores as above
  static const float kP[2][2][13] = {
      {{3.85f, 0.0931f, 0.517f, 0.0701f, 0.0234f, 4.0f, 1.25f, 4.04f, 0.52f, 2.01f, 0.171f, 0.0151f, 0.104f},
       {7.7f, 0.246f, 0.546f, 0.0936f, 0.0383f, 4.56f, 0.444f, 5.18f, 0.904f, 2.26f, 0.365f, 0.00727f, 0.317f}},
      {{4.15f, 0.0812f, 0.498f, 0.121f, 0.0111f, 3.54f, 0.912f, 4.91f, 0.837f, 2.56f, 0.252f, 0.0263f, 0.0236f},
       {9.37f, 0.0948f, 0.769f, 0.0749f, 0.00277f, 4.15f, 0.435f, 3.04f, 1.45f, 2.44f, 0.651f, 0.0953f, 0.000496f}}};
  const float* f = kP[bits == 8][p.rt * p.tt > 4];
  const float live = std::min(1.0f, (float)(p.ks * ((M + 32u * p.tt - 1) / (32u * p.tt))) / (float)prism::kLkWaves);
  const float doublings = p.ks == 8 ? 3.0f : p.ks == 4 ? 2.0f : p.ks == 2 ? 1.0f : 0.0f;
  return r * (f[0] + steps * (f[1] + (f[2] + doublings * f[3]) * live)) + f[4] * x_mb + f[5] +
         f[6] * (float)M * (float)K * 1e-6f + f[7] * sum + f[8] * partials + f[9] * odd +
         f[10] * unaligned + f[11] * astray + f[12] * apart;
}

// Where a call's scratch (packed X, partials) comes from: kept memory, the pool
// for this call, or none may be used.
enum class Scratch { kKept, kCall, kNone };

// The fastest plan by that estimate.  Every kernel is ahead somewhere (MI355X,
// with scratch kept, us of the fastest plan of each):
//  * k_gemm_lookup_x, up to 32 tokens the only one: above them in blocks of 32 tokens
//    where those fill the CUs better (2752 x 1792, 128 tokens 7.0 against 9.8 in
//    blocks of 64), and of 64 where 32 take more rounds (14336 x 4096, 33 tokens
//    14.5);
//  * k_gemm_lookup above 32 tokens: X is packed once and not read unpacked by each 64
//    rows (14336 x 4096, 256 tokens 39 against 52);
//  * k_gemm_w4, which decodes each block's weights once, above 32 (151936 x 896,
//    64 tokens 34.7 against 65.3);
//  * k_gemm8 where no scratch may be used, above 256 tokens at 8 bits (14336 x 4096,
//    2048 tokens 441 against 577 in k_gemm_lookup_x).
// Scratch of the call's own is allocated and freed on each call: 3..5 us more, and
// no call below about 22 us of host time (14336 x 4096, 80 / 300 tokens 23.6 / 51.5
// us with kept scratch, 28.6 / 54.4 with its own).
GemmPlan plan_gemm(uint32_t bits, uint32_t gi, uint32_t M, uint32_t N, uint32_t K, uint32_t num_cu,
                   Scratch scratch) {
  GemmPlan best;
  // (weights that run_gemm cuts into row slabs have no partials)
  const uint32_t max_split = (uint64_t)N * K * bits / 8 < kMaxIndexBytes ? 16 : 1;
  auto consider = [&](bool packed, int rt, int tt, uint32_t ks) {
    // (not with half the waves past M, nor splits of what fills the CUs four times: 1..2 us of host
    // time at 33..64 tokens)
    const uint32_t tiles = (M + 32u * tt - 1) / (32u * tt), waves = packed ? prism::kLkWaves / ks : 1;
    if (waves >= 2 * tiles) return;
    const uint64_t groups = (uint64_t)(N / (32u * rt)) * ((tiles + waves - 1) / waves);
    for (uint32_t split = 1; split <= max_split && (split == 1 || groups * split < 8 * num_cu); split *= 2) {
      GemmPlan p;
      p.packed = packed;
      p.rt = rt;
      p.tt = tt;
      p.ks = ks;
      p.split = split;
      if (!plan_sizes(&p, bits, M, N, K)) continue;
      if (scratch == Scratch::kNone && p.x_bytes + p.p_bytes) continue;
      p.us = gemm_plan_us(p, bits, gi, M, N, K, num_cu);
      if (scratch == Scratch::kCall && p.x_bytes + p.p_bytes) p.us = std::max(p.us + 4.0f, 22.0f);
      if (p.us < best.us) best = p;
    }
  };
  consider(false, 2, 1, prism::kLkWaves);
  if (M > 32) {
    consider(false, 2, 2, prism::kLkWaves);
    for (uint32_t ks = 1; ks <= prism::kLkWaves; ks *= 2) {
      consider(true, 2, 2, ks);
      if (bits == 4)
        consider(true, 4, 2, ks);
      else
        consider(true, 2, 4, ks);
    }
  }
  if (bits == 4 && M > 32 && K % prism::GW4_BK == 0 && (uint64_t)N * (K / 2) < (1ull << 31) &&
      (uint64_t)K * 512 < (1ull << 31))
    for (int mi = 2; mi <= 8; mi *= 2) {
      GemmPlan p;
      p.w4 = mi;
      p.us = gemm_plan_us(p, bits, gi, M, N, K, num_cu);
      if (p.us < best.us) best = p;
    }
  if (bits == 8 && scratch == Scratch::kNone && M > 256 && K % prism::GM8_BK == 0) {
    GemmPlan p;
    p.w8 = true;
    p.us = gemm_plan_us(p, bits, gi, M, N, K, num_cu);
    if (p.us < best.us) best = p;
  }
  if (best.us > 3e38f) {  // rows too long for the scratch: the kernel that needs none
    best = GemmPlan{};
    best.tt = 2;
    plan_sizes(&best, bits, M, N, K);
  }
  return best;
}

// Estimated time of M vectors (5..32; over GI weights 9 and more) as GEMV passes, us on MI355X:
//  * the matrix-core GEMV in passes of 16 where it runs: fixed us, then for each round
//    of workgroups a fixed part and us per 1000 elements of K, with none and with each
//    vector; and us per 1000 elements of K and row that the last workgroup lacks, whose
//    lanes all look up the last row's elements in one LDS bank;
//  * else over GI weights lane-per-row passes of two;
//  * else the tile GEMV in passes of 8 vectors (fewer for long rows): fixed us, more
//    for each doubling of its vectors, us per million weights, with none and with each
//    vector, and with each vector us per million rows and per 1000 elements of K.
// No pass is below a multiple of the weights' bytes at 5.5 TB/s.  Fitted to the
// passes of 450 shapes, within 4 (4 bits) and 8..10 % (8 bits, tile) root mean square.
float passes_us(uint32_t bits, uint32_t gi, uint32_t M, uint32_t N, uint32_t K, uint32_t num_cu) {
  const bool near = (uint64_t)N * K * bits / 8 < (1ull << 31);
  const float floor_us = (float)N * ((float)K * (float)bits / 8 + (float)(2u << bits)) / 5.5e6f;  // the weights' bytes
  const float k = (float)K * 1e-3f, m = (float)N * 1e-6f;
  float us = 0.0f;
  if (gi && bits == 4 && K % prism::kGmGroup != 0) return (float)((M + 1) / 2) * 1.4f * floor_us;
  if (gi || (K % prism::kGmGroup == 0 && N >= 4096 && near)) {
    static const float kMfma[2][2][6] = {
        {{2.59f, 0.67f, 0.83f, 0.031f, 1.2f, 0.004f}, {3.3f, 0.17f, 0.465f, 0.042f, 1.32f, 0.007f}},
        {{3.0f, 1.27f, 1.36f, 0.048f, 1.22f, 0.13f}, {4.67f, 0.0f, 1.06f, 0.045f, 1.29f, 0.13f}}};
    const float* f = kMfma[bits == 8][gi != 0];
    const float rounds = (float)(((N + prism::kGmRows - 1) / prism::kGmRows + num_cu - 1) / num_cu);
    const float lacks = k * (float)((prism::kGmRows - N % prism::kGmRows) % prism::kGmRows);
    for (uint32_t n = M; n; n -= std::min(n, 16u))
      us += std::max(f[4] * floor_us,
                     f[0] + rounds * (f[1] + k * (f[2] + f[3] * (float)std::min(n, 16u))) + f[5] * lacks);
    return us;
  }
  static const float kTile[2][7] = {{2.8f, 0.343f, 0.025f, 0.039f, 20.5f, 0.026f, 2.2f},
                                    {2.78f, 0.22f, 0.178f, 0.014f, 75.0f, 0.048f, 1.56f}};
  const float* f = kTile[bits == 8];
  for (uint32_t n = M; n;) {
    uint32_t c = std::min(n, 8u), nb, lg;
    for (;; c = nb / 2) {  // vectors of a pass whose x fits the registers of 8 waves
      for (nb = 1, lg = 0; nb < c; nb *= 2) lg++;
      if (near && (K / 8 + 511) / 512 <= std::min(8u, 16 / nb)) break;
      if (nb == 1) return 3.4e38f;  // the generic kernel, whatever it takes
    }
    us += std::max(f[6] * floor_us, f[0] + f[1] * (float)lg + m * (float)K * (f[2] + f[3] * (float)nb) +
                                        (float)nb * (f[4] * m + f[5] * k));
    n -= c;
  }
  return us;
}

// Whether M tokens can go to the GEMM kernels rather than to GEMV passes: 5 and
// more, rows in eights below 2^24, aligned x.  GI calls of up to 8 vectors have
// kernels of their own, and `gemv` (the GEMV entry points) keeps passes for those
// of more than 16.
bool gemm_can(const prism_hip_weight* w, const void* d_x, uint32_t M, bool gemv) {
  const uint32_t K = w->dim_n;
  if (K % 8 != 0 || reinterpret_cast<uintptr_t>(d_x) % 16 != 0) return false;
  // 31-bit offsets: 64 tokens of x (and with that a tile's rows of indices) below 2 GiB
  if ((uint64_t)K * 64 * 2 >= (1ull << 31)) return false;
  return w->gi ? M > 8 && !(gemv && M > 16) : M > 4;
}

// Whether the plan goes ahead of passes: above 32 tokens always, else by both
// estimates, with 3 % for passes (0.4 % over the faster side on average, at most 27).  MI355X, plan
// against passes on the context's stream: 14336 x 4096, 32 tokens, 4 bits 9.4
// against 23.0 us, 16 tokens 9.2 against 12.1; 14592 x 13184, 14 tokens 20.5 against
// 31.1; 4096 x 14336, 8 tokens 12.0 against 18.5, but 19.9 where it cannot split K
// (a caller's stream, capture: 24.3); 4096 x 4096, 9 tokens 8.4 against 6.9; 256 x
// 8192, 8 tokens 8.5 against 6.0, captured 15.8 against 7.1; 151936 x 896, 8
// tokens, 8 bits 76 against 57.
bool gemm_goes_first(const prism_hip_ctx* ctx, const prism_hip_weight* w, uint32_t M, const GemmPlan& p) {
  return M > 32 || 1.03f * p.us < passes_us(w->bits, w->gi, M, w->dim_m, w->dim_n, (uint32_t)ctx->num_cu);
}

// A call on the context's stream uses its buffer, one on a caller's stream memory
// of its own, and under the capture of a caller's stream none: a captured call
// is kernels alone, with no memory of its own in the graph.
int scratch_of(prism_hip_ctx* ctx, hipStream_t st, Scratch* out) {
  *out = Scratch::kKept;
  if (st == ctx->stream) return PRISM_HIP_OK;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  HIP_TRY(ctx, hipStreamIsCapturing(st, &cap));
  *out = cap == hipStreamCaptureStatusNone ? Scratch::kCall : Scratch::kNone;
  return PRISM_HIP_OK;
}

int launch_gemm(prism_hip_ctx* ctx, const prism_hip_weight* w, const void* d_X, uint32_t M, void* d_Y,
                hipStream_t st, float* fixed = nullptr, bool gemv = false) {
  if (gemm_can(w, d_X, M, gemv)) {
    Scratch sc = Scratch::kKept;  // (`fixed` is)
    const int rc = fixed ? PRISM_HIP_OK : scratch_of(ctx, st, &sc);
    if (rc) return rc;
    const GemmPlan p = plan_gemm(w->bits, w->gi, M, w->dim_m, w->dim_n, (uint32_t)ctx->num_cu, sc);
    if (gemm_goes_first(ctx, w, M, p)) return run_gemm(ctx, w, p, d_X, M, d_Y, st, fixed);
  }
  return launch_gemv_passes(ctx, w, nullptr, d_X, M, d_Y, st);
}

// prism_hip_gemv and its like: several vectors may be the GEMM kernels'.
int launch_gemv(prism_hip_ctx* ctx, const prism_hip_weight* w, const prism_hip_weight* w2, const void* d_x,
                uint32_t nb, void* d_y, hipStream_t st, void* d_y2 = nullptr) {
  if (w2) return launch_gemv_passes(ctx, w, w2, d_x, nb, d_y, st, d_y2);
  return launch_gemm(ctx, w, d_x, nb, d_y, st, nullptr, true);
}

int launch_decode(prism_hip_ctx* ctx, const prism_hip_weight* w, uint32_t row0, uint32_t nrows, void* d_out,
                  hipStream_t st) {
  const size_t total = (size_t)nrows * w->dim_n;
  if (total == 0) return PRISM_HIP_OK;
  size_t blocks = (total + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  const uint8_t* lut = w->lut();
  const uint8_t* idx = w->idx();
  uint32_t N = w->dim_m, K = w->dim_n;
  uint16_t* out = reinterpret_cast<uint16_t*>(d_out);
  uint32_t G = w->gi;
  void* args[] = {&lut, &idx, &N, &K, &row0, &nrows, &out, &G};
  const void* fn = w->bits == 8 ? (w->gi ? reinterpret_cast<const void*>(&prism::k_decode_rows<8, true>)
                                        : reinterpret_cast<const void*>(&prism::k_decode_rows<8>))
                   : w->gi      ? reinterpret_cast<const void*>(&prism::k_decode_rows<4, true>)
                                : reinterpret_cast<const void*>(&prism::k_decode_rows<4>);
  HIP_TRY(ctx, launch_fn(fn, dim3((unsigned)blocks), dim3(256), args, 0, st));
  return PRISM_HIP_OK;
}

// A 4-bit weight's LUT block and index rows in split-block form at dst_lut
// ([N][32] B) and dst_idx ([N][K/2] B), on stream st: copies, or for a GI
// weight the inverse regrouping.
int copy_split_rows(prism_hip_ctx* ctx, const prism_hip_weight* w, uint8_t* dst_lut, uint8_t* dst_idx,
                    hipStream_t st) {
  const uint32_t N = w->dim_m, K = w->dim_n;
  if (!w->gi) {
    HIP_TRY(ctx, hipMemcpyAsync(dst_lut, w->lut(), (size_t)N * 32, hipMemcpyDeviceToDevice, st));
    HIP_TRY(ctx, hipMemcpyAsync(dst_idx, w->idx(), (size_t)N * (K / 2), hipMemcpyDeviceToDevice, st));
    return PRISM_HIP_OK;
  }
  const size_t pieces = (size_t)N * (2 + K / 32);
  const unsigned grid = (unsigned)std::min<size_t>((pieces + 255) / 256, 16384);
  PRISM_LAUNCH(prism::k_gi_unpack, dim3(grid), dim3(256), 0, st, w->d, dst_lut, dst_idx, N, K, w->gi);
  HIP_TRY(ctx, hipGetLastError());
  return PRISM_HIP_OK;
}



}  // namespace

// =========================================================================
extern "C" {

const char* prism_hip_version(void) { return PRISM_HIP_VERSION; }

prism_hip_ctx* prism_hip_ctx_create(int device) {
  int n = 0;
  hipError_t e = hipGetDeviceCount(&n);
  if (e != hipSuccess || n == 0) {
    g_create_err = std::string("no HIP device: ") + hipGetErrorString(e);
    return nullptr;
  }
  if (device < 0 || device >= n) {
    g_create_err = "device index " + std::to_string(device) + " out of range (" + std::to_string(n) + " devices)";
    return nullptr;
  }
  DeviceGuard g(device);
  hipDeviceProp_t prop;
  if ((e = hipGetDeviceProperties(&prop, device)) != hipSuccess) {
    g_create_err = std::string("hipGetDeviceProperties: ") + hipGetErrorString(e);
    return nullptr;
  }
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
    g_create_err = std::string("device is ") + prop.gcnArchName + ", this library is built for gfx950";
    return nullptr;
  }
  auto* ctx = new prism_hip_ctx;
  ctx->device = device;
  ctx->num_cu = prop.multiProcessorCount;
  ctx->lds_max = prop.sharedMemPerBlock;
  if ((e = hipStreamCreateWithFlags(&ctx->stream, hipStreamNonBlocking)) != hipSuccess) {
    g_create_err = std::string("hipStreamCreate: ") + hipGetErrorString(e);
    delete ctx;
    return nullptr;
  }
  alloc_host_io(ctx);
  g_create_err.clear();
  return ctx;
}

void prism_hip_ctx_destroy(prism_hip_ctx* ctx) {
  if (!ctx) return;
  DeviceGuard g(ctx->device);
  for (prism_hip_weight* w : ctx->weights) w->ctx = nullptr;
  ctx->weights.clear();
  for (prism_hip_model* m : ctx->models) model_detach(m);
  ctx->models.clear();
  if (ctx->stream) {
    (void)hipStreamSynchronize(ctx->stream);
    (void)hipStreamDestroy(ctx->stream);
  }
  if (ctx->d_stage) (void)hipFree(ctx->d_stage);
  if (ctx->h_io) (void)hipHostFree(ctx->h_io);
  if (ctx->d_upload) (void)hipFree(ctx->d_upload);
  if (ctx->d_gemm) (void)hipFree(ctx->d_gemm);
  chunk_release(ctx->carve);
  for (int i = 0; i < prism_hip_ctx::kRingSlots; i++) {
    if (ctx->ring[i]) (void)hipHostFree(ctx->ring[i]);
    if (ctx->ring_done[i]) (void)hipEventDestroy(ctx->ring_done[i]);
  }
  if (ctx->pool) {
    (void)hipDeviceSynchronize();  // scratch freed on other streams
    (void)hipMemPoolDestroy(ctx->pool);
  }
  delete ctx;
}

const char* prism_hip_last_error(const prism_hip_ctx* ctx) {
  return ctx ? ctx->err.c_str() : g_create_err.c_str();
}

const char* prism_hip_last_kernels(prism_hip_ctx* ctx) {
  if (!ctx) return "";
  if (ctx->kernels.empty() && !ctx->launched.empty()) {
    // device names of the recorded host functions, demangled and shortened
    // to the kernel's own name and template arguments
    std::string out, prev;
    int run = 0;
    auto flush = [&] {
      if (prev.empty()) return;
      if (!out.empty()) out += " + ";
      out += prev;
      if (run > 1) out += " x" + std::to_string(run);
    };
    for (const void* fn : ctx->launched) {
      const char* raw = hipKernelNameRefByPtr(fn, ctx->stream);
      std::string name = raw ? raw : "?";
      int st = 0;
      char* dem = raw ? abi::__cxa_demangle(raw, nullptr, nullptr, &st) : nullptr;
      if (dem && st == 0) name = dem;
      std::free(dem);
      size_t depth = 0, cut = std::string::npos;
      for (size_t i = 0; i < name.size(); i++) {  // the parameter list: the last top-level '('
        if (name[i] == '<') depth++;
        else if (name[i] == '>' && depth) depth--;
        else if (name[i] == '(' && depth == 0) cut = i;
      }
      if (cut != std::string::npos) name.resize(cut);
      if (name.compare(0, 5, "void ") == 0) name.erase(0, 5);
      for (size_t p; (p = name.find("prism::")) != std::string::npos;) name.erase(p, 7);
      if (name == prev) {
        run++;
      } else {
        flush();
        prev = name;
        run = 1;
      }
    }
    flush();
    ctx->kernels = out;
  }
  return ctx->kernels.c_str();
}

// Host payloads go through the pinned ring (stage_h2d); device payloads
// are copied device-to-device.  GI weights are regrouped on the device
// from a split-block copy (the context's upload buffer for host payloads).
// `async`: return once the copies are enqueued on the context stream.
static prism_hip_weight* upload_impl(prism_hip_ctx* ctx, const void* src, bool src_dev, size_t bytes, uint32_t dm,
                                     uint32_t dn, uint32_t bits, uint32_t layout, bool async = false) {
  if (!ctx) return nullptr;
  if (!src) {
    fail(ctx, PRISM_HIP_ERR_NULL, "payload is NULL");
    return nullptr;
  }
  if (check_shape(ctx, dm, dn, bits, layout, bytes) != PRISM_HIP_OK) return nullptr;
  DeviceGuard g(ctx->device);
  auto* w = new prism_hip_weight;
  w->ctx = ctx;
  w->device = ctx->device;
  w->dim_m = dm;
  w->dim_n = dn;
  w->bits = bits;
  w->layout = layout;
  w->bytes = bytes;
  w->gi = gi_rows(ctx, dm, dn, bits);
  auto bail = [&](int rc) -> prism_hip_weight* {
    (void)rc;
    if (w->chunk) {
      (void)hipStreamSynchronize(ctx->stream);
      chunk_release(w->chunk);
    }
    delete w;
    return nullptr;
  };
  int rc = weight_alloc(ctx, w->gi ? prism::gi_bytes(w->gi, dm, dn, bits) : bytes, &w->d, &w->chunk);
  if (rc != PRISM_HIP_OK) return bail(rc);
  hipError_t e = hipSuccess;
  const void* s = src;
  if (!w->gi) {
    if (src_dev) {
      e = hipMemcpyAsync(w->d, src, bytes, hipMemcpyDeviceToDevice, ctx->stream);
      if (e != hipSuccess) rc = fail(ctx, PRISM_HIP_ERR_DEVICE, "weight upload: %s", hipGetErrorString(e));
    } else {
      rc = stage_h2d(ctx, w->d, src, bytes);
    }
  } else {
    if (!src_dev) {
      rc = ensure_upload_stage(ctx, bytes);
      if (rc == PRISM_HIP_OK) rc = stage_h2d(ctx, ctx->d_upload, src, bytes);
      s = ctx->d_upload;
    }
    if (rc == PRISM_HIP_OK) {
      const size_t pieces = prism::gi_bytes(w->gi, dm, dn, bits) / 16;
      const unsigned grid = (unsigned)std::min<size_t>((pieces + 255) / 256, 16384);
      PRISM_LAUNCH(prism::k_gi_pack, dim3(grid), dim3(256), 0, ctx->stream,
                         reinterpret_cast<const uint8_t*>(s), w->d, dm, dn, w->gi, bits);
      e = hipGetLastError();
      if (e != hipSuccess) rc = fail(ctx, PRISM_HIP_ERR_DEVICE, "GI pack: %s", hipGetErrorString(e));
    }
  }
  if (rc == PRISM_HIP_OK && (!async || src_dev)) {
    e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) rc = fail(ctx, PRISM_HIP_ERR_DEVICE, "weight upload (%zu bytes): %s", bytes, hipGetErrorString(e));
  }
  if (rc != PRISM_HIP_OK) return bail(rc);
  ctx->weights.insert(w);
  ctx->err.clear();
  return w;
}

prism_hip_weight* prism_hip_weight_upload(prism_hip_ctx* ctx, const uint8_t* payload, size_t bytes, uint32_t dim_m,
                                          uint32_t dim_n, uint32_t bits, uint32_t layout) {
  return upload_impl(ctx, payload, false, bytes, dim_m, dim_n, bits, layout);
}

prism_hip_weight* prism_hip_weight_upload_async(prism_hip_ctx* ctx, const uint8_t* payload, size_t bytes,
                                                uint32_t dim_m, uint32_t dim_n, uint32_t bits, uint32_t layout) {
  return upload_impl(ctx, payload, false, bytes, dim_m, dim_n, bits, layout, true);
}

prism_hip_weight* prism_hip_weight_upload_dev(prism_hip_ctx* ctx, const void* d_payload, size_t bytes, uint32_t dim_m,
                                              uint32_t dim_n, uint32_t bits, uint32_t layout) {
  return upload_impl(ctx, d_payload, true, bytes, dim_m, dim_n, bits, layout);
}

int prism_hip_ctx_synchronize(prism_hip_ctx* ctx) {
  if (!ctx) return PRISM_HIP_ERR_NULL;
  DeviceGuard g(ctx->device);
  HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
  ctx->err.clear();
  return PRISM_HIP_OK;
}

void prism_hip_weight_free(prism_hip_weight* w) {
  if (!w) return;
  DeviceGuard g(w->device);
  if (w->ctx) w->ctx->weights.erase(w);
  chunk_release(w->chunk);  // the chunk's last weight frees it (hipFree waits for work still using it)
  delete w;
}

int prism_hip_weight_info(const prism_hip_weight* w, uint32_t* dim_m, uint32_t* dim_n, uint32_t* bits, size_t* bytes) {
  if (!w) return PRISM_HIP_ERR_NULL;
  if (dim_m) *dim_m = w->dim_m;
  if (dim_n) *dim_n = w->dim_n;
  if (bits) *bits = w->bits;
  if (bytes) *bytes = w->bytes;
  return PRISM_HIP_OK;
}

// ---- GEMV
int prism_hip_gemv_dev(prism_hip_ctx* ctx, const prism_hip_weight* w, const void* d_x, uint32_t batch, void* d_y,
                       void* stream) {
  if (!ctx) return PRISM_HIP_ERR_NULL;
  int rc = check_weight(ctx, w);
  if (rc) return rc;
  if (!d_x || !d_y) return fail(ctx, PRISM_HIP_ERR_NULL, "x or y is NULL");
  if (batch == 0) return PRISM_HIP_OK;
  DeviceGuard g(ctx->device);
  LaunchLog log(ctx);
  rc = launch_gemv(ctx, w, nullptr, d_x, batch, d_y, pick_stream(ctx, stream));
  if (rc == PRISM_HIP_OK) ctx->err.clear();
  return rc;
}

int prism_hip_gemv(prism_hip_ctx* ctx, const prism_hip_weight* w, const uint16_t* x, uint32_t batch, uint16_t* y) {
  if (!ctx) return PRISM_HIP_ERR_NULL;
  int rc = check_weight(ctx, w);
  if (rc) return rc;
  if (!x || !y) return fail(ctx, PRISM_HIP_ERR_NULL, "x or y is NULL");
  if (batch == 0) return PRISM_HIP_OK;
  DeviceGuard g(ctx->device);
  LaunchLog log(ctx);
  const size_t xb = (size_t)batch * w->dim_n * 2, yb = (size_t)batch * w->dim_m * 2;
  HostCall call(ctx, xb, yb);
  if ((rc = call.begin(x))) return rc;
  if ((rc = launch_gemv(ctx, w, nullptr, call.d_in(), batch, call.d_out(), ctx->stream))) return rc;
  if ((rc = call.finish(y, yb))) return rc;
  ctx->err.clear();
  return PRISM_HIP_OK;
}

// ---- gate_up + SwiGLU
static int check_pair(prism_hip_ctx* ctx, const prism_hip_weight* g, const prism_hip_weight* u) {
  int rc = check_weight(ctx, g);
  if (rc) return rc;
  if ((rc = check_weight(ctx, u))) return rc;
  if (g->dim_m != u->dim_m || g->dim_n != u->dim_n || g->bits != u->bits)
    return fail(ctx, PRISM_HIP_ERR_MISMATCH, "gate %ux%u/%u-bit and up %ux%u/%u-bit differ", g->dim_m, g->dim_n,
                g->bits, u->dim_m, u->dim_n, u->bits);
  return PRISM_HIP_OK;
}

int prism_hip_gateup_swiglu_dev(prism_hip_ctx* ctx, const prism_hip_weight* gate, const prism_hip_weight* up,
                                const void* d_x, void* d_y, void* stream) {
  if (!ctx) return PRISM_HIP_ERR_NULL;
  int rc = check_pair(ctx, gate, up);
  if (rc) return rc;
  if (!d_x || !d_y) return fail(ctx, PRISM_HIP_ERR_NULL, "x or y is NULL");
  DeviceGuard g(ctx->device);
  LaunchLog log(ctx);
  rc = launch_gemv(ctx, gate, up, d_x, 1, d_y, pick_stream(ctx, stream));
  if (rc == PRISM_HIP_OK) ctx->err.clear();
  return rc;
}

int prism_hip_gateup_swiglu(prism_hip_ctx* ctx, const prism_hip_weight* gate, const prism_hip_weight* up,
                            const uint16_t* x, uint16_t* y) {
  if (!ctx) return PRISM_HIP_ERR_NULL;
  int rc = check_pair(ctx, gate, up);
  if (rc) return rc;
  if (!x || !y) return fail(ctx, PRISM_HIP_ERR_NULL, "x or y is NULL");
  DeviceGuard g(ctx->device);
  LaunchLog log(ctx);
  const size_t xb = (size_t)gate->dim_n * 2, yb = (size_t)gate->dim_m * 2;
  HostCall call(ctx, xb, yb);
  if ((rc = call.begin(x))) return rc;
  if ((rc = launch_gemv(ctx, gate, up, call.d_in(), 1, call.d_out(), ctx->stream))) return rc;
  if ((rc = call.finish(y, yb))) return rc;
  ctx->err.clear();
  return PRISM_HIP_OK;
}

// ---- gate and up without the activation: two outputs
int prism_hip_gate_up_dev(prism_hip_ctx* ctx, const prism_hip_weight* gate, const prism_hip_weight* up,
                          const void* d_x, void* d_gate_out, void* d_up_out, void* stream) {
  if (!ctx) return PRISM_HIP_ERR_NULL;
  int rc = check_pair(ctx, gate, up);
  if (rc) return rc;
  if (!d_x || !d_gate_out || !d_up_out) return fail(ctx, PRISM_HIP_ERR_NULL, "x or an output is NULL");
  DeviceGuard g(ctx->device);
  LaunchLog log(ctx);
  rc = launch_gemv(ctx, gate, up, d_x, 1, d_gate_out, pick_stream(ctx, stream), d_up_out);
  if (rc == PRISM_HIP_OK) ctx->err.clear();
  return rc;
}

int prism_hip_gate_up(prism_hip_ctx* ctx, const prism_hip_weight* gate, const prism_hip_weight* up, const uint16_t* x,
                      uint16_t* gate_out, uint16_t* up_out) {
  if (!ctx) return PRISM_HIP_ERR_NULL;
  int rc = check_pair(ctx, gate, up);
  if (rc) return rc;
  if (!x || !gate_out || !up_out) return fail(ctx, PRISM_HIP_ERR_NULL, "x or an output is NULL");
  DeviceGuard g(ctx->device);
  LaunchLog log(ctx);
  const size_t xb = (size_t)gate->dim_n * 2, yb = (size_t)gate->dim_m * 2;
  const size_t y2off = (yb + 255) & ~(size_t)255;
  HostCall call(ctx, xb, y2off + yb);
  if ((rc = call.begin(x))) return rc;
  if ((rc = launch_gemv(ctx, gate, up, call.d_in(), 1, call.d_out(), ctx->stream, call.d_out() + y2off))) return rc;
  if ((rc = call.finish(gate_out, yb, up_out, y2off))) return rc;
  ctx->err.clear();
  return PRISM_HIP_OK;
}

// ---- GEMM
int prism_hip_gemm_dev(prism_hip_ctx* ctx, const prism_hip_weight* w, const void* d_X, uint32_t M, void* d_Y,
                       void* stream) {
  if (!ctx) return PRISM_HIP_ERR_NULL;
  int rc = check_weight(ctx, w);
  if (rc) return rc;
  if (!d_X || !d_Y) return fail(ctx, PRISM_HIP_ERR_NULL, "X or Y is NULL");
  if (M == 0) return PRISM_HIP_OK;
  DeviceGuard g(ctx->device);
  LaunchLog log(ctx);
  rc = launch_gemm(ctx, w, d_X, M, d_Y, pick_stream(ctx, stream));
  if (rc == PRISM_HIP_OK) ctx->err.clear();
  return rc;
}

int prism_hip_gemm_dev_noalloc(prism_hip_ctx* ctx, const prism_hip_weight* w, const void* d_X, uint32_t M,
                               void* d_Y, void* stream) {
  if (!ctx) return PRISM_HIP_ERR_NULL;
  int rc = check_weight(ctx, w);
  if (rc) return rc;
  if (!d_X || !d_Y) return fail(ctx, PRISM_HIP_ERR_NULL, "X or Y is NULL");
  if (M == 0) return PRISM_HIP_OK;
  DeviceGuard g(ctx->device);
  LaunchLog log(ctx);
  if (!ctx->scratch) {
    const hipError_t e = device_scratch(ctx->device, &ctx->scratch);
    if (e != hipSuccess)
      return fail(ctx, PRISM_HIP_ERR_DEVICE, "hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
  }
  rc = launch_gemm(ctx, w, d_X, M, d_Y, pick_stream(ctx, stream), ctx->scratch);
  if (rc == PRISM_HIP_OK) ctx->err.clear();
  return rc;
}

int prism_hip_gemm(prism_hip_ctx* ctx, const prism_hip_weight* w, const uint16_t* X, uint32_t M, uint16_t* Y) {
  if (!ctx) return PRISM_HIP_ERR_NULL;
  int rc = check_weight(ctx, w);
  if (rc) return rc;
  if (!X || !Y) return fail(ctx, PRISM_HIP_ERR_NULL, "X or Y is NULL");
  if (M == 0) return PRISM_HIP_OK;
  DeviceGuard g(ctx->device);
  LaunchLog log(ctx);
  const size_t xb = (size_t)M * w->dim_n * 2, yb = (size_t)M * w->dim_m * 2;
  HostCall call(ctx, xb, yb);
  if ((rc = call.begin(X))) return rc;
  if ((rc = launch_gemm(ctx, w, call.d_in(), M, call.d_out(), ctx->stream))) return rc;
  if ((rc = call.finish(Y, yb))) return rc;
  ctx->err.clear();
  return PRISM_HIP_OK;
}

// ---- decode
int prism_hip_decode_rows_dev(prism_hip_ctx* ctx, const prism_hip_weight* w, uint32_t row0, uint32_t nrows,
                              void* d_out, void* stream) {
  if (!ctx) return PRISM_HIP_ERR_NULL;
  int rc = check_weight(ctx, w);
  if (rc) return rc;
  if (!d_out) return fail(ctx, PRISM_HIP_ERR_NULL, "out is NULL");
  if (row0 > w->dim_m || nrows > w->dim_m - row0)
    return fail(ctx, PRISM_HIP_ERR_SHAPE, "rows [%u, %u) outside 0..%u", row0, row0 + nrows, w->dim_m);
  DeviceGuard g(ctx->device);
  LaunchLog log(ctx);
  rc = launch_decode(ctx, w, row0, nrows, d_out, pick_stream(ctx, stream));
  if (rc == PRISM_HIP_OK) ctx->err.clear();
  return rc;
}

int prism_hip_lut_embed(prism_hip_ctx* ctx, const prism_hip_weight* w, uint32_t token, uint16_t* out) {
  if (!ctx) return PRISM_HIP_ERR_NULL;
  int rc = check_weight(ctx, w);
  if (rc) return rc;
  if (!out) return fail(ctx, PRISM_HIP_ERR_NULL, "out is NULL");
  if (token >= w->dim_m) {  // evaluator.rs:182-184: out-of-range token -> zeros
    std::memset(out, 0, (size_t)w->dim_n * 2);
    ctx->err.clear();
    return PRISM_HIP_OK;
  }
  DeviceGuard g(ctx->device);
  LaunchLog log(ctx);
  const size_t ob = (size_t)w->dim_n * 2;
  HostCall call(ctx, 0, ob);
  if ((rc = call.begin(nullptr))) return rc;
  if ((rc = launch_decode(ctx, w, token, 1, call.d_out(), ctx->stream))) return rc;
  if ((rc = call.finish(out, ob))) return rc;
  ctx->err.clear();
  return PRISM_HIP_OK;
}

// ---- measurement: the read floor
int prism_hip_stream_read_dev(prism_hip_ctx* ctx, const void* d_buf, size_t bytes, void* d_sink, void* stream) {
  if (!ctx) return PRISM_HIP_ERR_NULL;
  if (!d_buf || !d_sink) return fail(ctx, PRISM_HIP_ERR_NULL, "buffer or sink is NULL");
  if (bytes == 0) return PRISM_HIP_OK;
  if (bytes >= (1ull << 31)) return fail(ctx, PRISM_HIP_ERR_SIZE, "%zu bytes: at most 2 GiB - 1 per call", bytes);
  DeviceGuard g(ctx->device);
  LaunchLog log(ctx);
  const unsigned grid = (unsigned)((bytes + prism::kStreamBytesPerBlock - 1) / prism::kStreamBytesPerBlock);
  PRISM_LAUNCH(prism::k_stream_read, dim3(grid), dim3(64), 0, pick_stream(ctx, stream),
                     reinterpret_cast<const uint8_t*>(d_buf), (uint32_t)bytes, reinterpret_cast<uint32_t*>(d_sink));
  HIP_TRY(ctx, hipGetLastError());
  ctx->err.clear();
  return PRISM_HIP_OK;
}

// ---- measurement: one dependent launch, and the matrix cores' rate
int prism_hip_launch_empty_dev(prism_hip_ctx* ctx, void* stream) {
  if (!ctx) return PRISM_HIP_ERR_NULL;
  DeviceGuard g(ctx->device);
  LaunchLog log(ctx);
  PRISM_LAUNCH(prism::k_launch_empty, dim3(1), dim3(64), 0, pick_stream(ctx, stream));
  HIP_TRY(ctx, hipGetLastError());
  ctx->err.clear();
  return PRISM_HIP_OK;
}

int prism_hip_mfma_probe_dev(prism_hip_ctx* ctx, uint32_t groups, uint32_t iters, void* d_sink, void* stream) {
  if (!ctx) return PRISM_HIP_ERR_NULL;
  if (!d_sink) return fail(ctx, PRISM_HIP_ERR_NULL, "sink is NULL");
  if (groups == 0 || groups > 65536) return fail(ctx, PRISM_HIP_ERR_SIZE, "%u workgroups: 1..65536", groups);
  DeviceGuard g(ctx->device);
  LaunchLog log(ctx);
  PRISM_LAUNCH(prism::k_mfma_probe, dim3(groups), dim3(256), 0, pick_stream(ctx, stream), iters,
               reinterpret_cast<float*>(d_sink));
  HIP_TRY(ctx, hipGetLastError());
  ctx->err.clear();
  return PRISM_HIP_OK;
}

int prism_hip_issue_probe_dev(prism_hip_ctx* ctx, uint32_t op, uint32_t groups, uint32_t waves_per_simd,
                              uint32_t iters, void* d_sink, void* stream) {
  if (!ctx) return PRISM_HIP_ERR_NULL;
  if (!d_sink) return fail(ctx, PRISM_HIP_ERR_NULL, "sink is NULL");
  if (op > 3) return fail(ctx, PRISM_HIP_ERR_SHAPE, "instruction kind %u: 0..3", op);
  if (waves_per_simd != 1 && waves_per_simd != 2 && waves_per_simd != 4)
    return fail(ctx, PRISM_HIP_ERR_SHAPE, "%u waves per SIMD: 1, 2 or 4", waves_per_simd);
  if (groups == 0 || groups > 65536) return fail(ctx, PRISM_HIP_ERR_SIZE, "%u workgroups: 1..65536", groups);
  DeviceGuard g(ctx->device);
  LaunchLog log(ctx);
  const dim3 block(256 * waves_per_simd);
  hipStream_t st = pick_stream(ctx, stream);
  float* sink = reinterpret_cast<float*>(d_sink);
  switch (op) {
    case 0: PRISM_LAUNCH(prism::k_issue_probe<0>, dim3(groups), block, 0, st, iters, sink); break;
    case 1: PRISM_LAUNCH(prism::k_issue_probe<1>, dim3(groups), block, 0, st, iters, sink); break;
    case 2: PRISM_LAUNCH(prism::k_issue_probe<2>, dim3(groups), block, 0, st, iters, sink); break;
    default: PRISM_LAUNCH(prism::k_issue_probe<3>, dim3(groups), block, 0, st, iters, sink); break;
  }
  HIP_TRY(ctx, hipGetLastError());
  ctx->err.clear();
  return PRISM_HIP_OK;
}

}  // extern "C"

// GPU-resident decode step (prism_hip_model_*).

// ---- palette compiler
size_t prism_hip_palettize_bytes(uint32_t out_dim, uint32_t in_dim) {
  return (size_t)out_dim * 32 + (size_t)out_dim * ((in_dim + 1) / 2);
}

static int check_palettize(prism_hip_ctx* ctx, uint32_t k, const float* seeds, uint32_t nseeds,
                           prism::PaletteSeeds* ps) {
  if (k == 0 || k > (uint32_t)prism::kPaletteMaxK)
    return fail(ctx, PRISM_HIP_ERR_SHAPE, "palette size k=%u outside 1..%d (4-bit indices)", k, prism::kPaletteMaxK);
  *ps = prism::PaletteSeeds{};
  if (seeds) {
    if (nseeds == 0)  // the reference would index centroids[-1]
      return fail(ctx, PRISM_HIP_ERR_SHAPE, "seeds given with nseeds = 0");
    ps->n = std::min<uint32_t>(nseeds, prism::kPaletteMaxK);
    std::memcpy(ps->v, seeds, ps->n * sizeof(float));
  }
  return PRISM_HIP_OK;
}

// Rows run one wave each.  When a row's arrays fit the workgroup's LDS they
// live there; longer rows keep them in a stream-ordered workspace of at most
// kWsBytes per launch.
static int launch_palettize(prism_hip_ctx* ctx, const float* d_w, uint32_t out_dim, uint32_t in_dim, uint32_t k,
                            uint32_t max_iter, const prism::PaletteSeeds& seeds, uint8_t* d_payload,
                            hipStream_t st) {
  constexpr uint32_t kMaxGrid = 1u << 20;
  constexpr size_t kWsBytes = (size_t)256 << 20;
  uint8_t* lut = d_payload;
  uint8_t* idx = d_payload + (size_t)out_dim * 32;
  // as many rows a workgroup (4, 2, 1) as fit its LDS; longer rows in a
  // workspace, a wave each
  const size_t stat = 4 * (2 * prism::kPaletteMaxK + 1) * 4;
  for (uint32_t R = 4; in_dim && R; R /= 2) {
    const size_t lds = prism::palette_rows_bytes(R, in_dim);
    if (lds + stat > ctx->lds_max) continue;
    const bool full = k >= (uint32_t)prism::kPaletteMaxK && in_dim >= (uint32_t)prism::kPaletteMaxK;
    const void* fn;
#define PRISM_PAL(R_)                                                                \
  (full ? reinterpret_cast<const void*>(&prism::k_palettize_rows<R_, true>)          \
        : reinterpret_cast<const void*>(&prism::k_palettize_rows<R_, false>))
    fn = R == 4 ? PRISM_PAL(4) : R == 2 ? PRISM_PAL(2) : PRISM_PAL(1);
#undef PRISM_PAL
    for (uint32_t r0 = 0; r0 < out_dim; r0 += kMaxGrid * R) {
      uint32_t rows = out_dim;
      prism::PaletteSeeds sd = seeds;
      void* args[] = {&d_w, &in_dim, &k, &max_iter, &sd, &r0, &rows, &lut, &idx};
      const uint32_t grid = (std::min(kMaxGrid * R, out_dim - r0) + R - 1) / R;
      HIP_TRY(ctx, launch_fn(fn, dim3(grid), dim3(64 * R), args, lds, st));
    }
    return PRISM_HIP_OK;
  }
  const size_t row = prism::palette_row_bytes(in_dim);
  const uint32_t chunk =
      row ? (uint32_t)std::min<size_t>(kMaxGrid, std::max<size_t>(1, kWsBytes / row)) : kMaxGrid;
  void* ws = nullptr;  // (empty rows, in_dim 0, need none)
  if (row) HIP_TRY(ctx, hipMallocAsync(&ws, (size_t)std::min(chunk, out_dim) * row, st));
  for (uint32_t r0 = 0; r0 < out_dim; r0 += chunk) {
    const uint32_t rows = std::min(chunk, out_dim - r0);
    PRISM_LAUNCH(prism::k_palettize, dim3(rows), dim3(64), 0, st, d_w, in_dim, k, max_iter, seeds, r0,
                 reinterpret_cast<float*>(ws), lut, idx);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
      if (ws) (void)hipFreeAsync(ws, st);
      return fail(ctx, PRISM_HIP_ERR_DEVICE, "k_palettize launch failed: %s", hipGetErrorString(e));
    }
  }
  if (ws) HIP_TRY(ctx, hipFreeAsync(ws, st));
  return PRISM_HIP_OK;
}

int prism_hip_palettize(prism_hip_ctx* ctx, const float* w, uint32_t out_dim, uint32_t in_dim, uint32_t k,
                        uint32_t max_iter, const float* seeds, uint32_t nseeds, uint8_t* payload) {
  if (!ctx) return PRISM_HIP_ERR_NULL;
  prism::PaletteSeeds ps;
  int rc = check_palettize(ctx, k, seeds, nseeds, &ps);
  if (rc) return rc;
  if (out_dim == 0) return PRISM_HIP_OK;
  if (!payload || (!w && in_dim)) return fail(ctx, PRISM_HIP_ERR_NULL, "weights or payload is NULL");
  DeviceGuard g(ctx->device);
  LaunchLog log(ctx);
  const size_t wb = (size_t)out_dim * in_dim * 4, pb = prism_hip_palettize_bytes(out_dim, in_dim);
  const size_t poff = (wb + 255) & ~(size_t)255;
  if ((rc = ensure_stage(ctx, poff + pb))) return rc;
  uint8_t* st = reinterpret_cast<uint8_t*>(ctx->d_stage);
  if (wb) HIP_TRY(ctx, hipMemcpyAsync(st, w, wb, hipMemcpyHostToDevice, ctx->stream));
  if ((rc = launch_palettize(ctx, reinterpret_cast<const float*>(st), out_dim, in_dim, k, max_iter, ps, st + poff,
                             ctx->stream)))
    return rc;
  HIP_TRY(ctx, hipMemcpyAsync(payload, st + poff, pb, hipMemcpyDeviceToHost, ctx->stream));
  HIP_TRY(ctx, hipStreamSynchronize(ctx->stream));
  ctx->err.clear();
  return PRISM_HIP_OK;
}

int prism_hip_palettize_dev(prism_hip_ctx* ctx, const void* d_w, uint32_t out_dim, uint32_t in_dim, uint32_t k,
                            uint32_t max_iter, const float* seeds, uint32_t nseeds, void* d_payload, void* stream) {
  if (!ctx) return PRISM_HIP_ERR_NULL;
  prism::PaletteSeeds ps;
  int rc = check_palettize(ctx, k, seeds, nseeds, &ps);
  if (rc) return rc;
  if (out_dim == 0) return PRISM_HIP_OK;
  if (!d_payload || (!d_w && in_dim)) return fail(ctx, PRISM_HIP_ERR_NULL, "weights or payload is NULL");
  DeviceGuard g(ctx->device);
  LaunchLog log(ctx);
  rc = launch_palettize(ctx, reinterpret_cast<const float*>(d_w), out_dim, in_dim, k, max_iter, ps,
                        reinterpret_cast<uint8_t*>(d_payload), pick_stream(ctx, stream));
  if (rc == PRISM_HIP_OK) ctx->err.clear();
  return rc;
}

#include "model_step.hpp"
