// Context, error reporting and device memory helpers of the C-ABI.
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <unordered_map>
#include <vector>

#include "zr_internal.h"

// Scratch memory of the allocation-free entry point (zr_softmax_forward_static): every GPU the library runs on holds
// its own copy of this array until the process ends.  In host code the array's name is only a handle for
// hipGetSymbolAddress; the device address differs per GPU and is looked up once per device, with that device
// current (static_scratch_address), and only that address is ever passed to kernels.
static __device__ __align__(256) unsigned char scratch[ZR_STATIC_SCRATCH_BYTES];
static void* g_static_scratch[64];
static std::mutex g_static_scratch_mu;

// Device address of `scratch` on the current device (which must be `device`).
static int static_scratch_address(int device, void** out) {
  std::lock_guard<std::mutex> lock(g_static_scratch_mu);
  if (device < 0 || device >= 64) return zr_set_error(ZR_EINVAL, "device %d has no static scratch slot", device);
  if (!g_static_scratch[device]) {
    void* ptr = nullptr;
    ZR_HIP(hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch)));
    if (!ptr) return zr_set_error(ZR_EHIP, "hipGetSymbolAddress returned a null address for the static scratch array");
    g_static_scratch[device] = ptr;
  }
  *out = g_static_scratch[device];
  return ZR_OK;
}

static thread_local char g_err[512] = "";

// live contexts per device in this process (zr_live_contexts)
static std::atomic<int> g_live[64];

int zr_live_contexts(int device) { return (device >= 0 && device < 64) ? g_live[device].load() : 2; }

int zr_set_error(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

int zr_bind_device(zr_ctx* ctx) {
  ZR_CHECK_ARG(ctx != nullptr, "null context");
  ZR_HIP(hipSetDevice(ctx->device));
  return ZR_OK;
}

// ---- kept device memory
//
// hipMalloc and hipFree take 10 to 300 us, and hipFree waits for the whole device: a training step that packs its layers' new weights
// (destroy, create) drained the queue at every layer, a translation paid for its 100 MB and its handles each time (decode object of one sentence:
// created 340 and closed in 70 us, of 16 sentences 530 and 380).  So a context keeps what is given back, up to 32 blocks and
// 512 MiB, none larger than half of that, oldest out first, and only what zr_dev_alloc made.
// A block of a handle is reused without waiting for the work that is queued on it, which is sound as long as all of that, and all
// that comes, is on the context's own stream: nothing is kept where a caller's stream has ever been set or another context is alive.
// What callers hold themselves (zr_malloc) may be in use on any stream of theirs, so zr_free waits for the device as hipFree
// did, and zr_malloc for this stream where it hands out a handle's block.
// A second context on the device, and every allocation that fails, has the blocks of all contexts there given back first, and an
// allocation that fails all the same its own context's scratch buffers.
constexpr size_t kKeptTotal = (size_t)512 << 20, kKeptLargest = (size_t)256 << 20;

struct Block {
  size_t bytes;
  int device;
};
struct Blocks {
  std::mutex mu;                             // of everything here and of every context's kept blocks
  std::unordered_map<void*, Block> handed;   // made by zr_dev_alloc and not given back
  std::vector<zr_ctx*> contexts;             // of the process
};
static Blocks& blocks() {
  static Blocks* b = new Blocks();  // (handles may be destroyed behind static objects)
  return *b;
}

static void* take_kept(zr_ctx* ctx, int i) {
  void* p = ctx->kept[i].p;
  ctx->kept_bytes -= ctx->kept[i].bytes;
  for (--ctx->n_kept; i < ctx->n_kept; ++i) ctx->kept[i] = ctx->kept[i + 1];
  return p;
}
static void free_blocks(const std::vector<void*>& list) {
  for (void* p : list) (void)hipFree(p);  // (waits for the device)
}

int zr_give_back_kept(int device, zr_ctx* only) {
  std::vector<void*> list;
  {
    std::lock_guard<std::mutex> lock(blocks().mu);
    for (zr_ctx* c : blocks().contexts)
      while (c->device == device && (!only || c == only) && c->n_kept) list.push_back(take_kept(c, c->n_kept - 1));
  }
  free_blocks(list);
  return (int)list.size();
}

// On the list, and counted, before anything of the context is allocated: from here on nobody keeps blocks on its device.
static void register_context(zr_ctx* ctx) {
  {
    std::lock_guard<std::mutex> lock(blocks().mu);
    blocks().contexts.push_back(ctx);
    if (ctx->device < 64) g_live[ctx->device].fetch_add(1);
  }
  if (zr_live_contexts(ctx->device) > 1) (void)zr_give_back_kept(ctx->device, nullptr);
}
static void unregister_context(zr_ctx* ctx) {
  std::lock_guard<std::mutex> lock(blocks().mu);
  auto& all = blocks().contexts;
  all.erase(std::remove(all.begin(), all.end(), ctx), all.end());
  if (ctx->device < 64) g_live[ctx->device].fetch_sub(1);
}

// hipMalloc, if need be once more behind the kept blocks.
static void* hip_malloc(zr_ctx* ctx, size_t bytes) {
  void* p = nullptr;
  if (hipMalloc(&p, bytes) == hipSuccess) return p;
  (void)hipGetLastError();
  if (!zr_give_back_kept(ctx->device, nullptr)) return nullptr;
  if (hipMalloc(&p, bytes) == hipSuccess) return p;
  (void)hipGetLastError();
  return nullptr;
}

// Gives the context's scratch buffers back, which stay as large as the largest call so far made them (a backward sweep's hand-over memory: 315 MB for four
// layers of 512, 128 columns, 60 steps).  Only where no graph can hold their addresses; nothing lies in them from call to call.
static bool give_back_scratch(zr_ctx* ctx) {
  if (ctx->foreign_stream || (!ctx->d_scratch && !ctx->d_scratch2) || hipStreamSynchronize(ctx->stream) != hipSuccess) return false;
  if (ctx->d_scratch) (void)hipFree(ctx->d_scratch);
  if (ctx->d_scratch2) (void)hipFree(ctx->d_scratch2);
  ctx->d_scratch = ctx->d_scratch2 = nullptr;
  ctx->scratch_bytes = ctx->scratch2_bytes = 0;
  return true;
}

// Called at the entry points, before any scratch of theirs.
void* zr_dev_alloc(zr_ctx* ctx, size_t bytes, bool any_stream) {
  void* p = nullptr;
  Block block = {bytes, ctx->device};
  bool idle = false;
  {
    std::lock_guard<std::mutex> lock(blocks().mu);
    int best = -1;
    for (int i = 0; i < ctx->n_kept; ++i)
      if (ctx->kept[i].bytes >= bytes && ctx->kept[i].bytes - bytes <= bytes / 8 + 4096 && (best < 0 || ctx->kept[i].bytes < ctx->kept[best].bytes))
        best = i;
    if (best >= 0) {
      block.bytes = ctx->kept[best].bytes;
      idle = ctx->kept[best].idle;
      p = take_kept(ctx, best);
    }
  }
  if (p && any_stream && !idle && hipStreamSynchronize(ctx->own_stream) != hipSuccess) {
    (void)hipFree(p);
    (void)hipGetLastError();
    p = nullptr;
  }
  if (!p) {
    p = hip_malloc(ctx, bytes);
    if (!p && give_back_scratch(ctx)) p = hip_malloc(ctx, bytes);
    block.bytes = bytes;
  }
  if (p) {
    std::lock_guard<std::mutex> lock(blocks().mu);
    blocks().handed[p] = block;
  }
  return p;
}

// Waits for all work on the device, as hipFree does; hipDeviceSynchronize would end a capture that goes on meanwhile on another stream, which
// hipFree does not (relaxed mode).
static bool wait_for_device() {
  void* p = nullptr;
  if (hipMalloc(&p, 4) == hipSuccess && hipFree(p) == hipSuccess) return true;
  (void)hipGetLastError();
  return false;
}

int zr_dev_free(zr_ctx* ctx, void* p, bool callers) {
  if (!p) return ZR_OK;
  auto may_keep = [&](const Block& b) {
    return ctx->keep_memory && !ctx->foreign_stream && zr_live_contexts(ctx->device) == 1 && b.device == ctx->device && b.bytes <= kKeptLargest;
  };
  bool keep = false;
  {
    std::lock_guard<std::mutex> lock(blocks().mu);
    const auto it = blocks().handed.find(p);
    if (it != blocks().handed.end()) {
      keep = may_keep(it->second);
    } else {
      for (zr_ctx* c : blocks().contexts)
        for (int i = 0; i < c->n_kept; ++i)
          if (c->kept[i].p == p) return zr_set_error(ZR_EHIP, "device memory %p is freed twice", p);
    }
  }
  if (callers || !keep) ZR_HIP(hipStreamSynchronize(ctx->stream));
  if (callers && keep) keep = wait_for_device();
  std::vector<void*> list;
  {
    std::lock_guard<std::mutex> lock(blocks().mu);
    const auto it = blocks().handed.find(p);
    if (it != blocks().handed.end()) {
      const Block b = it->second;
      blocks().handed.erase(it);
      if (keep && may_keep(b)) {
        while (ctx->n_kept == ZR_MAX_KEPT || (ctx->n_kept && ctx->kept_bytes + b.bytes > kKeptTotal)) list.push_back(take_kept(ctx, 0));
        ctx->kept[ctx->n_kept++] = {p, b.bytes, callers};
        ctx->kept_bytes += b.bytes;
        p = nullptr;
      }
    }
  }
  free_blocks(list);
  if (p) ZR_HIP(hipFree(p));
  return ZR_OK;
}

int zr_dev_release(void* p) {
  if (!p) return ZR_OK;
  {
    std::lock_guard<std::mutex> lock(blocks().mu);
    blocks().handed.erase(p);
  }
  ZR_HIP(hipFree(p));
  return ZR_OK;
}

int zr_ctx_pinned(zr_ctx* ctx, size_t bytes, void** host, void** dev) {
  if (ctx->pinned_bytes < bytes) {
    ZR_HIP(hipStreamSynchronize(ctx->stream));
    if (ctx->h_pinned) ZR_HIP(hipHostFree(ctx->h_pinned));
    ctx->h_pinned = nullptr;
    ctx->pinned_bytes = 0;
    const size_t want = bytes + bytes / 4 + 4096;
    if (hipHostMalloc(&ctx->h_pinned, want, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      ctx->h_pinned = nullptr;
      return zr_set_error(ZR_ENOMEM, "allocation of %zu bytes of page-locked host memory failed", want);
    }
    ctx->pinned_bytes = want;
  }
  *host = ctx->h_pinned;
  ZR_HIP(hipHostGetDevicePointer(dev, ctx->h_pinned, 0));
  return ZR_OK;
}

int zr_ctx_scratch(zr_ctx* ctx, int slot, size_t bytes, void** out) {
  if (ctx->fixed_scratch) {
    if (bytes > ctx->fixed_bytes[slot])
      return zr_set_error(ZR_EINVAL, "this call needs %zu bytes of scratch memory (%s) but the allocation-free entry "
                          "point has %zu: use the allocating entry point for this size", bytes,
                          slot == 0 ? "re-laid-out activations" : "partial column statistics", ctx->fixed_bytes[slot]);
    *out = ctx->d_fixed[slot];
    return ZR_OK;
  }
  void** buf = slot == 0 ? &ctx->d_scratch : &ctx->d_scratch2;
  size_t* cap = slot == 0 ? &ctx->scratch_bytes : &ctx->scratch2_bytes;
  if (*cap < bytes) {
    // the old buffer may still be in use by queued kernels: drain the stream before releasing it
    ZR_HIP(hipStreamSynchronize(ctx->stream));
    if (*buf) ZR_HIP(hipFree(*buf));
    *buf = nullptr;
    *cap = 0;
    size_t want = bytes + bytes / 4;
    *buf = hip_malloc(ctx, want);
    if (!*buf) {
      return zr_set_error(ZR_ENOMEM, "scratch allocation of %zu bytes failed", want);
    }
    *cap = want;
  }
  *out = *buf;
  return ZR_OK;
}

int zr_ctx_scratch_if_room(zr_ctx* ctx, int slot, size_t bytes, void** out) {
  if (ctx->sweep_scratch_kib && bytes > (size_t)ctx->sweep_scratch_kib << 10)
    return zr_set_error(ZR_ENOMEM, "%zu bytes of scratch memory are more than ZR_OPT_LSTM_SWEEP_SCRATCH", bytes);
  const size_t cap = slot == 0 ? ctx->scratch_bytes : ctx->scratch2_bytes;
  size_t free_bytes = 0, total = 0, kept = 0;
  if (cap < bytes) {
    std::lock_guard<std::mutex> lock(blocks().mu);
    kept = ctx->kept_bytes;
  }
  if (cap < bytes && hipMemGetInfo(&free_bytes, &total) == hipSuccess && free_bytes + kept + cap < bytes + bytes / 4)
    return zr_set_error(ZR_ENOMEM, "no room for %zu bytes of scratch memory", bytes);
  (void)hipGetLastError();
  return zr_ctx_scratch(ctx, slot, bytes, out);
}

extern "C" {

const char* zr_last_error(void) { return g_err; }

const char* zr_version(void) { return "gfx950 hip zoph_rnn_amd 0.1"; }

int zr_ctx_create(int device, zr_ctx** out) {
  ZR_CHECK_ARG(out != nullptr, "zr_ctx_create: out is null");
  *out = nullptr;
  int ndev = 0;
  ZR_HIP(hipGetDeviceCount(&ndev));
  ZR_CHECK_ARG(device >= 0 && device < ndev, "zr_ctx_create: device %d not in [0,%d)", device, ndev);
  ZR_HIP(hipSetDevice(device));
  zr_ctx* c = new zr_ctx();
  memset(c, 0, sizeof(*c));
  c->device = device;
  c->keep_memory = 1;
  register_context(c);
  hipError_t e = hipStreamCreate(&c->own_stream);  // default priority
  if (e != hipSuccess) {
    unregister_context(c);
    delete c;
    return zr_set_error(ZR_EHIP, "hipStreamCreate failed: %s", hipGetErrorString(e));
  }
  c->stream = c->own_stream;
  const size_t flag_bytes = (32 + ZR_MAX_COUNTERS + ZR_MAX_STEP_FLAGS) * sizeof(int), slot_bytes = 2 * kSgdSlots * sizeof(unsigned long long);
  e = hipMalloc((void**)&c->d_flags, flag_bytes + slot_bytes);
  if (e != hipSuccess) {
    (void)hipStreamDestroy(c->own_stream);
    unregister_context(c);
    delete c;
    return zr_set_error(ZR_ENOMEM, "flag allocation failed: %s", hipGetErrorString(e));
  }
  (void)hipMemset(c->d_flags, 0, flag_bytes + slot_bytes);
  c->d_sgd_slots = (unsigned long long*)((char*)c->d_flags + flag_bytes);
  c->d_counters = c->d_flags + 32;  // (a line apart from the flags)
  c->d_step_flags = c->d_counters + ZR_MAX_COUNTERS;
  {
    const int rc = static_scratch_address(device, &c->d_static_scratch);
    if (rc) {
      (void)hipFree(c->d_flags);
      (void)hipStreamDestroy(c->own_stream);
      unregister_context(c);
      delete c;
      return rc;
    }
  }
  e = hipDeviceGetAttribute(&c->cu_count, hipDeviceAttributeMultiprocessorCount, device);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    c->cu_count = 256;
  }
  c->lstm_fused = 1;
  // ZR_LSTM_SWEEP in the environment presets ZR_OPT_LSTM_SWEEP for every context of the process (0 to 3): lets a
  // whole program, e.g. a test run, be put on one path or the other without touching its code
  if (const char* e = getenv("ZR_LSTM_SWEEP")) {
    const int v = atoi(e);
    if (v >= 0 && v <= 3) c->lstm_sweep = v;
  }
  // the same for ZR_OPT_LSTM_SWEEP_SPIN and ZR_OPT_LSTM_STEP_WAIT_EXTRA (tests of a whole program's give-up handling)
  if (const char* e = getenv("ZR_LSTM_SWEEP_SPIN")) {
    const int v = atoi(e);
    if (v >= 0) c->sweep_spin = v;
  }
  if (const char* e = getenv("ZR_LSTM_STEP_WAIT_EXTRA")) {
    const int v = atoi(e);
    if (v >= 0 && v <= 1024) c->step_wait_extra = v;
  }
  // ZR_LSTM_STACK_HELPERS=0 keeps the decoder step on its two-workgroups-per-tile schedules (timing comparisons)
  c->stack_helpers = 1;
  if (const char* e = getenv("ZR_LSTM_STACK_HELPERS")) c->stack_helpers = atoi(e) != 0 ? 1 : 0;
  *out = c;
  return ZR_OK;
}

int zr_ctx_destroy(zr_ctx* ctx) {
  if (!ctx) return ZR_OK;
  (void)hipSetDevice(ctx->device);
  (void)hipStreamSynchronize(ctx->stream);
  (void)zr_give_back_kept(ctx->device, ctx);
  if (ctx->h_pinned) (void)hipHostFree(ctx->h_pinned);
  if (ctx->d_scratch) (void)hipFree(ctx->d_scratch);
  if (ctx->d_scratch2) (void)hipFree(ctx->d_scratch2);
  if (ctx->d_flags) (void)hipFree(ctx->d_flags);
  for (int i = 0; i < ZR_MAX_PACKED_D; ++i)
    (void)zr_dev_release(ctx->packed_d[i].d_pack);
  if (ctx->ev_start) (void)hipEventDestroy(ctx->ev_start);
  if (ctx->ev_stop) (void)hipEventDestroy(ctx->ev_stop);
  (void)hipStreamDestroy(ctx->own_stream);
  unregister_context(ctx);
  delete ctx;
  return ZR_OK;
}

int zr_ctx_sync(zr_ctx* ctx) {
  int rc = zr_bind_device(ctx);
  if (rc) return rc;
  ZR_HIP(hipStreamSynchronize(ctx->stream));
  ZR_LAUNCH_CHECK("queued work");
  int flags[4] = {0, 0, 0, 0};
  ZR_HIP(hipMemcpy(flags, ctx->d_flags, sizeof(flags), hipMemcpyDeviceToHost));
  if (flags[2] != 0) {
    ZR_HIP(hipMemset(ctx->d_flags, 0, sizeof(flags)));
    return zr_set_error(ZR_EHIP, "a whole-sweep LSTM launch gave up waiting for another workgroup: the outputs of "
                        "zr_lstm_stack_forward since the last zr_ctx_sync are incomplete (ZR_OPT_LSTM_SWEEP = 1 "
                        "selects one launch per diagonal)");
  }
  if (flags[0] != 0 || flags[1] != 0) {
    ZR_HIP(hipMemset(ctx->d_flags, 0, sizeof(flags)));
    return zr_set_error(ZR_EDATA, "%d token id(s) outside [0, vocab) and %d source position(s) outside the "
                        "attention table were clamped", flags[0], flags[1]);
  }
  return ZR_OK;
}

int zr_ctx_query(zr_ctx* ctx, int what, int* h_value) {
  ZR_CHECK_ARG(ctx != nullptr, "null context");
  ZR_CHECK_ARG(h_value != nullptr, "zr_ctx_query: h_value is null");
  switch (what) {
    case ZR_QUERY_LSTM_STACK_PATH:
      *h_value = ctx->last_stack_path;
      return ZR_OK;
    case ZR_QUERY_LSTM_SWEEP_KERNEL:
      *h_value = ctx->last_sweep_kernel;
      return ZR_OK;
    case ZR_QUERY_LSTM_BACKWARD_PATH:
      *h_value = ctx->last_backward_path;
      return ZR_OK;
    case ZR_QUERY_SCRATCH_KIB:
      *h_value = (int)((ctx->scratch_bytes + ctx->scratch2_bytes + 1023) / 1024);
      return ZR_OK;
    case ZR_QUERY_ATTN_PATH:
      *h_value = ctx->last_attn_path;
      return ZR_OK;
    case ZR_QUERY_LSTM_SWEEP_ABANDONED: {
      int rc = zr_bind_device(ctx);
      if (rc) return rc;
      ZR_HIP(hipStreamSynchronize(ctx->stream));
      int flag = 0;
      ZR_HIP(hipMemcpy(&flag, ctx->d_flags + 2, sizeof(int), hipMemcpyDeviceToHost));
      // Everything queued behind the abandoned launch ran on its NaN outputs: the word ids picked from them and the
      // window positions derived from them are out of range, so the data flags are up as well.  They say nothing about
      // the caller's data; all four go down together, and the caller's re-run starts from a clean slate.
      if (flag != 0) ZR_HIP(hipMemset(ctx->d_flags, 0, 4 * sizeof(int)));
      *h_value = flag != 0 ? 1 : 0;
      return ZR_OK;
    }
    case ZR_QUERY_WAITS_REPAIRED: {
      int rc = zr_bind_device(ctx);
      if (rc) return rc;
      ZR_HIP(hipStreamSynchronize(ctx->stream));
      int gave_up[2] = {0, 0};
      ZR_HIP(hipMemcpy(gave_up, ctx->d_flags + 4, sizeof(gave_up), hipMemcpyDeviceToHost));
      *h_value = (ctx->sgd_epoch && gave_up[1] == ctx->sgd_epoch ? ZR_REPAIRED_SGD_UPDATE : 0) |
                 (ctx->back_epoch && gave_up[0] == ctx->back_epoch ? ZR_REPAIRED_LSTM_BACKWARD : 0);
      return ZR_OK;
    }
    default:
      return zr_set_error(ZR_EINVAL, "zr_ctx_query: unknown item %d", what);
  }
}

int zr_ctx_set_stream(zr_ctx* ctx, void* hip_stream) {
  ZR_CHECK_ARG(ctx != nullptr, "null context");
  if (hip_stream && !ctx->foreign_stream) {
    ctx->foreign_stream = 1;
    const int rc = zr_bind_device(ctx);
    if (rc) return rc;
    (void)zr_give_back_kept(ctx->device, ctx);
  }
  ctx->stream = hip_stream ? (hipStream_t)hip_stream : ctx->own_stream;
  return ZR_OK;
}

int zr_ctx_set_option(zr_ctx* ctx, int option, int value) {
  ZR_CHECK_ARG(ctx != nullptr, "null context");
  switch (option) {
    case ZR_OPT_LSTM_FUSED_EPILOGUE:
      ctx->lstm_fused = value ? 1 : 0;
      return ZR_OK;
    case ZR_OPT_LSTM_TN:
      ZR_CHECK_ARG(value == 0 || value == 1 || value == 2 || value == 4, "ZR_OPT_LSTM_TN must be 0, 1, 2 or 4");
      ctx->lstm_tn = value;
      return ZR_OK;
    case ZR_OPT_LSTM_KSPLIT:
      ZR_CHECK_ARG(value == 0 || value == 4 || value == 8, "ZR_OPT_LSTM_KSPLIT must be 0, 4 or 8");
      ctx->lstm_ksplit = value;
      return ZR_OK;
    case ZR_OPT_LSTM_KERNEL:
      ZR_CHECK_ARG(value >= 0 && value <= 3, "ZR_OPT_LSTM_KERNEL must be 0, 1, 2 or 3");
      ctx->lstm_kernel = value;
      return ZR_OK;
    case ZR_OPT_LSTM_KPARTS:
      ZR_CHECK_ARG(value >= 0 && value <= 16, "ZR_OPT_LSTM_KPARTS must be in [0, 16]");
      ctx->lstm_kparts = value;
      return ZR_OK;
    case ZR_OPT_LSTM_SWEEP:
      ZR_CHECK_ARG(value >= 0 && value <= 3, "ZR_OPT_LSTM_SWEEP must be 0, 1, 2 or 3");
      ctx->lstm_sweep = value;
      return ZR_OK;
    case ZR_OPT_LSTM_SWEEP_SPIN:
      ZR_CHECK_ARG(value >= 0, "ZR_OPT_LSTM_SWEEP_SPIN must not be negative");
      ctx->sweep_spin = value;
      return ZR_OK;
    case ZR_OPT_LSTM_SWEEP_SCRATCH:
      ZR_CHECK_ARG(value >= 0, "ZR_OPT_LSTM_SWEEP_SCRATCH must not be negative");
      ctx->sweep_scratch_kib = value;
      return ZR_OK;
    case ZR_OPT_LSTM_STEP_WAIT_EXTRA:
      ZR_CHECK_ARG(value >= 0 && value <= 1024, "ZR_OPT_LSTM_STEP_WAIT_EXTRA must be in [0, 1024]");
      ctx->step_wait_extra = value;
      return ZR_OK;
    case ZR_OPT_ATTN_SINGLE_LAUNCH:
      ZR_CHECK_ARG(value == 0 || value == 1, "ZR_OPT_ATTN_SINGLE_LAUNCH must be 0 or 1");
      ctx->attn_single = value;
      return ZR_OK;
    case ZR_OPT_KEEP_MEMORY:
      ZR_CHECK_ARG(value == 0 || value == 1, "ZR_OPT_KEEP_MEMORY must be 0 or 1");
      ctx->keep_memory = value;
      if (!value) {
        const int rc = zr_bind_device(ctx);
        if (rc) return rc;
        (void)zr_give_back_kept(ctx->device, ctx);
      }
      return ZR_OK;
    case ZR_OPT_BF16_ACTIVATION_TERMS:
      ZR_CHECK_ARG(value == 1 || value == 2, "ZR_OPT_BF16_ACTIVATION_TERMS must be 1 or 2");
      ctx->bf16_terms = value;
      return ZR_OK;
    case ZR_OPT_GEMM_CFG:
      ZR_CHECK_ARG(value >= 0 && value <= 14, "ZR_OPT_GEMM_CFG out of range");
      ctx->gemm_cfg = value;
      return ZR_OK;
    default:
      return zr_set_error(ZR_EINVAL, "unknown option %d", option);
  }
}

int zr_malloc(zr_ctx* ctx, size_t bytes, void** d_out) {
  int rc = zr_bind_device(ctx);
  if (rc) return rc;
  ZR_CHECK_ARG(d_out != nullptr, "zr_malloc: out is null");
  *d_out = nullptr;
  if (bytes == 0) bytes = 4;
  *d_out = zr_dev_alloc(ctx, bytes, true);
  return *d_out ? ZR_OK : zr_set_error(ZR_ENOMEM, "hipMalloc of %zu bytes failed", bytes);
}

int zr_free(zr_ctx* ctx, void* d_ptr) {
  int rc = zr_bind_device(ctx);
  if (rc) return rc;
  return zr_dev_free(ctx, d_ptr, true);
}

int zr_h2d(zr_ctx* ctx, void* d_dst, const void* h_src, size_t bytes) {
  int rc = zr_bind_device(ctx);
  if (rc) return rc;
  ZR_CHECK_ARG(bytes == 0 || (d_dst && h_src), "zr_h2d: null pointer");
  if (bytes == 0) return ZR_OK;
  // pageable host memory: the runtime stages the copy, and it is ordered after earlier work on the stream
  ZR_HIP(hipMemcpyAsync(d_dst, h_src, bytes, hipMemcpyHostToDevice, ctx->stream));
  ZR_HIP(hipStreamSynchronize(ctx->stream));
  return ZR_OK;
}

int zr_d2h(zr_ctx* ctx, void* h_dst, const void* d_src, size_t bytes) {
  int rc = zr_bind_device(ctx);
  if (rc) return rc;
  ZR_CHECK_ARG(bytes == 0 || (h_dst && d_src), "zr_d2h: null pointer");
  if (bytes == 0) return ZR_OK;
  ZR_HIP(hipMemcpyAsync(h_dst, d_src, bytes, hipMemcpyDeviceToHost, ctx->stream));
  ZR_HIP(hipStreamSynchronize(ctx->stream));
  return ZR_OK;
}

int zr_d2d(zr_ctx* ctx, void* d_dst, const void* d_src, size_t bytes) {
  int rc = zr_bind_device(ctx);
  if (rc) return rc;
  ZR_CHECK_ARG(bytes == 0 || (d_dst && d_src), "zr_d2d: null pointer");
  if (bytes == 0) return ZR_OK;
  ZR_HIP(hipMemcpyAsync(d_dst, d_src, bytes, hipMemcpyDeviceToDevice, ctx->stream));
  return ZR_OK;
}

}  // extern "C"

// Stream timer: two HIP events on the context's stream (the reference wraps phases in host wall-clock Timer
// objects after a device synchronise, src/memory_util.h:87-124).
extern "C" int zr_timer_start(zr_ctx* ctx) {
  int rc = zr_bind_device(ctx);
  if (rc) return rc;
  if (!ctx->ev_start) {
    ZR_HIP(hipEventCreate(&ctx->ev_start));
    ZR_HIP(hipEventCreate(&ctx->ev_stop));
  }
  ZR_HIP(hipEventRecord(ctx->ev_start, ctx->stream));
  return ZR_OK;
}

extern "C" int zr_timer_stop(zr_ctx* ctx, float* h_ms) {
  int rc = zr_bind_device(ctx);
  if (rc) return rc;
  ZR_CHECK_ARG(ctx->ev_start != nullptr && h_ms != nullptr, "zr_timer_stop: no running timer or null output");
  ZR_HIP(hipEventRecord(ctx->ev_stop, ctx->stream));
  ZR_HIP(hipEventSynchronize(ctx->ev_stop));
  ZR_HIP(hipEventElapsedTime(h_ms, ctx->ev_start, ctx->ev_stop));
  return ZR_OK;
}
