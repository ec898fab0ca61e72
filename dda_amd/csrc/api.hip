// Context, error reporting and plain memory helpers of the C ABI.
#include <algorithm>
#include <cstring>
#include <string>

#include "internal.hpp"

namespace dda {

static thread_local std::string g_last_error;

void set_error(const std::string& msg) { g_last_error = msg; }

}  // namespace dda

using namespace dda;

extern "C" const char* dda_last_error(void) { return g_last_error.c_str(); }

// A stream of different particles makes and destroys operators of similar sizes,
// and hipFree of a buffer of some ten megabytes takes 100 us and more (the three
// of a 96 x 72 x 60 box 590 us, allocating them anew 100). Up to kSpareBytes of a
// context's freed buffers wait for its next operators; work on its stream orders
// old and new use. Any allocation of the library that finds the memory short gives
// them back first, those of the other contexts on the device too.
constexpr size_t kSpareBytes = 1ull << 30;
constexpr size_t kSpareCount = 64;  // (the list is searched from end to end)

// The contexts alive, for dev_malloc (locked before a context's spare_mu).
static std::mutex g_ctx_mu;
static std::vector<dda_ctx_s*> g_ctx;

extern "C" dda_status dda_ctx_create(int device, dda_ctx_t* out) {
  if (!out) {
    set_error("dda_ctx_create: null output");
    return DDA_INVALID_ARG;
  }
  *out = nullptr;
  int n = 0;
  DDA_TRY_HIP(hipGetDeviceCount(&n));
  if (device < 0 || device >= n) {
    set_error("dda_ctx_create: no such device");
    return DDA_INVALID_ARG;
  }
  DDA_TRY_HIP(hipSetDevice(device));
  dda_ctx_s* c = new dda_ctx_s();
  c->device = device;
  c->spare_limit = kSpareBytes;
  hipError_t e = hipGetDeviceProperties(&c->prop, device);
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking);
  if (e != hipSuccess) {
    set_error(std::string("dda_ctx_create: ") + hipGetErrorString(e));
    delete c;
    return DDA_HIP_ERROR;
  }
  const dda_status rs = noalloc_scratch_setup(device);
  if (rs != DDA_OK) {
    (void)hipStreamDestroy(c->stream);
    delete c;
    return rs;
  }
  {
    std::lock_guard<std::mutex> lk(g_ctx_mu);
    g_ctx.push_back(c);
  }
  *out = c;
  return DDA_OK;
}

static bool free_spares(dda_ctx_s* c) {
  std::lock_guard<std::mutex> lk(c->spare_mu);
  for (auto& s : c->spare) (void)hipFree(s.ptr);
  const bool any = !c->spare.empty();
  c->spare.clear();
  return any;
}

hipError_t dda::dev_malloc(void** p, size_t bytes) {
  hipError_t e = hipMalloc(p, bytes);
  if (e == hipErrorOutOfMemory) {
    (void)hipGetLastError();
    int device = -1;
    (void)hipGetDevice(&device);
    bool any = false;
    {
      std::lock_guard<std::mutex> lk(g_ctx_mu);
      for (dda_ctx_s* c : g_ctx)
        if (c->device == device) any = free_spares(c) || any;
    }
    if (any) e = hipMalloc(p, bytes);
  }
  if (e != hipSuccess) {
    (void)hipGetLastError();  // (the next launch's check is not to find it)
    *p = nullptr;
  }
  return e;
}

hipError_t dda::ctx_alloc(dda_ctx_s* c, void** p, size_t bytes, Held* h) {
  {
    std::lock_guard<std::mutex> lk(c->spare_mu);
    auto best = c->spare.end();
    for (auto it = c->spare.begin(); it != c->spare.end(); ++it)
      if (it->bytes >= bytes && it->bytes <= bytes + bytes / 2 && (best == c->spare.end() || it->bytes < best->bytes))
        best = it;
    if (best != c->spare.end()) {
      *p = best->ptr;
      *h = {best->bytes, bytes};
      c->surplus += h->got - bytes;
      c->spare.erase(best);
      return hipSuccess;
    }
  }
  *h = {bytes, bytes};
  return dev_malloc(p, bytes);
}

void dda::ctx_free(dda_ctx_s* c, void* p, const Held& h) {
  if (!p) return;
  std::lock_guard<std::mutex> lk(c->spare_mu);
  c->surplus -= h.got - h.want;
  size_t total = c->surplus + h.got;
  for (auto& s : c->spare) total += s.bytes;
  // beyond the limit a buffer that was too large for its use goes before those
  // that fit theirs
  if (h.got + c->surplus > c->spare_limit || (total > c->spare_limit && h.got > h.want)) {
    (void)hipFree(p);
    return;
  }
  c->spare.push_back({p, h.got});
  while (total > c->spare_limit || c->spare.size() > kSpareCount) {
    total -= c->spare.front().bytes;
    (void)hipFree(c->spare.front().ptr);
    c->spare.erase(c->spare.begin());
  }
}

void dda::ctx_limit_spare(dda_ctx_s* c, size_t bytes) {
  std::lock_guard<std::mutex> lk(c->spare_mu);
  c->spare_limit = std::min(bytes, kSpareBytes);
}

extern "C" dda_status dda_ctx_destroy(dda_ctx_t ctx) {
  if (!ctx) return DDA_OK;
  {
    std::lock_guard<std::mutex> lk(g_ctx_mu);
    g_ctx.erase(std::find(g_ctx.begin(), g_ctx.end(), ctx));
  }
  (void)hipStreamSynchronize(ctx->stream);
  free_spares(ctx);
  (void)hipStreamDestroy(ctx->stream);
  delete ctx;
  return DDA_OK;
}

extern "C" dda_status dda_ctx_synchronize(dda_ctx_t ctx) {
  if (!ctx) {
    set_error("dda_ctx_synchronize: null context");
    return DDA_INVALID_ARG;
  }
  DDA_TRY(bind_device(ctx));
  DDA_TRY_HIP(hipStreamSynchronize(ctx->stream));
  return DDA_OK;
}

extern "C" dda_status dda_ctx_info(dda_ctx_t ctx, char* name, size_t name_len, size_t* hbm_bytes, int* cu_count) {
  if (!ctx) {
    set_error("dda_ctx_info: null context");
    return DDA_INVALID_ARG;
  }
  if (name && name_len) {
    std::strncpy(name, ctx->prop.gcnArchName, name_len - 1);
    name[name_len - 1] = 0;
  }
  if (hbm_bytes) *hbm_bytes = ctx->prop.totalGlobalMem;
  if (cu_count) *cu_count = ctx->prop.multiProcessorCount;
  return DDA_OK;
}

extern "C" dda_status dda_malloc(dda_ctx_t ctx, size_t bytes, void** out) {
  if (!ctx || !out) {
    set_error("dda_malloc: null argument");
    return DDA_INVALID_ARG;
  }
  DDA_TRY_HIP(hipSetDevice(ctx->device));
  DDA_TRY_HIP(dev_malloc(out, bytes ? bytes : 1));
  return DDA_OK;
}

extern "C" dda_status dda_free(dda_ctx_t ctx, void* ptr) {
  if (!ctx) {
    set_error("dda_free: null context");
    return DDA_INVALID_ARG;
  }
  DDA_TRY(bind_device(ctx));
  if (ptr) {
    DDA_TRY_HIP(hipStreamSynchronize(ctx->stream));
    DDA_TRY_HIP(hipFree(ptr));
  }
  return DDA_OK;
}

extern "C" dda_status dda_memcpy_h2d(dda_ctx_t ctx, void* dst, const void* src, size_t bytes) {
  if (!ctx || (bytes && (!dst || !src))) {
    set_error("dda_memcpy_h2d: null argument");
    return DDA_INVALID_ARG;
  }
  DDA_TRY(bind_device(ctx));
  DDA_TRY_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->stream));
  DDA_TRY_HIP(hipStreamSynchronize(ctx->stream));
  return DDA_OK;
}

extern "C" dda_status dda_memcpy_d2h(dda_ctx_t ctx, void* dst, const void* src, size_t bytes) {
  if (!ctx || (bytes && (!dst || !src))) {
    set_error("dda_memcpy_d2h: null argument");
    return DDA_INVALID_ARG;
  }
  DDA_TRY(bind_device(ctx));
  DDA_TRY_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
  DDA_TRY_HIP(hipStreamSynchronize(ctx->stream));
  return DDA_OK;
}

extern "C" dda_status dda_memcpy_d2d(dda_ctx_t ctx, void* dst, const void* src, size_t bytes) {
  if (!ctx || (bytes && (!dst || !src))) {
    set_error("dda_memcpy_d2d: null argument");
    return DDA_INVALID_ARG;
  }
  DDA_TRY(bind_device(ctx));
  DDA_TRY_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, ctx->stream));
  DDA_TRY_HIP(hipStreamSynchronize(ctx->stream));
  return DDA_OK;
}
