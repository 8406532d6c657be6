// Host runtime: diagnostics, allocation, per-device tables and the host-only
// angle utilities of the C ABI.
#include "runtime.hpp"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <mutex>
#include <vector>

namespace gx {

namespace {
thread_local std::string g_last_error;
std::atomic<int> g_fail_alloc_after{0};
std::atomic<int> g_oom_tries{0};

struct DeviceTables {
  float2* tw = nullptr;
};
std::mutex g_tables_mu;
std::vector<DeviceTables> g_tables;
}  // namespace

int fail(int status, const std::string& msg) {
  g_last_error = msg;
  return status;
}

int ok() { return GTOMX_OK; }

int hip_fail(hipError_t e, const char* what) {
  std::string m = std::string(what) + ": " + hipGetErrorName(e) + " (" + hipGetErrorString(e) + ")";
  if (e == hipErrorOutOfMemory || e == hipErrorMemoryAllocation)
    return fail(GTOMX_ERR_OUT_OF_MEMORY, m);
  return fail(GTOMX_ERR_DEVICE, m);
}

namespace {

// The fault-injection hook of one allocation.
int alloc_hook() {
  int n = g_fail_alloc_after.load();
  if (n > 0) {
    if (n == 1) {
      g_fail_alloc_after.store(0);
      return fail(GTOMX_ERR_OUT_OF_MEMORY, "device allocation failed (injected)");
    }
    g_fail_alloc_after.store(n - 1);
  }
  return GTOMX_OK;
}

// The scratch blocks kept between calls. Allocating per call cost more than the
// transforms (4 images of 4096^2, R2C + C2R: 9.2 to 15 ms with hipMallocAsync
// and hipMalloc, 1.2 ms of kernels), and passes queued without a wait grew the
// runtime's own pool. Each block carries the event of its last use, which the
// next taker's stream waits for, so a block is never written while an earlier
// user still reads it, whatever became of that user's stream. Unused blocks hold
// at most SCRATCH_CAP bytes per device: whenever a block is given back or a new one
// made, the least recently used beyond that go back to the runtime, and those not
// taken for SCRATCH_IDLE takes with them. All of them go when an allocation of this
// library fails, and when the program asks (gtomx_scratch_release). Blocks come
// from hipMallocAsync and go back through hipFreeAsync, which other threads' stream
// captures allow.
struct ScratchBlock {
  void* p = nullptr;  // nullptr: a free slot
  size_t bytes = 0;
  int dev = 0;
  hipEvent_t ev = nullptr;
  hipStream_t last = nullptr;
  bool busy = false;
  unsigned long long tick = 0;
};
constexpr size_t SCRATCH_CAP = 4ull << 30;
constexpr unsigned long long SCRATCH_IDLE = 256;
struct ScratchPool {
  std::mutex mu;
  std::vector<ScratchBlock> blocks;
  unsigned long long tick = 0;
};
// never destroyed: the HIP runtime may be gone before static destructors run
ScratchPool& scratch_pool() {
  static ScratchPool* pool = new ScratchPool();
  return *pool;
}

// With the pool locked: frees unused blocks of device dev, in the order of
// stream s, until at most `keep` bytes stay; idle ones go in any case.
void trim_locked(ScratchPool& pool, int dev, size_t keep, hipStream_t s) {
  auto drop = [&](ScratchBlock& b) {
    if (hipStreamWaitEvent(s, b.ev, 0) != hipSuccess || hipFreeAsync(b.p, s) != hipSuccess) (void)hipGetLastError();
    (void)hipEventDestroy(b.ev);
    b = ScratchBlock{};
  };
  size_t held = 0;
  for (auto& b : pool.blocks)
    if (b.p && b.dev == dev && !b.busy) {
      if (pool.tick - b.tick > SCRATCH_IDLE)
        drop(b);
      else
        held += b.bytes;
    }
  while (held > keep) {
    ScratchBlock* oldest = nullptr;
    for (auto& b : pool.blocks)
      if (b.p && b.dev == dev && !b.busy && (!oldest || b.tick < oldest->tick)) oldest = &b;
    if (!oldest) break;
    held -= oldest->bytes;
    drop(*oldest);
  }
}

// Gives every unused block of the current device back (an allocation has failed, or the program asks).
hipError_t trim_all() {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  ScratchPool& pool = scratch_pool();
  std::lock_guard<std::mutex> lk(pool.mu);
  trim_locked(pool, dev, 0, nullptr);
  return hipStreamSynchronize(nullptr);  // the runtime's pool releases what is free at a wait
}

// One try of an allocation (on stream s: hipMallocAsync), or the out-of-memory hook's answer.
hipError_t try_malloc(void** p, size_t bytes, bool ordered, hipStream_t s) {
  int n = g_oom_tries.load();
  while (n > 0)
    if (g_oom_tries.compare_exchange_weak(n, n - 1)) return hipErrorOutOfMemory;
  return ordered ? hipMallocAsync(p, bytes, s) : hipMalloc(p, bytes);
}

// hipMallocAsync, once more without the kept scratch if it fails. The pool is locked.
hipError_t malloc_async_or_trim(ScratchPool& pool, int dev, void** p, size_t bytes, hipStream_t s) {
  hipError_t e = try_malloc(p, bytes, true, s);
  if (e == hipSuccess) return e;
  (void)hipGetLastError();
  trim_locked(pool, dev, 0, s);
  (void)hipStreamSynchronize(s);
  e = try_malloc(p, bytes, true, s);
  if (e != hipSuccess) (void)hipGetLastError();
  return e;
}

}  // namespace

hipError_t malloc_or_trim(void** p, size_t bytes) {
  hipError_t e = try_malloc(p, bytes, false, nullptr);
  if (e != hipErrorOutOfMemory) return e;
  (void)hipGetLastError();
  (void)trim_all();
  return try_malloc(p, bytes, false, nullptr);
}

int dev_alloc(void** p, size_t bytes) {
  *p = nullptr;
  GX_TRY(alloc_hook());
  if (bytes == 0) bytes = 16;
  hipError_t e = malloc_or_trim(p, bytes);
  if (e != hipSuccess) {
    *p = nullptr;
    (void)hipGetLastError();
    return hip_fail(e, "hipMalloc");
  }
  return GTOMX_OK;
}

void dev_free(void* p) {
  if (p) (void)hipFree(p);
}

int StreamScratch::take(size_t n, hipStream_t st, bool counted) {
  s = st;
  if (counted) GX_TRY(alloc_hook());
  const size_t bytes = n * sizeof(float2);
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  const bool plain = hipStreamIsCapturing(st, &cap) == hipSuccess && cap == hipStreamCaptureStatusNone;
  if (!plain) (void)hipGetLastError();
  void* q = nullptr;
  if (!plain) {  // a capture records the allocation as a node of its graph
    GX_HIP(hipMallocAsync(&q, bytes, st));
    p = static_cast<float2*>(q);
    return GTOMX_OK;
  }
  int dev = 0;
  GX_HIP(hipGetDevice(&dev));
  ScratchPool& pool = scratch_pool();
  std::lock_guard<std::mutex> lk(pool.mu);
  if (bytes > SCRATCH_CAP) {  // not kept
    hipError_t e = malloc_async_or_trim(pool, dev, &q, bytes, st);
    if (e != hipSuccess) return hip_fail(e, "hipMallocAsync(scratch)");
    p = static_cast<float2*>(q);
    return GTOMX_OK;
  }
  ++pool.tick;
  // the smallest unused block of this stream that fits without wasting more than half of it; another
  // stream's only where the cap leaves no room for a block of this one's own (it would wait for the other)
  int best = -1, other = -1;
  size_t held = 0;
  for (int i = 0; i < (int)pool.blocks.size(); ++i) {
    const ScratchBlock& b = pool.blocks[i];
    if (!b.p || b.dev != dev || b.busy) continue;
    held += b.bytes;
    if (b.bytes < bytes || b.bytes > 2 * bytes + (1u << 20)) continue;
    int& pick = b.last == st ? best : other;
    if (pick < 0 || b.bytes < pool.blocks[pick].bytes) pick = i;
  }
  if (best < 0 && held + bytes > SCRATCH_CAP) best = other;
  if (best >= 0) {
    hipError_t e = hipStreamWaitEvent(st, pool.blocks[best].ev, 0);
    if (e != hipSuccess) return hip_fail(e, "hipStreamWaitEvent(FFT scratch)");
  } else {
    trim_locked(pool, dev, SCRATCH_CAP - bytes, st);
    ScratchBlock b;
    b.bytes = (std::max<size_t>(bytes, 1) + 0xffff) & ~(size_t)0xffff;
    b.dev = dev;
    hipError_t e = malloc_async_or_trim(pool, dev, &b.p, b.bytes, st);
    if (e != hipSuccess) return hip_fail(e, "hipMallocAsync(scratch)");
    e = hipEventCreateWithFlags(&b.ev, hipEventDisableTiming);
    if (e != hipSuccess) {
      (void)hipFreeAsync(b.p, st);
      return hip_fail(e, "hipEventCreate(FFT scratch)");
    }
    for (best = 0; best < (int)pool.blocks.size() && pool.blocks[best].p; ++best) {
    }
    if (best == (int)pool.blocks.size()) pool.blocks.emplace_back();
    pool.blocks[best] = b;
  }
  ScratchBlock& b = pool.blocks[best];
  b.busy = true;
  b.tick = pool.tick;
  p = static_cast<float2*>(b.p);
  block = best;
  return GTOMX_OK;
}

StreamScratch::~StreamScratch() {
  if (!p) return;
  if (block < 0) {
    (void)hipFreeAsync(p, s);
    return;
  }
  ScratchPool& pool = scratch_pool();
  std::lock_guard<std::mutex> lk(pool.mu);
  ScratchBlock& b = pool.blocks[block];
  const int dev = b.dev;
  b.busy = false;
  b.last = s;
  if (hipEventRecord(b.ev, s) != hipSuccess) {  // the end of its use is not known: not kept
    (void)hipGetLastError();
    (void)hipFreeAsync(b.p, s);
    (void)hipEventDestroy(b.ev);
    b = ScratchBlock{};
  }
  // a call with several blocks may have taken more than the cap together
  trim_locked(pool, dev, SCRATCH_CAP, s);
}

int twiddles(const float2** table) {
  int dev = 0;
  GX_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lk(g_tables_mu);
  if ((int)g_tables.size() <= dev) g_tables.resize(dev + 1);
  if (!g_tables[dev].tw) {
    const int total = TW_LEN_HOST + TW3_LEN_HOST;
    std::vector<float2> h(total);
    const long double twopi = 6.283185307179586476925286766559005768L;
    for (int m = 0; m < TW_LEN_HOST; ++m) {
      long double a = -twopi * (long double)m / (long double)TW_LEN_HOST;
      h[m] = make_float2((float)std::cos(a), (float)std::sin(a));
    }
    for (int m = 0; m < TW3_LEN_HOST; ++m) {
      long double a = -twopi * (long double)m / (long double)TW3_LEN_HOST;
      h[TW_LEN_HOST + m] = make_float2((float)std::cos(a), (float)std::sin(a));
    }
    void* d = nullptr;
    hipError_t e = malloc_or_trim(&d, sizeof(float2) * total);
    if (e != hipSuccess) return hip_fail(e, "hipMalloc(twiddles)");
    e = hipMemcpy(d, h.data(), sizeof(float2) * total, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
      (void)hipFree(d);
      return hip_fail(e, "hipMemcpy(twiddles)");
    }
    g_tables[dev].tw = static_cast<float2*>(d);
  }
  *table = g_tables[dev].tw;
  return GTOMX_OK;
}

int check_fft_dims(int ndims, gtomx_int3 d) {
  if (ndims < 1 || ndims > 3) return fail(GTOMX_ERR_INVALID_ARGUMENT, "ndims must be 1, 2 or 3");
  if (d.x < 1 || d.y < 1 || d.z < 1) return fail(GTOMX_ERR_INVALID_ARGUMENT, "dims must be positive");
  int want = 3 - (d.z == 1) - (d.z == 1 && d.y == 1);
  if (ndims != want)
    return fail(GTOMX_ERR_INVALID_ARGUMENT, "ndims does not match dims (trailing extents must be 1)");
  if (!fft_len_ok_any(d.x))
    return fail(GTOMX_ERR_UNSUPPORTED, "dims.x must be 2^a in [8, 4096] or 3*2^a in [12, 3072]");
  if (d.y != 1 && !fft_len_ok_any(d.y))
    return fail(GTOMX_ERR_UNSUPPORTED, "dims.y must be 1, 2^a in [8, 4096] or 3*2^a in [12, 3072]");
  if (d.z != 1 && !fft_len_ok_any(d.z))
    return fail(GTOMX_ERR_UNSUPPORTED, "dims.z must be 1, 2^a in [8, 4096] or 3*2^a in [12, 3072]");
  return GTOMX_OK;
}

int check_fft_dims_any(int ndims, gtomx_int3 d) {
  if (ndims < 1 || ndims > 3) return fail(GTOMX_ERR_INVALID_ARGUMENT, "ndims must be 1, 2 or 3");
  if (d.x < 1 || d.y < 1 || d.z < 1) return fail(GTOMX_ERR_INVALID_ARGUMENT, "dims must be positive");
  int want = 3 - (d.z == 1) - (d.z == 1 && d.y == 1);
  if (ndims != want)
    return fail(GTOMX_ERR_INVALID_ARGUMENT, "ndims does not match dims (trailing extents must be 1)");
  auto ok = [](int n) { return fft_len_ok_any(n) || n <= 2048; };
  if (!ok(d.x) || !ok(d.y) || !ok(d.z))
    return fail(GTOMX_ERR_UNSUPPORTED,
                "extents must be at most 2048, or 2^a up to 4096, or 3*2^a up to 3072");
  return GTOMX_OK;
}

}  // namespace gx

using namespace gx;

extern "C" {

const char* gtomx_version(void) { return "gtomx 0.1 (gfx950)"; }

const char* gtomx_status_string(int s) {
  switch (s) {
    case GTOMX_OK: return "ok";
    case GTOMX_ERR_INVALID_ARGUMENT: return "invalid argument";
    case GTOMX_ERR_UNSUPPORTED: return "unsupported";
    case GTOMX_ERR_OUT_OF_MEMORY: return "out of memory";
    case GTOMX_ERR_DEVICE: return "device error";
    case GTOMX_ERR_INTERNAL: return "internal error";
    default: return "unknown status";
  }
}

const char* gtomx_last_error(void) { return g_last_error.c_str(); }

int gtomx_scratch_release(void) {
  GX_HIP(trim_all());
  return GTOMX_OK;
}

int gtomx_scratch_held(size_t* bytes) {
  if (!bytes) return fail(GTOMX_ERR_INVALID_ARGUMENT, "bytes is NULL");
  *bytes = 0;
  int dev = 0;
  GX_HIP(hipGetDevice(&dev));
  ScratchPool& pool = scratch_pool();
  std::lock_guard<std::mutex> lk(pool.mu);
  for (const auto& b : pool.blocks)
    if (b.p && b.dev == dev && !b.busy) *bytes += b.bytes;
  return GTOMX_OK;
}

void gtomx_debug_fail_alloc_after(int n) { g_fail_alloc_after.store(n < 0 ? 0 : n); }
void gtomx_debug_out_of_memory(int n) { g_oom_tries.store(n < 0 ? 0 : n); }

// GetEqualAngularSpacing (src/Helpers/AngularSpacing.cu:46-67) with float32
// loop counters so that the orientation count and order match the reference.
int gtomx_equal_angular_spacing(float phimin, float phimax, float thetamin, float thetamax,
                                float psimin, float psimax, float increment,
                                gtomx_float3* h_angles, int capacity, int* count) {
  if (!count) return fail(GTOMX_ERR_INVALID_ARGUMENT, "count is NULL");
  if (!(increment > 0.0f)) return fail(GTOMX_ERR_INVALID_ARGUMENT, "increment must be positive");
  if (capacity < 0 || (capacity > 0 && !h_angles))
    return fail(GTOMX_ERR_INVALID_ARGUMENT, "bad output buffer");
  const float PI2f = 6.283185307179586476925286766559f;
  int n = 0;
  for (float tilt = thetamin; tilt <= thetamax + 1e-5f; tilt += increment) {
    int rot_nstep = tilt > 0 ? (int)std::ceil(PI2f * std::sin(tilt) / increment) : 1;
    float rot_sam = PI2f / (float)rot_nstep;
    for (float rot = phimin; rot <= phimax - rot_sam + 1e-5f; rot += rot_sam)
      for (float psi = psimin; psi <= psimax - increment + 1e-5f; psi += increment) {
        if (n < capacity) h_angles[n] = gtomx_float3{rot, tilt, psi};
        ++n;
      }
  }
  *count = n;
  return GTOMX_OK;
}

int gtomx_fibonacci_angles(int ndirs, int npsi, gtomx_float3* h_angles) {
  if (ndirs <= 0 || npsi <= 0 || !h_angles)
    return fail(GTOMX_ERR_INVALID_ARGUMENT, "ndirs and npsi must be positive, h_angles non-NULL");
  const double pi = 3.14159265358979323846;
  const double golden = pi * (3.0 - std::sqrt(5.0));
  for (int i = 0; i < ndirs; ++i) {
    double z = 1.0 - (2.0 * i + 1.0) / ndirs;
    double tilt = std::acos(std::max(-1.0, std::min(1.0, z)));
    double rot = std::fmod(golden * i, 2.0 * pi);
    for (int j = 0; j < npsi; ++j) {
      double psi = 2.0 * pi * j / npsi;
      h_angles[(size_t)i * npsi + j] = gtomx_float3{(float)rot, (float)tilt, (float)psi};
    }
  }
  return GTOMX_OK;
}

// transpose(Matrix3Euler(a)) * s, row-major (src/Relion/Project.cu:16,
// src/Helpers/Euler.cu:39-68), evaluated in double.
int gtomx_projector_matrices(const gtomx_float3* h_angles, unsigned n, float oversample,
                             float* h_matrices) {
  if ((n > 0 && (!h_angles || !h_matrices)))
    return fail(GTOMX_ERR_INVALID_ARGUMENT, "NULL angle or matrix buffer");
  for (unsigned i = 0; i < n; ++i) {
    double ca = std::cos((double)h_angles[i].x), sa = std::sin((double)h_angles[i].x);
    double cb = std::cos((double)h_angles[i].y), sb = std::sin((double)h_angles[i].y);
    double cg = std::cos((double)h_angles[i].z), sg = std::sin((double)h_angles[i].z);
    double cc = cb * ca, cs = cb * sa, sc = sb * ca, ss = sb * sa;
    double A[9] = {cg * cc - sg * sa,  cg * cs + sg * ca,  -cg * sb,
                   -sg * cc - cg * sa, -sg * cs + cg * ca, sg * sb,
                   sc,                 ss,                 cb};
    double s = oversample;
    float* M = h_matrices + 9 * (size_t)i;
    for (int r = 0; r < 3; ++r)
      for (int c = 0; c < 3; ++c) M[3 * r + c] = (float)(s * A[3 * c + r]);
  }
  return GTOMX_OK;
}

}  // extern "C"
