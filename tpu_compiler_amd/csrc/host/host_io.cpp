#include "host_io.hpp"

#include "host_cpus.hpp"

#include <unistd.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#if !defined(__HIP_DEVICE_COMPILE__) && defined(__x86_64__)
#include <immintrin.h>
#define TPUHIP_X86 1
#endif

namespace tpuhip {

// ---------------------------------------------------------------------------
// float <-> int8.  A float is an integer of the range when it equals its own rounding and lies between the bounds; a
// NaN fails the comparisons, which are all written so that an unordered result counts as bad.
// ---------------------------------------------------------------------------
namespace {

bool to_bytes_plain(const char *src, int8_t *dst, size_t n, float lo, float hi) {
  unsigned bad = 0;
  const float magic = 12582912.0f;   // 1.5 * 2^23: adding and subtracting it rounds below 2^22
  for (size_t i = 0; i < n; ++i) {
    float v;
    memcpy(&v, src + i * sizeof(float), sizeof v);
    bad |= (unsigned)!(v >= lo && v <= hi) | (unsigned)((v + magic) - magic != v);
    const float in_range = v >= lo && v <= hi ? v : 0.0f;
    dst[i] = (int8_t)(int32_t)in_range;
  }
  return bad != 0;
}

#ifdef TPUHIP_X86
__attribute__((target("avx512f,avx512bw"))) bool to_bytes_avx512(const char *src, int8_t *dst, size_t n, float lo, float hi,
                                                                 bool past_caches) {
  const __m512 vlo = _mm512_set1_ps(lo), vhi = _mm512_set1_ps(hi);
  __mmask16 bad = 0;
  size_t i = 0;
  if (past_caches && ((uintptr_t)dst & 63) == 0) {   // whole lines
    for (; i + 64 <= n; i += 64) {
      __m128i q[4];
#pragma GCC unroll 4
      for (int k = 0; k < 4; ++k) {
        const __m512 v = _mm512_loadu_ps(src + (i + 16 * k) * sizeof(float));
        const __m512i r = _mm512_cvtps_epi32(v);
        bad |= _mm512_cmp_ps_mask(v, vlo, _CMP_NGE_UQ) | _mm512_cmp_ps_mask(v, vhi, _CMP_NLE_UQ) |
               _mm512_cmp_ps_mask(v, _mm512_cvtepi32_ps(r), _CMP_NEQ_UQ);
        q[k] = _mm512_cvtepi32_epi8(r);
      }
      __m512i line = _mm512_castsi128_si512(q[0]);
      line = _mm512_inserti32x4(line, q[1], 1);
      line = _mm512_inserti32x4(line, q[2], 2);
      line = _mm512_inserti32x4(line, q[3], 3);
      _mm512_stream_si512((__m512i *)(dst + i), line);
    }
    _mm_sfence();
  }
  for (; i + 16 <= n; i += 16) {
    const __m512 v = _mm512_loadu_ps(src + i * sizeof(float));
    const __m512i q = _mm512_cvtps_epi32(v);   // rounds to nearest even
    bad |= _mm512_cmp_ps_mask(v, vlo, _CMP_NGE_UQ) | _mm512_cmp_ps_mask(v, vhi, _CMP_NLE_UQ) |
           _mm512_cmp_ps_mask(v, _mm512_cvtepi32_ps(q), _CMP_NEQ_UQ);
    _mm_storeu_si128((__m128i *)(dst + i), _mm512_cvtepi32_epi8(q));   // keeps the low byte
  }
  const bool tail = to_bytes_plain(src + i * sizeof(float), dst + i, n - i, lo, hi);
  return bad != 0 || tail;
}

__attribute__((target("avx2"))) bool to_bytes_avx2(const char *src, int8_t *dst, size_t n, float lo, float hi) {
  const __m256 vlo = _mm256_set1_ps(lo), vhi = _mm256_set1_ps(hi);
  const __m256i low = _mm256_set1_epi32(0xff);
  const __m256i order = _mm256_setr_epi32(0, 4, 1, 5, 2, 6, 3, 7);
  __m256 bad = _mm256_setzero_ps();
  size_t i = 0;
  for (; i + 32 <= n; i += 32) {
    __m256i q[4];
    for (int k = 0; k < 4; ++k) {
      const __m256 v = _mm256_loadu_ps((const float *)(src + (i + 8 * k) * sizeof(float)));
      q[k] = _mm256_cvtps_epi32(v);
      bad = _mm256_or_ps(bad, _mm256_or_ps(_mm256_or_ps(_mm256_cmp_ps(v, vlo, _CMP_NGE_UQ), _mm256_cmp_ps(v, vhi, _CMP_NLE_UQ)),
                                           _mm256_cmp_ps(v, _mm256_cvtepi32_ps(q[k]), _CMP_NEQ_UQ)));
      q[k] = _mm256_and_si256(q[k], low);
    }
    const __m256i a = _mm256_packus_epi32(q[0], q[1]), b = _mm256_packus_epi32(q[2], q[3]);
    _mm256_storeu_si256((__m256i *)(dst + i), _mm256_permutevar8x32_epi32(_mm256_packus_epi16(a, b), order));
  }
  const bool tail = to_bytes_plain(src + i * sizeof(float), dst + i, n - i, lo, hi);
  return _mm256_movemask_ps(bad) != 0 || tail;
}

__attribute__((target("avx512f"))) void to_floats_avx512(const int8_t *src, float *dst, size_t n, bool is_unsigned, bool past_caches) {
  size_t i = 0;
  if (past_caches) {
    for (; i < n && ((uintptr_t)(dst + i) & 63); ++i) dst[i] = is_unsigned ? (float)(uint8_t)src[i] : (float)src[i];
    for (; i + 16 <= n; i += 16) {
      const __m128i b = _mm_loadu_si128((const __m128i *)(src + i));
      _mm512_stream_ps(dst + i, _mm512_cvtepi32_ps(is_unsigned ? _mm512_cvtepu8_epi32(b) : _mm512_cvtepi8_epi32(b)));
    }
    _mm_sfence();
  }
  for (; i + 16 <= n; i += 16) {
    const __m128i b = _mm_loadu_si128((const __m128i *)(src + i));
    _mm512_storeu_ps(dst + i, _mm512_cvtepi32_ps(is_unsigned ? _mm512_cvtepu8_epi32(b) : _mm512_cvtepi8_epi32(b)));
  }
  for (; i < n; ++i) dst[i] = is_unsigned ? (float)(uint8_t)src[i] : (float)src[i];
}

__attribute__((target("avx2"))) void to_floats_avx2(const int8_t *src, float *dst, size_t n, bool is_unsigned) {
  size_t i = 0;
  for (; i + 8 <= n; i += 8) {
    const __m128i b = _mm_loadl_epi64((const __m128i *)(src + i));
    _mm256_storeu_ps(dst + i, _mm256_cvtepi32_ps(is_unsigned ? _mm256_cvtepu8_epi32(b) : _mm256_cvtepi8_epi32(b)));
  }
  for (; i < n; ++i) dst[i] = is_unsigned ? (float)(uint8_t)src[i] : (float)src[i];
}

// a copy whose destination's lines the bus reads next: they need not be fetched, nor be taken out of a cache then
__attribute__((target("avx512f"))) void copy_past_caches_avx512(const char *src, int8_t *dst, size_t n) {
  size_t i = 0;
  if (((uintptr_t)dst & 63) == 0) {
    for (; i + 64 <= n; i += 64) _mm512_stream_si512((__m512i *)(dst + i), _mm512_loadu_si512(src + i));
    _mm_sfence();
  }
  memcpy(dst + i, src + i, n - i);
}

int simd_level() {
  static const int level = __builtin_cpu_supports("avx512f") && __builtin_cpu_supports("avx512bw") ? 2
                           : __builtin_cpu_supports("avx2")                                        ? 1
                                                                                                   : 0;
  return level;
}
#endif

}  // namespace

bool floats_to_bytes(const void *values, int8_t *dst, size_t n, bool is_unsigned, bool past_caches) {
  const char *src = (const char *)values;
  const float lo = is_unsigned ? 0.0f : -128.0f, hi = is_unsigned ? 255.0f : 127.0f;
#ifdef TPUHIP_X86
  if (simd_level() == 2) return to_bytes_avx512(src, dst, n, lo, hi, past_caches);
  if (simd_level() == 1) return to_bytes_avx2(src, dst, n, lo, hi);
#endif
  return to_bytes_plain(src, dst, n, lo, hi);
}

namespace {
void copy_past_caches(const char *src, int8_t *dst, size_t n) {
#ifdef TPUHIP_X86
  if (simd_level() == 2) return copy_past_caches_avx512(src, dst, n);
#endif
  memcpy(dst, src, n);
}
}  // namespace

void bytes_to_floats(const int8_t *src, float *dst, size_t n, bool is_unsigned, bool past_caches) {
#ifdef TPUHIP_X86
  if (simd_level() == 2) return to_floats_avx512(src, dst, n, is_unsigned, past_caches);
  if (simd_level() == 1) return to_floats_avx2(src, dst, n, is_unsigned);
#endif
  for (size_t i = 0; i < n; ++i) dst[i] = is_unsigned ? (float)(uint8_t)src[i] : (float)src[i];
}

// ---------------------------------------------------------------------------
// A few threads for the host passes, shared by all contexts of the process and started with the first tensor that is
// worth them.  One caller has them at a time; another one that comes meanwhile does its pieces alone.  The caller takes
// pieces like any worker and waits only for pieces that a worker has taken, so a process without them (a fork's child)
// works the same, only slower.  They end with the process.
// ---------------------------------------------------------------------------
namespace {

struct HostJob {
  std::function<void(size_t)> piece;
  size_t pieces = 0;
  std::atomic<size_t> next{0}, finished{0};
  bool step() {
    const size_t i = next.fetch_add(1, std::memory_order_relaxed);
    if (i >= pieces) return false;
    piece(i);
    finished.fetch_add(1, std::memory_order_release);
    return true;
  }
};

class HostWorkers {
 public:
  static HostWorkers &get() {
    static HostWorkers w;
    return w;
  }

  // offers the job to the workers; false: they are busy with another caller's.  Ends with leave().
  bool enter(const std::shared_ptr<HostJob> &job) {
    if (!users_.try_lock()) return false;
    {
      std::lock_guard<std::mutex> l(mu_);
      if (threads_.empty()) start();
      job_ = job;
      ++serial_;
    }
    wake_.notify_all();
    return true;
  }
  void leave() {
    {
      std::lock_guard<std::mutex> l(mu_);
      job_.reset();
    }
    users_.unlock();
  }

 private:
  HostWorkers() = default;
  ~HostWorkers() {
    if (getpid() != pid_) {   // a fork's child: the threads are the parent's
      for (auto &t : threads_) t.detach();
      return;
    }
    {
      std::lock_guard<std::mutex> l(mu_);
      stop_ = true;
    }
    wake_.notify_all();
    for (auto &t : threads_) t.join();
  }

  void start() {
    pid_ = getpid();
    // seven beside the caller reach the memory bandwidth of a socket's share; never more than the CPUs there are
    const int count = std::max(0, std::min(7, usable_cpus() - 1));
    try {
      for (int i = 0; i < count; ++i) threads_.emplace_back([this] { work(); });
    } catch (const std::system_error &) {   // those there are, or none: the caller does what they do not
    }
  }

  void work() {
    uint64_t seen = 0;
    for (;;) {
      std::shared_ptr<HostJob> job;
      {
        std::unique_lock<std::mutex> l(mu_);
        wake_.wait(l, [&] { return stop_ || (job_ && serial_ != seen); });
        if (stop_) return;
        seen = serial_;
        job = job_;
      }
      while (job->step()) {
      }
    }
  }

  std::mutex users_, mu_;
  std::condition_variable wake_;
  std::shared_ptr<HostJob> job_;
  uint64_t serial_ = 0;
  bool stop_ = false;
  pid_t pid_ = 0;
  std::vector<std::thread> threads_;
};

// the caller's part of a job that needs nothing but its pieces done
void finish_job(HostJob &job) {
  while (job.step()) {
  }
  while (job.finished.load(std::memory_order_acquire) < job.pieces) std::this_thread::yield();
}

constexpr size_t kPiece = 256 << 10;        // bytes of the staging buffer per piece of a host pass
constexpr size_t kAlone = 192 << 10;        // up to here one thread is done before a worker has woken
// Floats on their way to the device: from this many bytes of them on the conversion is worth eight threads.  set_tensor of a
// buffer written just before, alone / on eight: 4 MB 136 / 69 us, 8 MB 268 / 95, 12 MB 407 / 119, 16 MB 531 / 145, 32 MB 1073 /
// 255; with the caller's next write of the buffer, whose lines the other cores then hold, 4 MB 238 / 181, 8 MB 436 / 301, 12 MB
// 638 / 409.  So eight are faster from 2 MB on (142 / 124); the line lies higher because below it they take two to three times
// the CPU time for it.  Bytes are copied by one thread at any size.
constexpr size_t kSharedFloats = 12 << 20;
// From these bytes on the lines of the staging buffer are written past the caches: cached stores fetch the lines to overwrite
// them, and the bus takes them out of the caches again.  Until the transfer has ended, cached / past the caches, source in the
// caches: 1 MB 60 / 60 us, 2 MB 100 / 87, 4 MB 194 / 166, 6 MB 267 / 222, 8 MB 349 / 292, 12 MB 515 / 418, 24 MB 1270 / 800.  The
// gain begins at 2 MB; with the caller's next write of the source it is 2 MB 130 / 133, 4 MB 272 / 246, 6 MB 366 / 337.
constexpr size_t kCachedBytes = 6 << 20;
constexpr size_t kStageMax = 32 << 20;      // the staging buffer grows to this; larger tensors go through it in parts

// the pinned buffer, free to be written: transfers out of it that are still in flight have ended
int stage_ready(tpuhip_ctx *ctx, size_t bytes) {
  TPUHIP_CHECK_HIP(hipSetDevice(ctx->device));
  if (int rc = flush_uploads(ctx)) return rc;   // left by a load that failed
  if (ctx->stage_busy) {
    TPUHIP_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    ctx->stage_busy = false;
  }
  ctx->stage_used = 0;
  bytes = std::min(bytes, kStageMax);
  if (bytes <= ctx->stage_bytes) return TPUHIP_OK;
  size_t want = 64 << 10;
  while (want < bytes) want *= 2;
  if (ctx->stage) TPUHIP_CHECK_HIP(hipHostFree(ctx->stage));
  ctx->stage = nullptr;
  ctx->stage_bytes = 0;
  TPUHIP_CHECK_HIP(hipHostMalloc(&ctx->stage, want, hipHostMallocDefault));
  ctx->stage_bytes = want;
  return TPUHIP_OK;
}

// device memory for a tensor that arrives in more than one piece
int landing_ready(tpuhip_ctx *ctx, size_t bytes) {
  if (bytes <= ctx->landing_bytes) return TPUHIP_OK;
  if (ctx->landing) {
    TPUHIP_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    TPUHIP_CHECK_HIP(hipFree(ctx->landing));
  }
  ctx->landing = nullptr;
  ctx->landing_bytes = 0;
  TPUHIP_CHECK_HIP(hipMalloc(&ctx->landing, bytes + 256));
  ctx->landing_bytes = bytes;
  return TPUHIP_OK;
}

// dwords between pinned and device memory (bus-bound: 57 GB/s from 256 workgroups on, wider accesses no faster); int8
// data may be rounded up to a dword, the staging and landing buffers have the room, floats are whole dwords
__global__ __launch_bounds__(256) void stage_copy_kernel(const uint32_t *src, uint32_t *dst, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) dst[i] = src[i];
}

int stage_copy(tpuhip_ctx *ctx, const void *src, void *dst, size_t bytes) {
  const size_t n = (bytes + 3) / 4;
  const unsigned blocks = (unsigned)std::min<size_t>((n + 255) / 256, 256);
  hipLaunchKernelGGL(stage_copy_kernel, dim3(blocks), dim3(256), 0, ctx->stream, (const uint32_t *)src, (uint32_t *)dst, n);
  TPUHIP_CHECK_HIP(hipGetLastError());
  return TPUHIP_OK;
}

// element -> bytes on the host side and in the staging buffer
size_t host_size(HostKind k) { return k == HostKind::kBytes ? 1 : sizeof(float); }
size_t stage_size(HostKind k) { return k == HostKind::kFloats ? sizeof(float) : 1; }

}  // namespace

// A recorded copy would take, at every replay, whatever lies in the pinned buffer then, and a wait cannot be recorded.
int not_captured(tpuhip_ctx *ctx, const char *what) {
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  TPUHIP_CHECK_HIP(hipStreamIsCapturing(ctx->stream, &capturing));
  TPUHIP_REQUIRE(capturing == hipStreamCaptureStatusNone, "%s: the context's stream is being captured", what);
  return TPUHIP_OK;
}

void parallel_pieces(size_t n, const std::function<void(size_t)> &piece) {
  if (n < 2) {
    if (n) piece(0);
    return;
  }
  auto job = std::make_shared<HostJob>();
  job->piece = piece;
  job->pieces = n;
  const bool shared = HostWorkers::get().enter(job);
  finish_job(*job);
  if (shared) HostWorkers::get().leave();
}

int host_to_device(tpuhip_ctx *ctx, const HostTensor &t, HostKind kind, const void *src, void *dst, bool *bad) {
  *bad = false;
  if (int rc = not_captured(ctx, "a tensor from the host")) return rc;
  const size_t count = (size_t)t.n * t.c * t.h * t.w;
  const size_t per = stage_size(kind), total = count * per;
  if (int rc = stage_ready(ctx, total)) return rc;
  auto pass = [&](size_t first, size_t elements, int8_t *to) {
    const char *from = (const char *)src + first * host_size(kind);
    const bool past_caches = total > (kind == HostKind::kBytes ? kCachedBytes : kAlone);
    if (kind == HostKind::kFloatStored) return floats_to_bytes(from, to, elements, t.is_unsigned, past_caches);
    if (past_caches) copy_past_caches(from, to, elements * per);
    else memcpy(to, from, elements * per);
    return false;
  };
  int8_t *stage = (int8_t *)ctx->stage;
  if (total <= kAlone) {
    *bad = pass(0, count, stage);
    if (*bad) return TPUHIP_OK;
    ctx->stage_busy = true;
    if (kind == HostKind::kFloats) return stage_copy(ctx, stage, dst, total);
    return tpuhip_nchw_to_nhwc_i8(ctx, stage, dst, t.n, t.c, t.h, t.w, t.cs);
  }
  // several pieces: each goes to a landing buffer on the device as soon as it and those before it are there; the tensor
  // itself is written once all of them have passed the check
  void *land = dst;
  if (kind != HostKind::kFloats) {
    if (int rc = landing_ready(ctx, total)) return rc;
    land = ctx->landing;
  }
  std::atomic<bool> any_bad{false};
  for (size_t part = 0; part < total; part += ctx->stage_bytes) {
    const size_t bytes = std::min(total - part, ctx->stage_bytes);
    if (part) TPUHIP_CHECK_HIP(hipStreamSynchronize(ctx->stream));   // the buffer is written anew
    auto job = std::make_shared<HostJob>();
    job->pieces = (bytes + kPiece - 1) / kPiece;
    std::unique_ptr<std::atomic<uint8_t>[]> there(new std::atomic<uint8_t>[job->pieces]);
    for (size_t i = 0; i < job->pieces; ++i) there[i].store(0, std::memory_order_relaxed);
    job->piece = [&, part, bytes](size_t i) {
      const size_t at = i * kPiece, len = std::min(kPiece, bytes - at);
      if (pass((part + at) / per, len / per, stage + at)) any_bad.store(true, std::memory_order_relaxed);
      there[i].store(1, std::memory_order_release);
    };
    HostWorkers &workers = HostWorkers::get();
    const bool shared = kind != HostKind::kBytes && count * sizeof(float) >= kSharedFloats && workers.enter(job);
    int rc = TPUHIP_OK;
    size_t sent = 0;   // pieces handed to the device
    ctx->stage_busy = true;
    for (bool more = true; sent < job->pieces;) {
      if (more) more = job->step();
      size_t run = sent;
      while (run < job->pieces && there[run].load(std::memory_order_acquire)) ++run;
      // one launch moves what is there: at least two pieces (of one thread; four of several) while there is still
      // something to do meanwhile
      if (run == sent || (more && run - sent < (shared ? 4u : 2u))) {
        if (!more) std::this_thread::yield();
        continue;
      }
      const size_t at = sent * kPiece, end = std::min(run * kPiece, bytes);
      if (!rc && !any_bad.load(std::memory_order_relaxed)) rc = stage_copy(ctx, stage + at, (char *)land + part + at, end - at);
      sent = run;
    }
    while (job->finished.load(std::memory_order_acquire) < job->pieces) std::this_thread::yield();
    if (shared) workers.leave();
    if (rc) return rc;
    if (any_bad.load()) {
      *bad = true;
      return TPUHIP_OK;
    }
  }
  if (kind == HostKind::kFloats) return TPUHIP_OK;
  return tpuhip_nchw_to_nhwc_i8(ctx, land, dst, t.n, t.c, t.h, t.w, t.cs);
}

// What a round of device_to_host() does: `Fetch`es fill the staging buffer, `Part`s are passed on to the callers' memory.
namespace {

constexpr size_t kTurn = 8 * kPiece;            // bytes of the staging buffer behind one event
constexpr size_t kDirect = 2 * kPiece;          // laid out straight into the staging buffer up to here
constexpr size_t kSpanLeast = 4 * kPiece, kSpanMost = 8 * kPiece;
constexpr size_t kPastCaches = 16 << 20;        // host bytes of a call from which its floats go past the caches: half of the
                                                // last level; they would evict each other, and the stores read nothing
struct Part {
  const HostRead *r;
  size_t first, count;      // elements
  size_t at;                // byte of the staging buffer
  size_t span;              // there when this many spans have arrived
};

void pass_part(const Part &p, const int8_t *stage, bool past_caches) {
  const HostRead &r = *p.r;
  char *to = (char *)r.dst + p.first * host_size(r.kind);
  if (r.kind == HostKind::kFloatStored)
    bytes_to_floats(stage + p.at, (float *)to, p.count, r.t.is_unsigned, past_caches);
  else
    memcpy(to, stage + p.at, p.count * stage_size(r.kind));
}

size_t elements(const HostRead &r) { return (size_t)r.t.n * r.t.c * r.t.h * r.t.w; }

}  // namespace

// events of the context, at least so many
static int events_ready(tpuhip_ctx *ctx, size_t n) {
  while (ctx->stage_events.size() < n) {
    hipEvent_t e;
    TPUHIP_CHECK_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    ctx->stage_events.push_back(e);
  }
  return TPUHIP_OK;
}

// int8 tensors that fit the staging buffer one by one: their dense forms are made on the device in one launch per filling of the
// buffer.  Up to kDirect together they are laid out straight into it; otherwise they lie in the landing buffer as they will lie
// there and come over in spans of half of what is left, within bounds: a launch and an event cost the bus 5 us a span, and the
// host passes of the last span have no transfer to hide behind.  The host passes run on several threads while the next spans are
// on the bus.  Those threads wait for spans by looking again and again: they are called once the work in front has ended, which
// this thread waits for alone (a read 25 ms behind its launch kept all eight busy for as long, 200 ms of CPU time).
// *done: false where there is no memory for it.
static int read_dense(tpuhip_ctx *ctx, const std::vector<HostRead> &reads, bool past_caches, bool *done) {
  *done = false;
  size_t total = 0;
  for (const HostRead &r : reads) total += (elements(r) + 63) / 64 * 64;
  if (int rc = stage_ready(ctx, total)) return rc;
  const bool direct = total <= kDirect;
  if (!direct && landing_ready(ctx, std::min(total, ctx->stage_bytes)) != TPUHIP_OK) {
    (void)hipGetLastError();
    return TPUHIP_OK;
  }
  *done = true;
  int8_t *stage = (int8_t *)ctx->stage, *to = direct ? stage : (int8_t *)ctx->landing;
  std::vector<Part> parts;
  std::vector<DenseItem> dense;
  std::vector<size_t> ends;   // of the spans
  for (size_t i = 0; i < reads.size();) {
    parts.clear();
    dense.clear();
    ends.clear();
    size_t at = 0;
    for (; i < reads.size(); ++i) {
      const HostRead &r = reads[i];
      const size_t bytes = elements(r);
      if (bytes > ctx->stage_bytes - at) break;
      dense.push_back({(const int8_t *)r.src, to + at, (int64_t)r.t.h * r.t.w, r.t.n, r.t.c, r.t.h, r.t.w, r.t.cs});
      for (size_t p = 0; p < bytes; p += kPiece) parts.push_back({&r, p, std::min(kPiece, bytes - p), at + p, 0});
      at += (bytes + 63) / 64 * 64;
    }
    ctx->stage_busy = true;
    if (direct) {
      if (int rc = lay_out_dense(ctx, dense.data(), dense.size())) return rc;
      TPUHIP_CHECK_HIP(hipStreamSynchronize(ctx->stream));
      ctx->stage_busy = false;
      parallel_pieces(parts.size(), [&](size_t k) { pass_part(parts[k], stage, past_caches); });
      return TPUHIP_OK;
    }
    for (size_t from = 0; from < at; from = ends.back())
      ends.push_back(std::min(at, from + std::min(std::max((at - from) / 2 / kPiece * kPiece, kSpanLeast), kSpanMost)));
    size_t span = 0;
    for (Part &p : parts) {
      while (p.at + p.count > ends[span]) ++span;
      p.span = span;
    }
    if (int rc = events_ready(ctx, ends.size() + 1)) return rc;
    auto job = std::make_shared<HostJob>();
    job->pieces = parts.size();
    std::atomic<size_t> arrived{0};     // spans that are in the buffer
    std::atomic<bool> lost{false};      // the device failed: nothing more arrives
    job->piece = [&](size_t k) {
      const Part &p = parts[k];
      while (arrived.load(std::memory_order_acquire) <= p.span) {
        if (lost.load(std::memory_order_relaxed)) return;
        std::this_thread::yield();
      }
      pass_part(p, stage, past_caches);
    };
    HostWorkers &workers = HostWorkers::get();
    int rc = TPUHIP_OK;
    auto hip = [&](hipError_t e, const char *what) {
      if (!rc && e != hipSuccess) rc = set_error(TPUHIP_ERR_HIP, "%s failed: %s", what, hipGetErrorString(e));
    };
    const hipEvent_t front = ctx->stage_events[ends.size()];
    const bool waits = hipStreamQuery(ctx->stream) != hipSuccess;
    if (waits) hip(hipEventRecord(front, ctx->stream), "hipEventRecord");
    if (!rc) rc = lay_out_dense(ctx, dense.data(), dense.size());
    for (size_t k = 0, from = 0; !rc && k < ends.size(); from = ends[k++]) {
      rc = stage_copy(ctx, (const int8_t *)ctx->landing + from, stage + from, ends[k] - from);
      if (!rc) hip(hipEventRecord(ctx->stage_events[k], ctx->stream), "hipEventRecord");
    }
    if (waits && !rc) hip(hipEventSynchronize(front), "hipEventSynchronize");
    const bool shared = !rc && parts.size() > 1 && workers.enter(job);
    for (size_t k = 0; !rc && k < ends.size(); ++k) {
      hip(hipEventSynchronize(ctx->stage_events[k]), "hipEventSynchronize");
      if (!rc) arrived.store(k + 1, std::memory_order_release);
    }
    if (rc) lost.store(true);
    finish_job(*job);
    if (shared) workers.leave();
    if (rc) return rc;
    ctx->stage_busy = false;
  }
  return TPUHIP_OK;
}

// Float tensors, those that are larger than the staging buffer, and others where read_dense() has no memory.  Tensors of up to
// two pieces are laid out straight into the staging buffer; the dense form of larger ones is made on the device and comes over
// in spans, with an event behind each, and behind small tensors that make one up together.  The threads of the host pass are
// called as there.
static int read_in_turn(tpuhip_ctx *ctx, const std::vector<HostRead> &reads, bool past_caches) {
  const size_t n = reads.size();
  size_t total = 0, largest = 0;
  for (size_t i = 0; i < n; ++i) {
    const size_t bytes = elements(reads[i]) * stage_size(reads[i].kind);
    total += (bytes + 63) / 64 * 64;
    if (bytes > kDirect && reads[i].kind != HostKind::kFloats) largest = std::max(largest, bytes);
  }
  if (int rc = stage_ready(ctx, total)) return rc;
  if (largest)
    if (int rc = landing_ready(ctx, largest)) return rc;
  int8_t *stage = (int8_t *)ctx->stage;
  const size_t room = ctx->stage_bytes;
  auto lay_out = [&](const HostRead &r, void *to) {
    return tpuhip_nhwc_to_nchw_i8(ctx, r.src, to, r.t.n, r.t.c, r.t.h, r.t.w, r.t.cs);
  };

  struct Fetch {
    const HostRead *r;
    size_t from, bytes, at;   // bytes [from, from + bytes) of the dense form -> byte `at` of the buffer
    bool whole, closes;       // laid out in one launch; an event behind it
  };
  std::vector<Fetch> fetches;
  std::vector<Part> parts;
  for (size_t i = 0, done = 0; i < n;) {
    // a round: what fits the buffer
    fetches.clear();
    parts.clear();
    size_t at = 0, spans = 0, open = 0;   // open: bytes fetched behind the last event
    while (i < n) {
      const HostRead &r = reads[i];
      const size_t per = stage_size(r.kind), bytes = elements(r) * per;
      if (at && bytes > room - at && bytes <= room) break;   // in parts only where a round of its own does not help
      const bool whole = bytes <= kDirect;
      while (done < bytes && at < room) {
        const size_t len = std::min({bytes - done, room - at, kTurn});
        fetches.push_back({&r, done, len, at, whole, false});
        open += len;
        for (size_t p = 0; p < len; p += kPiece) {
          const size_t l = std::min(kPiece, len - p);
          parts.push_back({&r, (done + p) / per, l / per, at + p, spans});
        }
        if (open >= kTurn / 2) {
          fetches.back().closes = true;
          ++spans;
          open = 0;
        }
        done += len;
        at += (len + 63) / 64 * 64;
      }
      if (done < bytes) break;
      ++i;
      done = 0;
    }
    if (open) {
      fetches.back().closes = true;
      ++spans;
    }
    if (int rc = events_ready(ctx, spans + 1)) return rc;   // the last one stands behind the work in front
    auto job = std::make_shared<HostJob>();
    job->pieces = parts.size();
    std::atomic<size_t> arrived{0};     // spans that are in the buffer
    std::atomic<bool> lost{false};      // the device failed: nothing more arrives
    job->piece = [&](size_t k) {
      const Part &p = parts[k];
      while (arrived.load(std::memory_order_acquire) <= p.span) {
        if (lost.load(std::memory_order_relaxed)) return;
        std::this_thread::yield();
      }
      pass_part(p, stage, past_caches);
    };
    HostWorkers &workers = HostWorkers::get();
    bool called = false, shared = false;
    auto call_workers = [&] {
      called = true;
      shared = parts.size() > 1 && workers.enter(job);
    };
    int rc = TPUHIP_OK;
    size_t recorded = 0, there = 0;
    auto hip = [&](hipError_t e, const char *what) {
      if (!rc && e != hipSuccess) rc = set_error(TPUHIP_ERR_HIP, "%s failed: %s", what, hipGetErrorString(e));
    };
    const hipEvent_t front = ctx->stage_events[spans];
    if (hipStreamQuery(ctx->stream) == hipSuccess) call_workers();
    else hip(hipEventRecord(front, ctx->stream), "hipEventRecord");
    ctx->stage_busy = true;
    for (const Fetch &f : fetches) {
      if (rc) break;
      if (f.whole) {
        rc = f.r->kind == HostKind::kFloats ? stage_copy(ctx, f.r->src, stage + f.at, f.bytes) : lay_out(*f.r, stage + f.at);
      } else {
        const void *dense = f.r->src;
        if (f.r->kind != HostKind::kFloats) {
          dense = ctx->landing;
          if (f.from == 0) rc = lay_out(*f.r, ctx->landing);
        }
        if (!rc) rc = stage_copy(ctx, (const char *)dense + f.from, stage + f.at, f.bytes);
      }
      if (!rc && f.closes) hip(hipEventRecord(ctx->stage_events[recorded++], ctx->stream), "hipEventRecord");
      if (rc) break;
      if (!called && hipEventQuery(front) == hipSuccess) call_workers();
      while (there < recorded && hipEventQuery(ctx->stage_events[there]) == hipSuccess)
        arrived.store(++there, std::memory_order_release);
    }
    if (!rc && !called) {
      hip(hipEventSynchronize(front), "hipEventSynchronize");
      call_workers();
    }
    while (!rc && there < spans) {
      hip(hipEventSynchronize(ctx->stage_events[there]), "hipEventSynchronize");
      if (!rc) arrived.store(++there, std::memory_order_release);
    }
    if (rc) lost.store(true);
    finish_job(*job);
    if (shared) workers.leave();
    if (rc) return rc;
    ctx->stage_busy = false;
  }
  return TPUHIP_OK;
}

int device_to_host(tpuhip_ctx *ctx, const HostRead *reads, size_t n) {
  if (int rc = not_captured(ctx, "a tensor to the host")) return rc;
  size_t host_total = 0;
  std::vector<HostRead> dense, others;
  for (size_t i = 0; i < n; ++i) {
    host_total += elements(reads[i]) * host_size(reads[i].kind);
    (reads[i].kind != HostKind::kFloats && elements(reads[i]) <= kStageMax ? dense : others).push_back(reads[i]);
  }
  if (n == 1 && host_total <= kAlone) {   // done before a worker has woken
    const size_t bytes = elements(*reads) * stage_size(reads->kind);
    if (int rc = stage_ready(ctx, bytes)) return rc;
    const HostTensor &t = reads->t;
    const int rc = reads->kind == HostKind::kFloats ? stage_copy(ctx, reads->src, ctx->stage, bytes)
                                                    : tpuhip_nhwc_to_nchw_i8(ctx, reads->src, ctx->stage, t.n, t.c, t.h, t.w, t.cs);
    if (rc) return rc;
    TPUHIP_CHECK_HIP(hipStreamSynchronize(ctx->stream));
    pass_part(Part{reads, 0, elements(*reads), 0, 0}, (const int8_t *)ctx->stage, false);
    return TPUHIP_OK;
  }
  const bool past_caches = host_total >= kPastCaches;
  if (!dense.empty()) {
    bool done = false;
    if (int rc = read_dense(ctx, dense, past_caches, &done)) return rc;
    if (!done) others.insert(others.end(), dense.begin(), dense.end());
  }
  return others.empty() ? TPUHIP_OK : read_in_turn(ctx, others, past_caches);
}

AheadRead::~AheadRead() {
  if (dense) (void)hipFree(dense);
  if (pinned) (void)hipHostFree(pinned);
}

// behind the launch whose writes it announces
__global__ void arrived_kernel(uint32_t *flag, uint32_t value) {
  __hip_atomic_store(flag, value, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

int read_ahead(tpuhip_ctx *ctx, AheadRead &a, const HostTensor &t, const void *src, bool *done) {
  *done = false;
  const size_t bytes = ((size_t)t.n * t.c * t.h * t.w + 63) / 64 * 64;
  drop_ahead(ctx, a);
  if (!a.pinned) {
    if (a.refused) return TPUHIP_OK;
    if ((!ctx->copy_stream && hipStreamCreateWithFlags(&ctx->copy_stream, hipStreamNonBlocking) != hipSuccess) ||
        hipMalloc(&a.dense, bytes + 256) != hipSuccess || hipHostMalloc(&a.pinned, bytes + 64, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();   // a read does without
      if (a.dense) (void)hipFree(a.dense);
      a.dense = nullptr;
      a.refused = true;
      return TPUHIP_OK;
    }
    a.flag = (uint32_t *)((char *)a.pinned + bytes);
    *a.flag = 0;
  }
  if (int rc = tpuhip_nhwc_to_nchw_i8(ctx, src, a.dense, t.n, t.c, t.h, t.w, t.cs)) return rc;
  launch(ctx, arrived_kernel, dim3(1), dim3(1), a.flag, ++a.serial);
  TPUHIP_CHECK_HIP(hipGetLastError());
  a.bytes = (size_t)t.n * t.c * t.h * t.w;
  a.fetched = false;
  ctx->ahead.push_back(&a);
  *done = true;
  return TPUHIP_OK;
}

void drop_ahead(tpuhip_ctx *ctx, AheadRead &a) {
  ctx->ahead.erase(std::remove(ctx->ahead.begin(), ctx->ahead.end(), &a), ctx->ahead.end());
}

// The host sees from the flag that the dense form is there and starts a copy engine on it: that needs no wait of one
// stream for another (which costs the host 12 us a piece, 60 in front of a copy), and unlike a kernel the engine takes no
// compute unit from the launches that are still running.
// A wait of some milliseconds gives its CPU back in between.
constexpr int kLooks = 4096;
static int fetch_ahead(tpuhip_ctx *ctx, AheadRead &a) {
  if (a.fetched) return TPUHIP_OK;
  for (int spin = 0; __atomic_load_n(a.flag, __ATOMIC_ACQUIRE) != a.serial; ++spin) {
    if (spin % 256 == 255) {   // a stream that is done, or has failed, without the flag: nothing more will come
      const hipError_t e = hipStreamQuery(ctx->stream);
      if (e != hipErrorNotReady && __atomic_load_n(a.flag, __ATOMIC_ACQUIRE) != a.serial) {
        TPUHIP_CHECK_HIP(e);
        return set_error(TPUHIP_ERR_HIP, "a result laid out early did not arrive");
      }
    }
    if (spin < kLooks) std::this_thread::yield();
    else std::this_thread::sleep_for(std::chrono::microseconds(20));
  }
  TPUHIP_CHECK_HIP(hipSetDevice(ctx->device));
  TPUHIP_CHECK_HIP(hipMemcpyAsync(a.pinned, a.dense, a.bytes, hipMemcpyDeviceToHost, ctx->copy_stream));
  a.fetched = true;
  return TPUHIP_OK;
}

int finish_ahead(tpuhip_ctx *ctx, AheadRead &a, const HostRead &r) {
  if (int rc = not_captured(ctx, "a tensor to the host")) return rc;
  if (int rc = fetch_ahead(ctx, a)) return rc;
  TPUHIP_CHECK_HIP(hipStreamSynchronize(ctx->copy_stream));
  const size_t count = elements(r), grain = kPiece / host_size(r.kind);
  parallel_pieces((count + grain - 1) / grain, [&](size_t i) {
    pass_part(Part{&r, i * grain, std::min(grain, count - i * grain), i * grain, 0}, (const int8_t *)a.pinned, false);
  });
  return TPUHIP_OK;
}

int settle_ahead(tpuhip_ctx *ctx) {
  for (AheadRead *a : ctx->ahead)
    if (int rc = fetch_ahead(ctx, *a)) return rc;
  TPUHIP_CHECK_HIP(hipStreamSynchronize(ctx->stream));
  if (ctx->copy_stream) TPUHIP_CHECK_HIP(hipStreamSynchronize(ctx->copy_stream));
  return TPUHIP_OK;
}

// The copies of a loading module, a row of workgroups each; the list lies in the pinned buffer too.  Bound by the bus, as long as
// enough of it is asked for at once: the largest filter's workgroups hold 1 MB in flight (a thread four 16-byte loads, or dwords
// where a copy's ends do not lie on 16 bytes).  With one dword a thread the filter of 1280 x 1000 among 3.5 MB was 80 trips to
// host memory one behind the other, 133 us, now 78 (45 GB/s).
constexpr int kCopyThreads = 1024, kCopyAhead = 4;

template <class T>
__device__ __forceinline__ void copy_ahead(const uint32_t *src, uint32_t *dst, size_t n) {
  const T *const from = reinterpret_cast<const T *>(src);
  T *const to = reinterpret_cast<T *>(dst);
  constexpr size_t kPass = (size_t)kCopyThreads * kCopyAhead;
  for (size_t at = (size_t)blockIdx.x * kPass + threadIdx.x; at < n; at += gridDim.x * kPass) {
    T v[kCopyAhead];
#pragma unroll
    for (int k = 0; k < kCopyAhead; ++k)
      if (at + k * kCopyThreads < n) v[k] = from[at + k * kCopyThreads];
#pragma unroll
    for (int k = 0; k < kCopyAhead; ++k)
      if (at + k * kCopyThreads < n) to[at + k * kCopyThreads] = v[k];
  }
}

__global__ __launch_bounds__(kCopyThreads) void staged_copies_kernel(const StagedCopy *list) {
  const StagedCopy c = list[blockIdx.y];
  if (((uintptr_t)c.src | (uintptr_t)c.dst) & 15) {
    copy_ahead<uint32_t>(c.src, c.dst, c.dwords);
    return;
  }
  const size_t quads = c.dwords / 4;
  copy_ahead<uint4>(c.src, c.dst, quads);
  if (blockIdx.x == 0 && threadIdx.x < c.dwords % 4) c.dst[4 * quads + threadIdx.x] = c.src[4 * quads + threadIdx.x];
}

// A network of 52 convs took three launches for each, 440 us of a 5 ms tool run; all of them together take three.
int flush_uploads(tpuhip_ctx *ctx) {
  if (ctx->staged.empty() && ctx->packs.empty() && ctx->params.empty()) return TPUHIP_OK;
  if (int rc = not_captured(ctx, "packed weights")) return rc;
  auto place = [&](const void *list, size_t bytes) -> void * {   // stage_upload() leaves the room for it
    void *at = (int8_t *)ctx->stage + ctx->stage_used;
    memcpy(at, list, bytes);
    ctx->stage_used += (bytes + 15) / 16 * 16;
    return at;
  };
  ctx->stage_busy = true;
  if (!ctx->staged.empty()) {
    size_t largest = 0;
    for (auto &c : ctx->staged) largest = std::max(largest, c.dwords);
    constexpr size_t kPass = (size_t)kCopyThreads * kCopyAhead * 4;   // dwords of a workgroup's pass, of 16 bytes a load
    const dim3 grid((unsigned)std::min<size_t>((largest + kPass - 1) / kPass, 16), (unsigned)ctx->staged.size());
    const void *list = place(ctx->staged.data(), ctx->staged.size() * sizeof(StagedCopy));
    hipLaunchKernelGGL(staged_copies_kernel, grid, dim3(kCopyThreads), 0, ctx->stream, (const StagedCopy *)list);
    ctx->staged.clear();
    TPUHIP_CHECK_HIP(hipGetLastError());
  }
  if (!ctx->packs.empty()) {
    int64_t largest = 0;
    for (auto &f : ctx->packs) largest = std::max(largest, f.total);
    const void *list = place(ctx->packs.data(), ctx->packs.size() * sizeof(FilterPack));
    const size_t n = ctx->packs.size();
    ctx->packs.clear();
    if (int rc = pack_filters(ctx, (const FilterPack *)list, n, largest)) return rc;
  }
  if (!ctx->params.empty()) {
    int largest = 0;
    for (auto &p : ctx->params) largest = std::max(largest, p.nparam);
    const void *list = place(ctx->params.data(), ctx->params.size() * sizeof(ParamExpand));
    const size_t n = ctx->params.size();
    ctx->params.clear();
    if (int rc = expand_params(ctx, (const ParamExpand *)list, n, largest)) return rc;
  }
  return TPUHIP_OK;
}

int stage_upload(tpuhip_ctx *ctx, void *dst, const void *src, size_t bytes) {
  // many small uploads pass without a wait between them, those of a usual module without any
  const size_t kRoom = ctx->loading ? 8 << 20 : 4 << 20;
  constexpr size_t kLists = 64 << 10, kMost = 256;   // room for flush_uploads(), and the launches it gathers at most
  for (size_t at = 0; at < bytes;) {
    if (ctx->staged.size() >= kMost || ctx->packs.size() >= kMost || ctx->params.size() >= kMost)
      if (int rc = flush_uploads(ctx)) return rc;
    if (!ctx->stage || ctx->stage_used + kLists + 16 > ctx->stage_bytes ||
        (at == 0 && bytes + kLists <= kRoom && ctx->stage_used + bytes + kLists > ctx->stage_bytes)) {
      if (int rc = stage_ready(ctx, kRoom)) return rc;   // issues what has gathered first
    }
    const size_t len = std::min(bytes - at, ctx->stage_bytes - kLists - ctx->stage_used);
    int8_t *to = (int8_t *)ctx->stage + ctx->stage_used;
    memcpy(to, (const char *)src + at, len);
    ctx->stage_busy = true;
    if (len % 4) {   // a ragged end: whole dwords are copied, and dst need not have the room for the last one
      hipError_t e = hipMemcpyAsync((char *)dst + at, to, len, hipMemcpyHostToDevice, ctx->stream);
      TPUHIP_CHECK_HIP(e);
    } else if (ctx->loading) {
      ctx->staged.push_back({(const uint32_t *)to, (uint32_t *)((char *)dst + at), len / 4});
    } else if (int rc = stage_copy(ctx, to, (char *)dst + at, len)) {
      return rc;
    }
    ctx->stage_used += (len + 15) / 16 * 16;
    at += len;
  }
  return TPUHIP_OK;
}

int prepack_done(tpuhip_ctx *ctx) {
  if (ctx->loading) return TPUHIP_OK;
  TPUHIP_CHECK_HIP(hipStreamSynchronize(ctx->stream));
  return TPUHIP_OK;
}

void host_io_release(tpuhip_ctx *ctx) {
  if (ctx->stage) (void)hipHostFree(ctx->stage);
  if (ctx->landing) (void)hipFree(ctx->landing);
  for (hipEvent_t e : ctx->stage_events) (void)hipEventDestroy(e);
  if (ctx->copy_stream) (void)hipStreamDestroy(ctx->copy_stream);
  ctx->copy_stream = nullptr;
  ctx->stage = ctx->landing = nullptr;
  ctx->stage_bytes = ctx->landing_bytes = 0;
  ctx->stage_events.clear();
}

}  // namespace tpuhip
