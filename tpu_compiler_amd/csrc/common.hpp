// Shared declarations of the tpuhip library: context, error reporting and the
// device-side requantisation arithmetic every kernel epilogue uses.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <map>
#include <string>
#include <unordered_map>
#include <vector>

#include "tpuhip.h"

namespace tpuhip {
// one filter to be packed for a tile variant (conv.hip)
struct FilterPack {
  const int8_t *raw;
  void *out;
  int oc, ic, taps, c16, kp, bm, bk, tm, reg;
  int smallc;
  int64_t total;   // 16-byte groups
};
struct AheadRead;   // host/host_io.hpp
// one piece of the pinned buffer on its way to the device, in dwords
struct StagedCopy {
  const uint32_t *src;
  uint32_t *dst;
  size_t dwords;
};

// A layer's requantisation parameters, made from the three numbers of each channel (conv.hip)
struct ParamExpand {
  const int32_t *raw;    // biases, multipliers, right shifts of oc channels
  int32_t *out;          // nparam biases, then [records], planes, [addends or the narrow form's planes]
  int oc, nparam;
  int records, narrow;
};
}  // namespace tpuhip

struct tpuhip_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  bool owns_stream = false;
  int num_cu = 0;
  bool autotune = true;  // time the conv tile variants on a layer's first use
  // when set, every kernel launch carries these events: they bracket the dispatch
  // itself (begin / end of execution), not the gaps around it
  hipEvent_t prof_start = nullptr, prof_stop = nullptr;
  // device memory kernels use beyond their operands (partial sums of average pools over large windows): allocated on first
  // need, replaced when a larger one comes, freed with the context; never used by a launch that is being recorded
  void *workspace = nullptr;
  size_t workspace_bytes = 0;
  // host tensors on their way to and from the device (host/host_io.cpp): a pinned buffer of at most 32 MiB, device memory
  // for the dense form of a tensor that takes more than one piece, events behind the pieces; made on first use
  void *stage = nullptr, *landing = nullptr;
  size_t stage_bytes = 0, landing_bytes = 0;
  size_t stage_used = 0;     // bytes of the pinned buffer that stage_upload has handed out since it was last free
  bool stage_busy = false;   // kernels that read or write the pinned buffer may still be in flight
  std::vector<hipEvent_t> stage_events;
  // Memory of a module's tensors and packed weights, most of them small and made by the hundred: parts of slabs
  // (api.hip), while `loading`
  struct Slab {
    char *base;
    size_t size;
    std::map<size_t, size_t> unused;   // offset -> bytes
  };
  std::vector<Slab> slabs;
  std::unordered_map<void *, std::pair<char *, size_t>> slab_parts;   // allocation -> its slab's base, its bytes
  // a module is being loaded: packed weights need not be on the device when a prepack call returns, and what is to be
  // uploaded, packed and expanded for them gathers here until flush_uploads() (host_io.cpp) issues all of it in three launches
  bool loading = false;
  std::vector<tpuhip::StagedCopy> staged;
  std::vector<tpuhip::FilterPack> packs;
  std::vector<tpuhip::ParamExpand> params;
  bool in_interpreter = false;   // a module loads or invokes its kernels: device addresses asked for now go to those
  hipStream_t copy_stream = nullptr;   // results laid out early leave on it while `stream` works on; made on first use
  std::vector<tpuhip::AheadRead *> ahead;   // those that may still be asked for
  bool single_pass = false;   // what is issued now runs once: no layer's tile variants are timed for it
};

// conv.hip: looks up this device's copy of the library's static scratch array (the one the
// allocation-free entry point works in); called once per context with the device current
extern "C" int tpuhip_static_scratch_init(int device);
// conv.hip: a context being destroyed stops being the static scratch's last user
extern "C" void tpuhip_static_scratch_forget(const tpuhip_ctx *ctx);

namespace tpuhip {

// sets a flag for as long as it lives
struct FlagScope {
  explicit FlagScope(bool &f) : flag(f), before(f) { flag = true; }
  ~FlagScope() { flag = before; }
  FlagScope(const FlagScope &) = delete;
  bool &flag;
  bool before;
};

// host/host_io.cpp: frees a context's staging buffers
void host_io_release(tpuhip_ctx *ctx);
// host/host_io.cpp: refuses what moves host memory while the context's stream is being captured
int not_captured(tpuhip_ctx *ctx, const char *what);
// host/host_io.cpp: tpuhip_upload without the wait -- src may be reused on return, the bytes are there for what is issued to
// the context's stream afterwards
int stage_upload(tpuhip_ctx *ctx, void *dst, const void *src, size_t bytes);
// issues what has gathered in ctx->staged, ctx->packs and ctx->params
int flush_uploads(tpuhip_ctx *ctx);
// A 256-entry table that is y -> max(y, (y * m + 2^(r - 1)) >> r) with 0 < m <= 2^r and products within 16 bits: a leaky ReLU's,
// which the conv kernels compute instead of looking it up.  m == 0: none.
struct LeakySlope {
  int m = 0, r = 0;
};
// conv.hip: the line of the fewest bits, if the table is one (1.3 us: for whoever loads a model, not for a call)
bool slope_of_table(const int8_t *table, LeakySlope *out);
// conv.hip: tpuhip_conv2d_post_i8 by a caller that knows what slope_of_table() says of post->lut (NULL: does not)
int conv2d_post(tpuhip_ctx *ctx, const tpuhip_conv_weights *w, const void *x, void *y, const tpuhip_conv_post *post,
                const LeakySlope *slope);
// elementwise.hip: channels-last int8 tensors to dense NCHW bytes, all in one launch as far as it takes them
struct DenseItem {
  const int8_t *src;
  int8_t *dst;
  int64_t hw;
  int n, c, h, w, cs;
};
int lay_out_dense(tpuhip_ctx *ctx, const DenseItem *items, size_t n);
// entries of a conv's plane of biases, multipliers, ...: they cover every tile's padding
__host__ __device__ constexpr int param_entries(int oc) { return ((oc + 255) & ~255) + 16; }
// conv.hip: packs n filters; the list is in memory the device reads
int pack_filters(tpuhip_ctx *ctx, const FilterPack *list, size_t n, int64_t largest);
// conv.hip: makes the requantisation parameters of n layers; the list likewise
int expand_params(tpuhip_ctx *ctx, const ParamExpand *list, size_t n, int largest);
// waits for what a prepack call has issued, unless a module is being loaded: packed weights may be used from any context
int prepack_done(tpuhip_ctx *ctx);

// api.hip: makes ctx->workspace at least this large; waits for the stream when it has to be replaced.  TPUHIP_ERR_NOMEM: there
// is none, and the call may do without
int grow_workspace(tpuhip_ctx *ctx, size_t bytes);

// api.hip: raises a kernel's dynamic LDS limit, once per device, kernel and size: the limit is a setting of the device that is
// current, and the context's becomes it (kernels of one signature share their function-pointer type, so the record is keyed by the
// kernel's address); on failure the runtime's last error stays set for the caller to report
bool raise_lds_limit(int device, const void *kernel, unsigned bytes);

int set_error(int status, const char *fmt, ...) __attribute__((format(printf, 2, 3)));

#define TPUHIP_CHECK_HIP(expr)                                                          \
  do {                                                                                  \
    hipError_t e__ = (expr);                                                            \
    if (e__ != hipSuccess)                                                              \
      return ::tpuhip::set_error(TPUHIP_ERR_HIP, "%s failed: %s (%s:%d)", #expr,        \
                                 hipGetErrorString(e__), __FILE__, __LINE__);           \
  } while (0)

#define TPUHIP_REQUIRE(cond, ...)                                                       \
  do {                                                                                  \
    if (!(cond)) return ::tpuhip::set_error(TPUHIP_ERR_INVALID, __VA_ARGS__);           \
  } while (0)

// Launches on the context's stream; with profiling events set the dispatch records
// its own begin / end timestamps into them.
template <typename F, typename... Args>
inline void launch(tpuhip_ctx *ctx, F kernel, dim3 grid, dim3 block, Args... args) {
  if (ctx->prof_start)
    hipExtLaunchKernelGGL(kernel, grid, block, 0, ctx->stream, ctx->prof_start, ctx->prof_stop, 0,
                          args...);
  else
    hipLaunchKernelGGL(kernel, grid, block, 0, ctx->stream, args...);
}

inline int round_up(int v, int m) { return (v + m - 1) / m * m; }
inline int64_t ceil_div64(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Division of 31-bit numbers by a divisor the host knows, as a multiply and a shift (two instructions; the compiler's own
// division by an unknown number is some thirty, its 64-bit one a hundred and more): q = (umulhi(x, mul) + x) >> shift with
// 2^(shift-1) < d <= 2^shift and mul = floor(2^32 * (2^shift - d) / d) + 1, exact for x < 2^31.
struct FastDiv {
  uint32_t d = 1, mul = 0, shift = 0;
  FastDiv() = default;
  explicit FastDiv(int64_t divisor) : d((uint32_t)divisor) {
    while ((1ull << shift) < d) ++shift;
    mul = (uint32_t)(((1ull << 32) * ((1ull << shift) - d)) / d + 1);
  }
  __device__ __forceinline__ uint32_t div(uint32_t x) const { return (__umulhi(x, mul) + x) >> shift; }
  // x -> quotient, remainder in x
  __device__ __forceinline__ uint32_t split(uint32_t &x) const {
    const uint32_t q = div(x);
    x -= q * d;
    return q;
  }
};

// 256-entry int8 table passed to kernels by value (lives in the kernel-argument
// segment, so no device allocation or copy is needed and launches stay capturable).
struct Table256 {
  uint32_t w[64];
};

// ---------------------------------------------------------------------------
// Requantisation arithmetic (QuantizationArithmetic.cpp:487-539), device side.
// ---------------------------------------------------------------------------

// SaturatingRoundingDoublingHighMul (:501-509).  The reference adds a
// sign-dependent nudge and divides by 2^31 truncating toward zero; for every
// pair of int32 that equals floor((a*b + 2^30) / 2^31), i.e. one 64-bit
// multiply-add and an arithmetic shift.  The cast keeps the low 32 bits like
// the reference's static_cast.
__device__ __forceinline__ int32_t srdhm(int32_t a, int32_t b) {
  const int64_t ab = (int64_t)a * (int64_t)b;
  return (int32_t)((ab + (1ll << 30)) >> 31);
}

// RoundingDivideByPOT (:487-499) with mask = 2^e - 1 and half = mask >> 1
// precomputed per channel; exact for e in [0,31] (e == 0 gives mask 0, so the
// value passes through) and for x == 0.
__device__ __forceinline__ int32_t rdbp(int32_t x, int32_t e, int32_t mask, int32_t half) {
  const int32_t rem = x & mask;
  const int32_t thr = half - (x >> 31);  // + 1 when x < 0
  return (x >> e) + (rem > thr ? 1 : 0);
}

__device__ __forceinline__ int32_t clamp_i32(int32_t v, int32_t lo, int32_t hi) {
  return min(max(v, lo), hi);
}

// applyMultiplierAndRShiftAndSaturateInt8(int32, rshift, multiplier, qdm=true) (:530-539)
// followed by the optional ReLU of :866-868, folded into the lower clamp bound.
__device__ __forceinline__ int32_t requant_qdm(int32_t v, int32_t mult, int32_t e, int32_t mask,
                                               int32_t half, int32_t lo) {
  return clamp_i32(rdbp(srdhm(v, mult), e, mask, half), lo, 127);
}

// saturateInt8 (:301-334) of a float that holds v * m / 2^r computed the
// reference's way (float product, float quotient): floor(f + 0.5) evaluated
// exactly, then the clamp.
__device__ __forceinline__ int32_t saturate_int8_f(float f) {
  f = fminf(fmaxf(f, -1024.0f), 1024.0f);   // the clamp makes the range harmless
  const float fl = floorf(f);
  const float frac = f - fl;                // exact
  int32_t q = (int32_t)fl + (frac >= 0.5f ? 1 : 0);
  return clamp_i32(q, -128, 127);
}

}  // namespace tpuhip
