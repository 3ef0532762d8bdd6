// Pure data movement on int8 channels-last tensors: Pad, Crop, Permute, Reorg, Tile,
// Reverse, ShuffleChannel, DepthToSpace, SwapChannel, Dilate, ReflectionPad (core/pad.cpp, crop.cpp, permute.cpp,
// reorg.cpp, tile.cpp, reverse.cpp, shuffle_channel.cpp, depthtospace.cpp, swap_channel.cpp,
// dilate.cpp, reflectionpad.cpp).  Each is an index map from the logical (n, c, h, w) of an
// output element to that of its source, known at compile time to the kernel that evaluates it;
// a lane produces 16 consecutive output channels of a pixel, pad channels written as zero.
#include "common.hpp"

#include <cstring>

using namespace tpuhip;

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
constexpr int kThreads = 256;

// the index maps; the three that move single channels are at the end
enum Form {
  kPadConst, kPadCut, kPadEdge, kCrop, kReorg, kTile, kTileChannel, kReverse, kDilate, kReflectionPad, kDepthDcr,
  kReverseChannel, kShuffle, kWeave, kSwap, kStrided
};

// What a kernel reads of it is in the MoveArgs of its form: up to 112 bytes of arguments a launch costs the host 3.1 us
// back to back, with more 3.65 us, and these kernels take less than that (ten of them on 4 x 96 x 78 x 66: 43 -> 38 us).
struct MovePlan {
  const int8_t *x;
  int8_t *y;
  int in, ic, ih, iw, ics;
  int on, oc, oh, ow, ocs;
  int p[12];
  int fill;        // the byte of an element without a source (0 except for Dilate)
  FastDiv by_groups, by_ow, by_oh;
  FastDiv by_a, by_b, by_c;   // what the map divides by
};

struct MoveBase {
  const int8_t *x;
  int8_t *y;
  int ih, iw, ics, oc;
  FastDiv by_groups, by_ow, by_oh;
  uint32_t pix0;   // first output pixel of this launch
  uint32_t total;  // output pixels * 16-channel groups of this launch, below 2^31
  __host__ __device__ int ocs() const { return (int)by_groups.d * 16; }
};
template <int N, bool A = false, bool B = false>
struct MoveTail {
  int ic;
  int p[N];
  FastDiv by_a, by_b;
  void take(const MovePlan &m) {
    ic = m.ic;
    for (int k = 0; k < N; ++k) p[k] = m.p[k];
    by_a = m.by_a, by_b = m.by_b;
  }
};
template <int N>
struct MoveTail<N, true, false> {
  int ic;
  int p[N];
  FastDiv by_a;
  void take(const MovePlan &m) {
    ic = m.ic;
    for (int k = 0; k < N; ++k) p[k] = m.p[k];
    by_a = m.by_a;
  }
};
template <int N>
struct MoveTail<N, false, false> {
  int ic;
  int p[N];
  void take(const MovePlan &m) {
    ic = m.ic;
    for (int k = 0; k < N; ++k) p[k] = m.p[k];
  }
};
struct MoveTailTile {
  FastDiv by_a, by_b, by_c;
  void take(const MovePlan &m) { by_a = m.by_a, by_b = m.by_b, by_c = m.by_c; }
};
struct MoveTailDilate {
  int fill;
  FastDiv by_a, by_b;
  void take(const MovePlan &m) { fill = m.fill, by_a = m.by_a, by_b = m.by_b; }
};
struct MoveTailCrop {   // p[0..7] less the channels' step
  int p[8];
  void take(const MovePlan &m) {
    for (int k = 0; k < 8; ++k) p[k] = m.p[k];
    p[5] = m.ic;
  }
};
struct MoveTailReverse {
  int in, axis;
  void take(const MovePlan &m) { in = m.in, axis = m.p[0]; }
};
struct MoveTailDepth {
  int ow;
  void take(const MovePlan &m) { ow = m.ow; }
};

template <Form F> struct TailOf { using type = MoveTail<1>; };                     // kReflectionPad, kReverseChannel
template <> struct TailOf<kPadConst> { using type = MoveTail<5>; };                // p[4]: input images
template <> struct TailOf<kPadCut> { using type = MoveTail<12>; };
template <> struct TailOf<kPadEdge> { using type = MoveTail<4>; };
template <> struct TailOf<kCrop> { using type = MoveTailCrop; };
template <> struct TailOf<kReorg> { using type = MoveTail<1, true, true>; };
template <> struct TailOf<kTile> { using type = MoveTailTile; };
template <> struct TailOf<kTileChannel> { using type = MoveTail<1, true>; };
template <> struct TailOf<kReverse> { using type = MoveTailReverse; };
template <> struct TailOf<kDilate> { using type = MoveTailDilate; };
template <> struct TailOf<kDepthDcr> { using type = MoveTail<1, true>; };
template <> struct TailOf<kShuffle> { using type = MoveTail<2, true>; };
template <> struct TailOf<kWeave> { using type = MoveTail<2, true>; };               // kShuffle of two or four groups
template <> struct TailOf<kSwap> { using type = MoveTail<8>; };
template <> struct TailOf<kStrided> { using type = MoveTail<9, true>; };

template <class Tail>
struct MoveWith : MoveBase, Tail {};
template <Form F>
using MoveArgs = MoveWith<typename TailOf<F>::type>;
static_assert(sizeof(MoveArgs<kTile>) <= 112 && sizeof(MoveArgs<kCrop>) <= 112 && sizeof(MoveArgs<kReorg>) <= 112 &&
                  sizeof(MoveArgs<kPadConst>) <= 112 && sizeof(MoveArgs<kSwap>) <= 112 && sizeof(MoveArgs<kDilate>) <= 112,
              "see MovePlan");

// 4 x 4 bytes: byte k of row i becomes byte i of t[k]
__device__ __forceinline__ void transpose_bytes(const uint32_t (&r)[4], uint32_t (&t)[4]) {
  const uint32_t lo0 = __builtin_amdgcn_perm(r[1], r[0], 0x05010400u), hi0 = __builtin_amdgcn_perm(r[1], r[0], 0x07030602u);
  const uint32_t lo1 = __builtin_amdgcn_perm(r[3], r[2], 0x05010400u), hi1 = __builtin_amdgcn_perm(r[3], r[2], 0x07030602u);
  t[0] = __builtin_amdgcn_perm(lo1, lo0, 0x05040100u);
  t[1] = __builtin_amdgcn_perm(lo1, lo0, 0x07060302u);
  t[2] = __builtin_amdgcn_perm(hi1, hi0, 0x05040100u);
  t[3] = __builtin_amdgcn_perm(hi1, hi0, 0x07060302u);
}

// where output channel c of pixel (n, h, w) comes from, and how many channels from it on, c included, lie one after the other
// in the source as well (p null: without a source, that many take a.fill).  A source row that ends with the output's ends in
// zero pad bytes up to a multiple of 16: `left` is then 16.
struct Run {
  const int8_t *p;
  int left;
};

template <Form F>
__device__ __forceinline__ Run run_at(const MoveArgs<F> &a, int n, int h, int w, int c) {
  auto at = [&](int sn, int sc, int sh, int sw) { return a.x + ((int64_t)(sn * a.ih + sh) * a.iw + sw) * a.ics + sc; };
  if constexpr (F == kPadConst) {   // nothing is cut: p[0..3] where the input's first element lands, p[4] its images
    const int sn = n - a.p[0], sc = c - a.p[1], sh = h - a.p[2], sw = w - a.p[3];
    if (sn < 0 || sn >= a.p[4] || sh < 0 || sh >= a.ih || sw < 0 || sw >= a.iw || sc >= a.ic) return {nullptr, a.oc - c};
    if (sc < 0) return {nullptr, -sc};
    return {at(sn, sc, sh, sw), a.ic == a.oc && sc == c ? 16 : a.ic - sc};
  } else if constexpr (F == kPadCut) {
    // p[0..3] where the first kept input element lands, p[4..7] its index, p[8..11] end of the kept input range
    const int sn = n - a.p[0] + a.p[4], sc = c - a.p[1] + a.p[5], sh = h - a.p[2] + a.p[6], sw = w - a.p[3] + a.p[7];
    if (sn < a.p[4] || sn >= a.p[8] || sh < a.p[6] || sh >= a.p[10] || sw < a.p[7] || sw >= a.p[11] || sc >= a.p[9])
      return {nullptr, a.oc - c};
    if (sc < a.p[5]) return {nullptr, a.p[5] - sc};
    return {at(sn, sc, sh, sw), a.ic == a.oc && sc == c ? 16 : a.p[9] - sc};
  } else if constexpr (F == kPadEdge) {
    return {at(n, c, min(max(h - a.p[2], 0), a.ih - 1), min(max(w - a.p[3], 0), a.iw - 1)), 16};
  } else if constexpr (F == kCrop) {   // p[0..3] offsets, p[4..7] steps, but for the channels' (1), whose place has the input's channels
    return {at(n * a.p[4] + a.p[0], c + a.p[1], h * a.p[6] + a.p[2], w * a.p[7] + a.p[3]), a.p[5] == a.oc ? 16 : a.oc - c};
  } else if constexpr (F == kReorg) {   // by_a: input channels, by_b: the stride p[0]
    uint32_t sc = (uint32_t)c, dw = a.by_a.split(sc);
    const int dh = (int)a.by_b.split(dw);
    return {at(n, (int)sc, h * a.p[0] + dh, w * a.p[0] + (int)dw), a.ic - (int)sc};
  } else if constexpr (F == kTile) {   // p[0]: the axis; by_a, by_b, by_c: input n, h, w
    uint32_t sn = (uint32_t)n, sh = (uint32_t)h, sw = (uint32_t)w;
    a.by_a.split(sn), a.by_b.split(sh), a.by_c.split(sw);
    return {at((int)sn, c, (int)sh, (int)sw), 16};
  } else if constexpr (F == kTileChannel) {   // by_a: input channels
    uint32_t sc = (uint32_t)c;
    a.by_a.split(sc);
    return {at(n, (int)sc, h, w), a.ic - (int)sc};
  } else if constexpr (F == kReverse) {
    return {at(a.axis == 0 ? a.in - 1 - n : n, c, a.axis == 2 ? a.ih - 1 - h : h, a.axis == 3 ? a.iw - 1 - w : w), 16};
  } else if constexpr (F == kDilate) {   // by_a = ins_w + 1, by_b = ins_h + 1: input elements sit on that grid
    uint32_t rw = (uint32_t)w, rh = (uint32_t)h;
    const int sw = (int)a.by_a.split(rw), sh = (int)a.by_b.split(rh);
    if (rw | rh) return {nullptr, a.oc - c};
    return {at(n, c, sh, sw), 16};
  } else if constexpr (F == kReflectionPad) {   // p[0]: columns added on the left; mirrored about the first / last column
    const int j = w - a.p[0];
    return {at(n, c, h, j < 0 ? -j : j >= a.iw ? 2 * (a.iw - 1) - j : j), 16};
  } else {   // kDepthDcr, by_a = the upscale factor p[0]
    uint32_t dw = (uint32_t)w, dh = (uint32_t)h;
    const int sw = (int)a.by_a.split(dw), sh = (int)a.by_a.split(dh);
    return {at(n, ((int)dh * a.p[0] + (int)dw) * a.oc + c, sh, sw), a.oc - c};
  }
}

// 16 channels of runs: one load at any alignment where they lie in one run, else a dword or a byte at a time
template <Form F>
__device__ __forceinline__ v4i group_of_runs(const MoveArgs<F> &a, int n, int h, int w, int c0) {
  uint32_t fill = 0;
  if constexpr (F == kDilate) fill = (uint32_t)(uint8_t)a.fill * 0x01010101u;
  v4i out = {(int)fill, (int)fill, (int)fill, (int)fill};
  const Run r = run_at<F>(a, n, h, w, c0);
  if (r.left >= 16) {
    if (r.p) __builtin_memcpy(&out, r.p, 16);
    return out;
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int c = c0 + q * 4;
    uint32_t word = 0;
    const Run d = c < a.oc ? run_at<F>(a, n, h, w, c) : Run{nullptr, 0};
    if (d.left >= 4) {
      word = fill;
      if (d.p) __builtin_memcpy(&word, d.p, 4);
    } else {
      for (int b = 0; b < 4 && c + b < a.oc; ++b) {
        const Run e = run_at<F>(a, n, h, w, c + b);
        word |= (e.p ? (uint32_t)(uint8_t)*e.p : fill & 255u) << (8 * b);
      }
    }
    out[q] = (int)word;
  }
  return out;
}

// 16 channels that do not follow each other in the source: byte loads, all in flight, out of lines the wave shares
template <Form F>
__device__ __forceinline__ v4i group_of_bytes(const MoveArgs<F> &a, int n, int h, int w, int c0) {
  v4i out = {0, 0, 0, 0};
  const int live = min(a.oc - c0, 16);
  if constexpr (F == kReverseChannel) {
    const int8_t *end = a.x + ((int64_t)(n * a.ih + h) * a.iw + w) * a.ics + (a.ic - c0);   // behind channel c0's source
    if (live == 16) {
      uint32_t t[4];
      __builtin_memcpy(t, end - 16, 16);
#pragma unroll
      for (int q = 0; q < 4; ++q) out[q] = (int)__builtin_bswap32(t[3 - q]);
      return out;
    }
    for (int b = 0; b < live; ++b) out[b >> 2] |= (int)((uint32_t)(uint8_t)end[-1 - b] << (8 * (b & 3)));
    return out;
  }
  const int8_t *row;
  int64_t at, step = 1;       // kStrided: bytes from one channel's source to the next one's
  uint32_t g = 0, col = 0;    // kShuffle, kWeave: group (by_a) and column (p[1] of them) of the channel
  if constexpr (F == kStrided) {
    if (a.p[8]) {             // depth to space, CRD; by_a = the factor p[0]
      uint32_t dw = (uint32_t)w, dh = (uint32_t)h;
      const int sw = (int)a.by_a.split(dw), sh = (int)a.by_a.split(dh);
      row = a.x + ((int64_t)(n * a.ih + sh) * a.iw + sw) * a.ics;
      step = (int64_t)a.p[0] * a.p[0];
      at = c0 * step + dh * a.p[0] + dw;
    } else {                  // crop with a step over the channels
      row = a.x + ((int64_t)((n * a.p[4] + a.p[0]) * a.ih + h * a.p[6] + a.p[2]) * a.iw + w * a.p[7] + a.p[3]) * a.ics;
      step = a.p[5];
      at = c0 * step + a.p[1];
    }
  } else {
    row = a.x + ((int64_t)(n * a.ih + h) * a.iw + w) * a.ics;
    if constexpr (F == kShuffle || F == kWeave) {
      g = (uint32_t)c0;
      col = a.by_a.split(g);
    }
    // 16 channels that exist: runs of 8 or 4 bytes of each group, at any alignment, woven in registers.  Replayed from a graph, byte
    // by byte and now: four groups of 4 x 96 x 78 x 66 3.72 -> 2.33 us, 16 x 320 x 100 x 90 43 -> 15.  A form of its own: asking for it
    // cost the other numbers of groups 2 to 3 % (three of 1 x 24 x 7 x 7: 2.65 and 2.74; eight of 16 x 320 x 100 x 90: 31.1 and 31.7).
    if constexpr (F == kWeave) {
      if (live == 16 && a.by_a.d == 4) {
        uint32_t r[4], t[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) __builtin_memcpy(&r[k], row + (int64_t)k * a.p[1] + col, 4);
        transpose_bytes(r, t);
        return v4i{(int)t[0], (int)t[1], (int)t[2], (int)t[3]};
      }
      if (live == 16) {
        uint32_t r[2][2];
        __builtin_memcpy(r[0], row + col, 8);
        __builtin_memcpy(r[1], row + a.p[1] + col, 8);
#pragma unroll
        for (int q = 0; q < 4; ++q)
          out[q] = (int)__builtin_amdgcn_perm(r[1][q >> 1], r[0][q >> 1], q & 1 ? 0x07030602u : 0x05010400u);
        return out;
      }
    }
  }
  uint32_t bytes[16];
#pragma unroll
  for (int b = 0; b < 16; ++b) {
    if constexpr (F == kSwap) {
      at = 0;
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (b == k) at = a.p[k];
    } else if constexpr (F == kShuffle || F == kWeave) {
      at = (int64_t)g * a.p[1] + col;
      if (++g == a.by_a.d) g = 0, ++col;
    }
    bytes[b] = b < live ? (uint8_t)row[at] : 0;
    if constexpr (F == kStrided) at += step;
  }
#pragma unroll
  for (int q = 0; q < 4; ++q)
    out[q] = (int)(bytes[q * 4] | bytes[q * 4 + 1] << 8 | bytes[q * 4 + 2] << 16 | bytes[q * 4 + 3] << 24);
  return out;
}

// Bound by memory at size and by the launch below: on 4 x 96 x 78 x 66 the maps that a general kernel made byte by byte,
// with the map chosen at run time, took 7 to 13 us each.
template <Form F>
__global__ __launch_bounds__(kThreads) void move_kernel(MoveArgs<F> a) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= a.total) return;
  uint32_t cg = i;
  const uint32_t pix = a.pix0 + a.by_groups.split(cg);
  uint32_t w = pix, h = a.by_ow.split(w);
  const int n = (int)a.by_oh.split(h), c0 = (int)cg * 16;
  v4i out = {0, 0, 0, 0};
  if (c0 < a.oc) {
    if constexpr (F >= kReverseChannel) out = group_of_bytes<F>(a, n, (int)h, (int)w, c0);
    else out = group_of_runs<F>(a, n, (int)h, (int)w, c0);
  }
  *reinterpret_cast<v4i *>(a.y + (int64_t)pix * a.ocs() + c0) = out;
}

// depth to space by two, CRD: the four bytes of an input dword go to the same channel of four output pixels.  A lane reads 64
// bytes of an input pixel and writes a group of each of the four.
__global__ __launch_bounds__(kThreads) void depth_by_two_kernel(MoveWith<MoveTailDepth> a) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= a.total) return;
  uint32_t cg = i;
  const uint32_t pix = a.pix0 + a.by_groups.split(cg);   // input pixel
  uint32_t w = pix;
  const uint32_t row = a.by_ow.split(w);                 // by_ow: input columns here
  const int c0 = (int)cg * 16;
  uint32_t out[4][4] = {};
  if (c0 < a.oc) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      // channels past the last are the zero pad bytes of the input's row, or lie beyond its stride
      v4i v = {0, 0, 0, 0};
      if (c0 * 4 + q * 16 < a.ics) v = *reinterpret_cast<const v4i *>(a.x + (int64_t)pix * a.ics + c0 * 4 + q * 16);
      const uint32_t r[4] = {(uint32_t)v[0], (uint32_t)v[1], (uint32_t)v[2], (uint32_t)v[3]};
      uint32_t t[4];
      transpose_bytes(r, t);
#pragma unroll
      for (int k = 0; k < 4; ++k) out[k][q] = t[k];
    }
  }
  int8_t *to = a.y + ((int64_t)row * 2 * a.ow + 2 * w) * a.ocs() + c0;
#pragma unroll
  for (int k = 0; k < 4; ++k)
    *reinterpret_cast<v4i *>(to + ((int64_t)(k >> 1) * a.ow + (k & 1)) * a.ocs()) =
        v4i{(int)out[k][0], (int)out[k][1], (int)out[k][2], (int)out[k][3]};
}

// QuantOp at the graph edges (core/quant.cpp).  The float side is NCHW like the reference's
// tensors, the int8 side channels-last: the layout change rides along.
__device__ __forceinline__ float bf16_rne(float v) {   // QuantizationArithmetic.cpp:893-905
  uint32_t u = __float_as_uint(v);
  u += 0x7fffu + ((u >> 16) & 1u);
  uint32_t h = u >> 16;
  if ((h & 0x7f80u) == 0x7f80u) h = 0x7f7fu;
  return __uint_as_float(h << 16);
}

__global__ __launch_bounds__(kThreads) void quant_f32_to_i8_kernel(const float *x, int8_t *y, int n,
                                                                   int c, int h, int w, int cs,
                                                                   float scale) {
  const int64_t total = (int64_t)n * h * w * cs;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int ch = (int)(i % cs);
    const int64_t pix = i / cs;
    int8_t out = 0;
    if (ch < c) {
      const int iw = (int)(pix % w), ih = (int)((pix / w) % h), in = (int)(pix / ((int64_t)w * h));
      const float v = x[(((int64_t)in * c + ch) * h + ih) * w + iw];
      const float r = roundf(__fmul_rn(v, scale));   // std::round: half away from zero
      out = (int8_t)(r > 127.0f ? 127 : r < -128.0f ? -128 : (int)r);
    }
    y[i] = out;
  }
}

__global__ __launch_bounds__(kThreads) void dequant_i8_to_f32_kernel(const int8_t *x, float *y,
                                                                     int n, int c, int h, int w,
                                                                     int cs, float scale_bf16) {
  const int64_t total = (int64_t)n * c * h * w;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int iw = (int)(i % w), ih = (int)((i / w) % h);
    const int ch = (int)((i / ((int64_t)w * h)) % c), in = (int)(i / ((int64_t)w * h * c));
    const float v = (float)x[(((int64_t)in * h + ih) * w + iw) * cs + ch];   // exact in bf16
    y[i] = bf16_rne(__fmul_rn(v, scale_bf16));
  }
}

}  // namespace

extern "C" int tpuhip_quant_f32_to_i8(tpuhip_ctx *ctx, const void *x_nchw_f32, void *y, int n, int c,
                                      int h, int w, int cs, float scale) {
  TPUHIP_REQUIRE(ctx && x_nchw_f32 && y, "quant: NULL argument");
  TPUHIP_REQUIRE(n > 0 && c > 0 && h > 0 && w > 0 && cs >= c && cs % 16 == 0, "quant: bad shape");
  TPUHIP_CHECK_HIP(hipSetDevice(ctx->device));
  const int64_t total = (int64_t)n * h * w * cs;
  const unsigned blocks = (unsigned)std::max<int64_t>(
      1, std::min<int64_t>(ceil_div64(total, kThreads), (int64_t)ctx->num_cu * 32));
  launch(ctx, quant_f32_to_i8_kernel, dim3(blocks), dim3(kThreads), (const float *)x_nchw_f32,
         (int8_t *)y, n, c, h, w, cs, scale);
  TPUHIP_CHECK_HIP(hipGetLastError());
  return TPUHIP_OK;
}

extern "C" int tpuhip_dequant_i8_to_f32(tpuhip_ctx *ctx, const void *x, void *y_nchw_f32, int n, int c,
                                        int h, int w, int cs, float scale) {
  TPUHIP_REQUIRE(ctx && x && y_nchw_f32, "dequant: NULL argument");
  TPUHIP_REQUIRE(n > 0 && c > 0 && h > 0 && w > 0 && cs >= c && cs % 16 == 0, "dequant: bad shape");
  TPUHIP_CHECK_HIP(hipSetDevice(ctx->device));
  // scale = BF16(scale) on the host (quant.cpp:110), same rounding as the device function
  uint32_t u;
  memcpy(&u, &scale, 4);
  u += 0x7fffu + ((u >> 16) & 1u);
  uint32_t hbits = u >> 16;
  if ((hbits & 0x7f80u) == 0x7f80u) hbits = 0x7f7fu;
  hbits <<= 16;
  float sb;
  memcpy(&sb, &hbits, 4);
  const int64_t total = (int64_t)n * c * h * w;
  const unsigned blocks = (unsigned)std::max<int64_t>(
      1, std::min<int64_t>(ceil_div64(total, kThreads), (int64_t)ctx->num_cu * 32));
  launch(ctx, dequant_i8_to_f32_kernel, dim3(blocks), dim3(kThreads), (const int8_t *)x,
         (float *)y_nchw_f32, n, c, h, w, cs, sb);
  TPUHIP_CHECK_HIP(hipGetLastError());
  return TPUHIP_OK;
}

namespace {

// Reduce over consecutive logical (NCHW) axes: kind 0 mean / 1 sum / 2 max / 3 min
// (core/reduce.cpp:54-117, INT8).  A lane produces four consecutive channels of an output
// pixel; each walks its `axis` sources through the logical index map.
struct ReduceArgs {
  const int8_t *x;
  int8_t *y;
  int kind, requant;
  int ic, ih, iw, ics;
  int oc, oh, ow, ocs;
  int axis, inner;
  float mult, inv_pot;
  int64_t total;   // output pixels * (ocs / 4)
};

__global__ __launch_bounds__(kThreads) void reduce_kernel(ReduceArgs a) {
  const int c4 = a.ocs >> 2;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < a.total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int cq = (int)(i % c4);
    const int pix = (int)(i / c4);
    const int w = pix % a.ow;
    const int h = (pix / a.ow) % a.oh;
    const int n = pix / (a.ow * a.oh);
    uint32_t word = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int c = cq * 4 + b;
      if (c >= a.oc) continue;
      // logical flat index of the output element, split at the reduced axes
      const int64_t e = (((int64_t)n * a.oc + c) * a.oh + h) * a.ow + w;
      const int64_t o = e / a.inner, in = e - o * a.inner;
      int acc = a.kind == 2 ? -128 : a.kind == 3 ? 127 : 0;
      for (int k = 0; k < a.axis; ++k) {
        const int64_t l = (o * a.axis + k) * a.inner + in;
        const int sw = (int)(l % a.iw);
        const int64_t t1 = l / a.iw;
        const int sh = (int)(t1 % a.ih);
        const int64_t t2 = t1 / a.ih;
        const int sc = (int)(t2 % a.ic);
        const int64_t sn = t2 / a.ic;
        const int v = a.x[((sn * a.ih + sh) * a.iw + sw) * a.ics + sc];
        acc = a.kind <= 1 ? acc + v : a.kind == 2 ? max(acc, v) : min(acc, v);
      }
      int r = acc;
      if (a.requant) {
        // the float overload of applyMultiplierAndRShiftAndSaturateInt8 without qdm
        const float prod = __fmul_rn((float)acc, a.mult);
        r = saturate_int8_f(__fmul_rn(prod, a.inv_pot));   // power-of-two scaling: exact
      }
      word |= (uint32_t)(uint8_t)(int8_t)r << (8 * b);
    }
    *reinterpret_cast<uint32_t *>(a.y + (int64_t)pix * a.ocs + cq * 4) = word;
  }
}

}  // namespace

extern "C" int tpuhip_reduce_i8(tpuhip_ctx *ctx, int kind, const void *x, void *y, const int *in_nchw,
                                int x_cs, const int *out_nchw, int y_cs, int first_axis, int last_axis,
                                int rshift, uint32_t multiplier) {
  TPUHIP_REQUIRE(ctx && x && y && in_nchw && out_nchw, "reduce: NULL argument");
  TPUHIP_REQUIRE(kind >= 0 && kind <= 3, "reduce: unknown kind %d", kind);
  TPUHIP_REQUIRE(first_axis >= 0 && first_axis <= last_axis && last_axis < 4, "reduce: axes %d..%d", first_axis,
                 last_axis);
  int64_t outer = 1, axis = 1, inner = 1, out_count = 1;
  for (int k = 0; k < 4; ++k) {
    TPUHIP_REQUIRE(in_nchw[k] > 0 && out_nchw[k] > 0, "reduce: non-positive dimension");
    (k < first_axis ? outer : k <= last_axis ? axis : inner) *= in_nchw[k];
    out_count *= out_nchw[k];
  }
  TPUHIP_REQUIRE(out_count == outer * inner, "reduce: the result holds %lld elements, expected %lld",
                 (long long)out_count, (long long)(outer * inner));
  TPUHIP_REQUIRE(x_cs >= in_nchw[1] && x_cs % 16 == 0 && y_cs >= out_nchw[1] && y_cs % 16 == 0,
                 "reduce: channel strides must be multiples of 16 covering the channels");
  TPUHIP_REQUIRE(outer * axis * inner < (1ll << 31) && axis * 128 < (1ll << 24),
                 "reduce: tensor too large (the reference's float sum must stay exact)");
  TPUHIP_REQUIRE(rshift >= 0 && rshift <= 30, "reduce: rshift %d outside [0,30]", rshift);
  const bool requant = rshift != 0 || multiplier != 1;
  TPUHIP_REQUIRE(requant || kind >= 2 || axis == 1,
                 "reduce: a sum with rshift 0 and multiplier 1 has no int8 value (the reference leaves "
                 "the raw sum in its float tensor)");
  TPUHIP_CHECK_HIP(hipSetDevice(ctx->device));
  ReduceArgs a{};
  a.x = (const int8_t *)x;
  a.y = (int8_t *)y;
  a.kind = kind;
  a.requant = requant ? 1 : 0;
  a.ic = in_nchw[1]; a.ih = in_nchw[2]; a.iw = in_nchw[3]; a.ics = x_cs;
  a.oc = out_nchw[1]; a.oh = out_nchw[2]; a.ow = out_nchw[3]; a.ocs = y_cs;
  a.axis = (int)axis;
  a.inner = (int)inner;
  a.mult = (float)multiplier;
  a.inv_pot = 1.0f / (float)(1u << rshift);
  a.total = (int64_t)out_nchw[0] * out_nchw[2] * out_nchw[3] * (y_cs / 4);
  const unsigned blocks = (unsigned)std::max<int64_t>(
      1, std::min<int64_t>(ceil_div64(a.total, kThreads), (int64_t)ctx->num_cu * 32));
  launch(ctx, reduce_kernel, dim3(blocks), dim3(kThreads), a);
  TPUHIP_CHECK_HIP(hipGetLastError());
  return TPUHIP_OK;
}

namespace {

// ---------------------------------------------------------------------------
// Permute without the per-byte index map.  S[k]: byte stride of input dimension k in the input,
// T[k]: byte stride, in the output, of the output dimension that input dimension k becomes.
// ---------------------------------------------------------------------------
struct PermRowsArgs {
  const int8_t *x;
  int8_t *y;
  int64_t S[3], T[3];   // of n, h and w
  FastDiv by_groups, by_w, by_h;
  int ics;              // channel stride of the input
  uint32_t total;       // input pixels * 16-byte groups of an output row, below 2^31
};

// channels stay channels (j == 1): a pixel's channel row moves as 16-byte chunks.  The two channel
// strides may differ (a padded stride on either side): groups of the output row beyond the input's
// stride are written as zero, never read from the next pixel.
__global__ __launch_bounds__(kThreads) void permute_rows_kernel(PermRowsArgs q) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= q.total) return;
  uint32_t cg = i, w = q.by_groups.split(cg), h = q.by_w.split(w);   // an input pixel, in input order
  const int64_t n = q.by_h.split(h);
  v4i v = {0, 0, 0, 0};
  if ((int)cg * 16 < q.ics) v = *reinterpret_cast<const v4i *>(q.x + n * q.S[0] + h * q.S[1] + w * q.S[2] + cg * 16);
  *reinterpret_cast<v4i *>(q.y + n * q.T[0] + h * q.T[1] + w * q.T[2] + cg * 16) = v;
}

// j: the input dimension that becomes the output's channels; a, b: the other two besides c
struct PermTileArgs {
  const int8_t *x;
  int8_t *y;
  int64_t Sj, Sa, Sb, Tc, Ta, Tb;
  FastDiv by_b;
  int dim_j, dim_c;
  int ocs;           // channel stride of the output
  uint32_t plane0;   // first of this launch's (a, b) pairs
  // RUNS: all tiles; narrow: FastDivs by the tiles of the channels and of j, wide: by the planes of this launch, which mul_j is
  uint32_t n_tiles, mul_c, shift_c, mul_j, shift_j;
};
static_assert(sizeof(PermRowsArgs) <= 112 && sizeof(PermTileArgs) <= 112, "see MovePlan");

// The channels change places with dimension j: tiles of 64 (Q 16) or 128 channels (32) x 64 of j, 4 x 4 bytes of a lane transposed
// in registers, dwords through LDS, so that the input is read in runs of 64 or 128 bytes and the output written in runs of 64 (its
// pad channels as zero: rows past the end of dimension j are zeros).
// RUNS: an XCD takes tiles that follow each other, since the parts of a line that lie in several tiles are fetched, and written,
// once for every L2 they meet in.  Narrow tiles: the channels of the same rows, then the next of j, then the next plane.  Wide ones,
// where j is one tile: the planes, then the next channels; the output's 16 to 32 bytes of a plane lie beside the next plane's.
// Else the grid is (j, channels, planes).
// Bound: by memory at size, where it reaches what a copy does (6.5 TB/s), by launch and one trip below.  To NHWC order, replayed from
// a graph, with bytes read from LDS and tiles of 64 in a grid / tiles of 128 in a grid / now: 4 x 80 x 96 x 96 4.31 / 3.42 / 3.46 us,
// 64 x 192 x 90 x 90 (205 MB) 56.8 / 68.2 / 29.7, 32 x 256 x 110 x 110 59.2 / 45.4 / 29.4, 1 x 256 x 62 x 62 2.87 / 2.77 / 2.45.
template <int Q, bool RUNS>
__global__ __launch_bounds__(kThreads) void permute_tile_kernel(PermTileArgs q) {
  __shared__ uint32_t tile[Q * 4 * 17];   // [channel][four of j]
  int c0 = blockIdx.y * (Q * 4), j0 = blockIdx.x * 64;
  uint32_t ib = q.plane0 + blockIdx.z;   // below 2^31, as all pixels are
  if constexpr (RUNS) {
    const uint32_t wt = (blockIdx.x & 7) * ((q.n_tiles + 7) >> 3) + (blockIdx.x >> 3);
    if (wt >= q.n_tiles) return;   // uniform over the workgroup
    if constexpr (Q == 16) {
      const uint32_t at_j = (__umulhi(wt, q.mul_c) + wt) >> q.shift_c, plane = (__umulhi(at_j, q.mul_j) + at_j) >> q.shift_j;
      c0 = (int)(wt - at_j * (uint32_t)((q.dim_c + 63) / 64)) * 64;
      j0 = (int)(at_j - plane * (uint32_t)((q.ocs + 63) / 64)) * 64;
      ib = q.plane0 + plane;
    } else {
      const uint32_t ct = (__umulhi(wt, q.mul_c) + wt) >> q.shift_c;
      c0 = (int)ct * 128;
      j0 = 0;
      ib = q.plane0 + wt - ct * q.mul_j;
    }
  }
  const int64_t ia = q.by_b.split(ib);
  const int8_t *src = q.x + ia * q.Sa + ib * q.Sb;
  int8_t *dst = q.y + ia * q.Ta + ib * q.Tb;
  constexpr int kPasses = 16 * Q / kThreads;
  const int cq = threadIdx.x % Q, cc = c0 + cq * 4;
  uint32_t r[kPasses][4];
  // the input's pad channels are zero and its channel stride is a multiple of 16, so a dword that starts inside the row may be
  // read whole
#pragma unroll
  for (int u = 0; u < kPasses; ++u)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int jj = j0 + (threadIdx.x / Q + u * (kThreads / Q)) * 4 + k;
      r[u][k] = jj < q.dim_j && cc < q.dim_c ? *reinterpret_cast<const uint32_t *>(src + jj * q.Sj + cc) : 0u;
    }
#pragma unroll
  for (int u = 0; u < kPasses; ++u) {
    uint32_t t[4];
    transpose_bytes(r[u], t);
#pragma unroll
    for (int k = 0; k < 4; ++k) tile[(cq * 4 + k) * 17 + threadIdx.x / Q + u * (kThreads / Q)] = t[k];
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < Q / 4; ++k) {
    const int row = threadIdx.x / 16 + k * 16, c = c0 + row, j = j0 + (threadIdx.x & 15) * 4;
    if (c < q.dim_c && j < q.ocs) *reinterpret_cast<uint32_t *>(dst + c * q.Tc + j) = tile[row * 17 + (threadIdx.x & 15)];
  }
}

// permute of dense row-major bytes over the full rank (at most 6): a lane owns an output element
struct FlatPermArgs {
  const int8_t *x;
  int8_t *y;
  int rank;
  int oshape[6];
  int64_t istr[6];   // input stride of the input dimension that output dimension d is
  int64_t total;
};
__global__ __launch_bounds__(kThreads) void permute_flat_kernel(FlatPermArgs q) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < q.total; i += (int64_t)gridDim.x * blockDim.x) {
    int64_t r = i, off = 0;
    for (int d = q.rank - 1; d >= 0; --d) {
      const int64_t c = r % q.oshape[d];
      r /= q.oshape[d];
      off += c * q.istr[d];
    }
    q.y[i] = q.x[off];
  }
}

// S[k]: byte stride of input dimension k in the input, T[k]: byte stride, in the output, of the output dimension that input
// dimension k becomes
int run_permute(tpuhip_ctx *ctx, const tpuhip_move_desc *d, const void *x, void *y) {
  const int dim[4] = {d->in, d->ic, d->ih, d->iw};
  const int64_t S[4] = {(int64_t)d->ih * d->iw * d->x_cs, 1, (int64_t)d->iw * d->x_cs, d->x_cs};
  const int64_t tout[4] = {(int64_t)d->oh * d->ow * d->y_cs, 1, (int64_t)d->ow * d->y_cs, d->y_cs};
  int64_t T[4];
  for (int k = 0; k < 4; ++k) T[d->p[k]] = tout[k];   // output dimension k is input dimension p[k]
  const int j = d->p[1];
  TPUHIP_CHECK_HIP(hipSetDevice(ctx->device));
  if (j == 1) {
    PermRowsArgs q{(const int8_t *)x, (int8_t *)y, {S[0], S[2], S[3]}, {T[0], T[2], T[3]}, FastDiv(d->y_cs / 16), FastDiv(d->iw),
                   FastDiv(d->ih), d->x_cs, 0};
    const int64_t image = (int64_t)d->ih * d->iw * (d->y_cs / 16);
    TPUHIP_REQUIRE(image < (1ll << 31), "permute: an image of 2^31 16-byte groups or more");
    const int most = (int)std::min<int64_t>(((1ll << 31) - 1) / image, d->in);   // images a 31-bit index reaches
    for (int left = d->in; left > 0; left -= most) {
      q.total = (uint32_t)(image * std::min(left, most));
      launch(ctx, permute_rows_kernel, dim3((unsigned)ceil_div64(q.total, kThreads)), dim3(kThreads), q);
      q.x += most * S[0];
      q.y += most * T[0];
    }
  } else {
    int rest[2], nr = 0;
    for (int k = 0; k < 4; ++k)
      if (k != 1 && k != j) rest[nr++] = k;
    const int a = rest[0], b = rest[1];
    PermTileArgs q{(const int8_t *)x, (int8_t *)y, S[j], S[a], S[b], T[1], T[a], T[b], FastDiv(dim[b]), dim[j], dim[1], d->y_cs, 0};
    const int64_t planes = (int64_t)dim[a] * dim[b];
    const int tiles_j = (d->y_cs + 63) / 64;
    // Wide tiles where j is so short that a narrow one is half empty at least, and there are four a CU: from a graph, narrow and
    // wide, order (1, 0, 2, 3), 1 x 80 x 111 x 111 17.6 and 12.9 us, 1 x 256 x 108 x 108 34.2 and 24, 1 x 100 x 14 x 14 2.43 and 2.70;
    // 64 x 128 x 110 x 110 30.7 and 32.5.
    const bool wide = d->ic > 64 && d->y_cs <= 32 && planes * ((d->ic + 63) / 64) >= 4 * (int64_t)ctx->num_cu;
    const int tiles_c = (d->ic + (wide ? 127 : 63)) / (wide ? 128 : 64);
    // In a grid as it is: a single tile of channels, whose lines end with it, for fewer instructions (512 x 16 x 110 x 110, order
    // (0, 3, 1, 2): 61 us, 73 in runs); wide tiles that come in whole rounds of the XCDs, which share the channels so by themselves
    // (8 x 1024 x 110 x 110, order (1, 0, 2, 3): 97 and 130).
    const bool runs = wide ? tiles_c % 8 != 0 : d->ic > 64;
    const int64_t most = runs ? std::max<int64_t>(1, (1ll << 30) / ((int64_t)tiles_j * tiles_c)) : 65535;   // planes of a launch
    for (int64_t p0 = 0; p0 < planes; p0 += most) {
      const uint32_t now = (uint32_t)std::min(most, planes - p0);
      q.plane0 = (uint32_t)p0;
      q.n_tiles = now * tiles_j * tiles_c;
      const FastDiv by_c(wide ? now : tiles_c), by_j(tiles_j);
      q.mul_c = by_c.mul; q.shift_c = by_c.shift;
      q.mul_j = wide ? now : by_j.mul; q.shift_j = by_j.shift;
      const dim3 grid = runs ? dim3((q.n_tiles + 7) / 8 * 8) : dim3((unsigned)tiles_j, (unsigned)tiles_c, now);
      launch(ctx, wide ? runs ? permute_tile_kernel<32, true> : permute_tile_kernel<32, false>
                       : runs ? permute_tile_kernel<16, true> : permute_tile_kernel<16, false>, grid, dim3(kThreads), q);
    }
  }
  TPUHIP_CHECK_HIP(hipGetLastError());
  return TPUHIP_OK;
}

}  // namespace

extern "C" int tpuhip_move_i8(tpuhip_ctx *ctx, const tpuhip_move_desc *d, const void *x, void *y) {
  TPUHIP_REQUIRE(ctx && d && x && y, "move: NULL argument");
  TPUHIP_REQUIRE(d->kind >= TPUHIP_MOVE_PAD_CONST && d->kind <= TPUHIP_MOVE_REFLECTION_PAD,
                 "move: unknown kind %d", d->kind);
  TPUHIP_REQUIRE(d->in > 0 && d->ic > 0 && d->ih > 0 && d->iw > 0 && d->on > 0 && d->oc > 0 &&
                     d->oh > 0 && d->ow > 0,
                 "move: non-positive dimension");
  TPUHIP_REQUIRE(d->x_cs >= d->ic && d->x_cs % 16 == 0 && d->y_cs >= d->oc && d->y_cs % 16 == 0,
                 "move: channel strides must be multiples of 16 covering the channels");
  TPUHIP_REQUIRE((int64_t)d->in * d->ih * d->iw * d->x_cs < (1ll << 31) &&
                     (int64_t)d->on * d->oh * d->ow < (1ll << 31),
                 "move: tensor too large");
  const int is[4] = {d->in, d->ic, d->ih, d->iw}, os[4] = {d->on, d->oc, d->oh, d->ow};
  const int *p = d->p;
  MovePlan a{};
  Form form = kPadConst;
  // every kind: check that the map stays inside the input for every output element
  switch (d->kind) {
    case TPUHIP_MOVE_PAD_CONST:
      // p[0..3] pads at the beginning, p[4..7] at the end (negative: cut), as the op's attribute
      for (int k = 0; k < 4; ++k) {
        TPUHIP_REQUIRE(os[k] == is[k] + p[k] + p[4 + k], "pad: output dimension %d is %d, expected %d",
                       k, os[k], is[k] + p[k] + p[4 + k]);
        a.p[k] = p[k] < 0 ? 0 : p[k];
        a.p[4 + k] = p[k] < 0 ? -p[k] : 0;
        a.p[8 + k] = p[4 + k] < 0 ? is[k] + p[4 + k] : is[k];
        TPUHIP_REQUIRE(a.p[4 + k] <= a.p[8 + k], "pad: dimension %d is cut away entirely", k);
        if (p[k] < 0 || p[4 + k] < 0) form = kPadCut;
      }
      if (form == kPadConst) a.p[4] = is[0];
      break;
    case TPUHIP_MOVE_PAD_EDGE:
      TPUHIP_REQUIRE(p[0] == 0 && p[1] == 0 && p[4] == 0 && p[5] == 0, "pad: edge mode pads h and w only");
      TPUHIP_REQUIRE(p[2] >= 0 && p[3] >= 0 && p[6] >= 0 && p[7] >= 0, "pad: edge mode needs pads >= 0");
      for (int k = 0; k < 4; ++k) {
        TPUHIP_REQUIRE(os[k] == is[k] + p[k] + p[4 + k], "pad: output dimension %d is %d, expected %d",
                       k, os[k], is[k] + p[k] + p[4 + k]);
        a.p[k] = p[k];
      }
      form = kPadEdge;
      break;
    case TPUHIP_MOVE_CROP:
      // p[0..3] offsets, p[4..7] steps
      for (int k = 0; k < 4; ++k) {
        TPUHIP_REQUIRE(p[k] >= 0 && p[4 + k] >= 1 && (int64_t)(os[k] - 1) * p[4 + k] + p[k] < is[k],
                       "crop: dimension %d reads past the input", k);
        a.p[k] = p[k];
        a.p[4 + k] = p[4 + k];
      }
      form = p[5] == 1 ? kCrop : kStrided;
      break;
    case TPUHIP_MOVE_PERMUTE: {
      int seen = 0;
      for (int k = 0; k < 4; ++k) {
        TPUHIP_REQUIRE(p[k] >= 0 && p[k] < 4, "permute: order[%d] = %d", k, p[k]);
        seen |= 1 << p[k];
        TPUHIP_REQUIRE(os[k] == is[p[k]], "permute: output dimension %d is %d, expected %d", k, os[k],
                       is[p[k]]);
      }
      TPUHIP_REQUIRE(seen == 15, "permute: order is not a permutation");
      return run_permute(ctx, d, x, y);
    }
    case TPUHIP_MOVE_REORG:
      TPUHIP_REQUIRE(p[0] >= 1 && is[2] % p[0] == 0 && is[3] % p[0] == 0, "reorg: bad stride %d", p[0]);
      TPUHIP_REQUIRE(os[0] == is[0] && os[1] == is[1] * p[0] * p[0] && os[2] == is[2] / p[0] &&
                         os[3] == is[3] / p[0],
                     "reorg: output shape does not match");
      a.p[0] = p[0];
      a.by_a = FastDiv(is[1]);
      a.by_b = FastDiv(p[0]);
      form = kReorg;
      break;
    case TPUHIP_MOVE_TILE:
      TPUHIP_REQUIRE(p[0] >= 0 && p[0] < 4 && p[1] >= 1, "tile: bad axis %d / tiles %d", p[0], p[1]);
      for (int k = 0; k < 4; ++k)
        TPUHIP_REQUIRE(os[k] == (k == p[0] ? is[k] * p[1] : is[k]), "tile: output dimension %d is %d", k,
                       os[k]);
      a.by_a = FastDiv(is[p[0] == 1 ? 1 : 0]);
      a.by_b = FastDiv(is[2]);
      a.by_c = FastDiv(is[3]);
      form = p[0] == 1 ? kTileChannel : kTile;
      break;
    case TPUHIP_MOVE_REVERSE:
      TPUHIP_REQUIRE(p[0] >= 0 && p[0] < 4, "reverse: bad axis %d", p[0]);
      for (int k = 0; k < 4; ++k) TPUHIP_REQUIRE(os[k] == is[k], "reverse: shapes differ");
      a.p[0] = p[0];
      form = p[0] == 1 ? kReverseChannel : kReverse;
      break;
    case TPUHIP_MOVE_SHUFFLE_CHANNEL:
      TPUHIP_REQUIRE(p[0] >= 1 && is[1] % p[0] == 0, "shuffle_channel: wrong group size, c=%d, group=%d",
                     is[1], p[0]);
      for (int k = 0; k < 4; ++k) TPUHIP_REQUIRE(os[k] == is[k], "shuffle_channel: shapes differ");
      a.p[1] = is[1] / p[0];
      a.by_a = FastDiv(p[0]);
      form = p[0] == 2 || p[0] == 4 ? kWeave : kShuffle;
      break;
    case TPUHIP_MOVE_SWAP_CHANNEL:
      TPUHIP_REQUIRE(is[1] <= 8, "swap_channel: at most 8 channels (%d)", is[1]);
      for (int k = 0; k < 4; ++k) TPUHIP_REQUIRE(os[k] == is[k], "swap_channel: shapes differ");
      for (int k = 0; k < is[1]; ++k) {
        TPUHIP_REQUIRE(p[k] >= 0 && p[k] < is[1], "swap_channel: channel_order[%d] = %d", k, p[k]);
        a.p[k] = p[k];
      }
      form = kSwap;
      break;
    case TPUHIP_MOVE_DILATE:
      // p[0] = ins_w, p[1] = ins_h, p[2] = fill_constant
      TPUHIP_REQUIRE(p[0] >= 0 && p[1] >= 0, "dilate: negative ins (%d, %d)", p[0], p[1]);
      TPUHIP_REQUIRE(p[2] >= -128 && p[2] <= 127, "dilate: fill_constant %d is no int8 value", p[2]);
      TPUHIP_REQUIRE(os[0] == is[0] && os[1] == is[1] &&
                         (int64_t)os[2] == (int64_t)(is[2] - 1) * (p[1] + 1) + 1 &&
                         (int64_t)os[3] == (int64_t)(is[3] - 1) * (p[0] + 1) + 1,
                     "dilate: output shape does not match");
      a.by_a = FastDiv((int64_t)p[0] + 1);
      a.by_b = FastDiv((int64_t)p[1] + 1);
      a.fill = p[2];
      form = kDilate;
      break;
    case TPUHIP_MOVE_REFLECTION_PAD:
      // p[0] / p[1] columns added on the left / right; a mirror image needs a column to mirror
      TPUHIP_REQUIRE(p[0] >= 0 && p[1] >= 0 && p[0] < is[3] && p[1] < is[3],
                     "reflection_pad: pads (%d, %d) must be in [0, w = %d)", p[0], p[1], is[3]);
      TPUHIP_REQUIRE(os[0] == is[0] && os[1] == is[1] && os[2] == is[2] && os[3] == is[3] + p[0] + p[1],
                     "reflection_pad: output shape does not match");
      a.p[0] = p[0];
      form = kReflectionPad;
      break;
    default:
      TPUHIP_REQUIRE(p[0] >= 1 && is[1] % (p[0] * p[0]) == 0, "depth_to_space: bad upscale factor %d", p[0]);
      TPUHIP_REQUIRE(os[0] == is[0] && os[1] == is[1] / (p[0] * p[0]) && os[2] == is[2] * p[0] &&
                         os[3] == is[3] * p[0],
                     "depth_to_space: output shape does not match");
      a.p[0] = p[0];
      a.p[8] = 1;
      a.by_a = FastDiv(p[0]);
      form = p[1] ? kDepthDcr : kStrided;
      break;
  }
  TPUHIP_CHECK_HIP(hipSetDevice(ctx->device));
  a.x = (const int8_t *)x; a.y = (int8_t *)y;
  a.in = d->in; a.ic = d->ic; a.ih = d->ih; a.iw = d->iw; a.ics = d->x_cs;
  a.on = d->on; a.oc = d->oc; a.oh = d->oh; a.ow = d->ow; a.ocs = d->y_cs;
  a.by_groups = FastDiv(d->y_cs / 16);
  a.by_ow = FastDiv(d->ow);
  a.by_oh = FastDiv(d->oh);
  auto run = [&](auto args, auto *kernel, int64_t pixels) {
    args.x = a.x; args.y = a.y; args.ih = a.ih; args.iw = a.iw; args.ics = a.ics; args.oc = a.oc;
    args.by_groups = a.by_groups; args.by_ow = a.by_ow; args.by_oh = a.by_oh;
    args.take(a);
    const int64_t most = ((1ll << 31) - 1) / a.by_groups.d;   // as many pixels as the 31-bit index reaches
    for (int64_t p0 = 0; p0 < pixels; p0 += most) {
      args.pix0 = (uint32_t)p0;
      args.total = (uint32_t)(std::min(most, pixels - p0) * a.by_groups.d);
      launch(ctx, kernel, dim3((unsigned)ceil_div64(args.total, kThreads)), dim3(kThreads), args);
    }
  };
  const int64_t pixels = (int64_t)d->on * d->oh * d->ow;
  if (d->kind == TPUHIP_MOVE_DEPTH_TO_SPACE && form == kStrided && d->p[0] == 2) {   // the factor in use, a dword per channel
    a.by_ow = FastDiv(d->iw);
    run(MoveWith<MoveTailDepth>(), depth_by_two_kernel, (int64_t)d->in * d->ih * d->iw);
  } else {
    switch (form) {
#define TPUHIP_MOVE_FORM(F) case F: run(MoveArgs<F>(), move_kernel<F>, pixels); break
      TPUHIP_MOVE_FORM(kPadConst);
      TPUHIP_MOVE_FORM(kPadCut);
      TPUHIP_MOVE_FORM(kPadEdge);
      TPUHIP_MOVE_FORM(kCrop);
      TPUHIP_MOVE_FORM(kReorg);
      TPUHIP_MOVE_FORM(kTile);
      TPUHIP_MOVE_FORM(kTileChannel);
      TPUHIP_MOVE_FORM(kReverse);
      TPUHIP_MOVE_FORM(kDilate);
      TPUHIP_MOVE_FORM(kReflectionPad);
      TPUHIP_MOVE_FORM(kDepthDcr);
      TPUHIP_MOVE_FORM(kReverseChannel);
      TPUHIP_MOVE_FORM(kShuffle);
      TPUHIP_MOVE_FORM(kWeave);
      TPUHIP_MOVE_FORM(kSwap);
      TPUHIP_MOVE_FORM(kStrided);
#undef TPUHIP_MOVE_FORM
    }
  }
  TPUHIP_CHECK_HIP(hipGetLastError());
  return TPUHIP_OK;
}

extern "C" int tpuhip_permute_flat_i8(tpuhip_ctx *ctx, const void *x, void *y, int rank, const int64_t *in_shape,
                                      const int *order) {
  TPUHIP_REQUIRE(ctx && x && y && in_shape && order, "permute_flat: NULL argument");
  TPUHIP_REQUIRE(rank >= 1 && rank <= 6, "permute_flat: rank %d outside [1,6]", rank);
  FlatPermArgs q{};
  q.x = (const int8_t *)x;
  q.y = (int8_t *)y;
  q.rank = rank;
  int64_t istride[6], total = 1;
  int seen = 0;
  for (int d = rank - 1; d >= 0; --d) {
    TPUHIP_REQUIRE(in_shape[d] >= 1 && in_shape[d] < (1ll << 31), "permute_flat: bad dimension %d", d);
    istride[d] = total;
    total *= in_shape[d];
  }
  TPUHIP_REQUIRE(total < (1ll << 31), "permute_flat: tensor too large");
  for (int d = 0; d < rank; ++d) {
    TPUHIP_REQUIRE(order[d] >= 0 && order[d] < rank, "permute_flat: order[%d] = %d", d, order[d]);
    seen |= 1 << order[d];
    q.oshape[d] = (int)in_shape[order[d]];
    q.istr[d] = istride[order[d]];
  }
  TPUHIP_REQUIRE(seen == (1 << rank) - 1, "permute_flat: order is not a permutation");
  q.total = total;
  TPUHIP_CHECK_HIP(hipSetDevice(ctx->device));
  const unsigned blocks = (unsigned)std::max<int64_t>(
      1, std::min<int64_t>(ceil_div64(total, kThreads), (int64_t)ctx->num_cu * 32));
  launch(ctx, permute_flat_kernel, dim3(blocks), dim3(kThreads), q);
  TPUHIP_CHECK_HIP(hipGetLastError());
  return TPUHIP_OK;
}
