// INT8 max / average pooling for gfx950, channels-last: one lane owns 16
// channels of one output pixel (16-byte loads and stores).  Bandwidth-bound,
// no MFMA.
#include "common.hpp"

#include <algorithm>
#include <type_traits>

using namespace tpuhip;

typedef int v4i __attribute__((ext_vector_type(4)));

namespace {

struct PoolArgs {   // up to 112 bytes: a launch with more of arguments costs the host 0.5 us more
  const int8_t *x;
  int8_t *y;
  int ih, iw, kh, kw, sh, sw, pt, pl, x_cs, y_cs;
  float mult;       // (float)multiplier
  float inv_pot;    // 2^-rshift
  FastDiv by_c16, by_ow, by_oh;
  uint32_t total;   // 16-channel groups of all output pixels, below 2^31 (each_part)
  __host__ __device__ int c16() const { return (int)by_c16.d; }
  __host__ __device__ int oh() const { return (int)by_oh.d; }
  __host__ __device__ int ow() const { return (int)by_ow.d; }
};
static_assert(sizeof(PoolArgs) <= 112, "see above");

__device__ __forceinline__ int32_t sb(int32_t word, int i) {
  return (int32_t)(int8_t)(word >> (8 * i));
}

// Workgroups are dealt to the 8 XCDs round-robin.  With a grid that is a multiple of 8 this
// renumbering gives every XCD a contiguous run of logical blocks, i.e. of output rows, so the
// input rows that neighbouring windows share are fetched into one L2 instead of several.
__device__ __forceinline__ unsigned xcd_block() {
  return (blockIdx.x & 7u) * (gridDim.x >> 3) + (blockIdx.x >> 3);
}

// The window positions of a thread's output group.  K > 0: a K x K window, whose loads are all requested before one is
// used; one after the other behind their bounds checks, the nine of a 3 x 3 window took 5.7 us on 4 x 120 x 75 x 75, 3.9
// now.  For a max, a position outside the image is the nearest one inside, which belongs to the window as well; for a sum
// it is zero.
template <int K, bool MAX, class F>
__device__ __forceinline__ void each_tap(const PoolArgs &a, int b, int oh, int ow, int cg, F fn) {
  const int8_t *base = a.x + (int64_t)b * a.ih * a.iw * a.x_cs + cg * 16;
  if constexpr (K > 0) {
    v4i v[K * K];
#pragma unroll
    for (int kh = 0; kh < K; ++kh)
#pragma unroll
      for (int kw = 0; kw < K; ++kw) {
        const int ih = oh * a.sh - a.pt + kh, iw = ow * a.sw - a.pl + kw;
        const int h = min(max(ih, 0), a.ih - 1), w = min(max(iw, 0), a.iw - 1);
        v4i t = *reinterpret_cast<const v4i *>(base + ((int64_t)h * a.iw + w) * a.x_cs);
        if (!MAX && (h != ih || w != iw)) t = v4i{0, 0, 0, 0};
        v[kh * K + kw] = t;
      }
#pragma unroll
    for (int t = 0; t < K * K; ++t) fn(v[t]);
  } else {
    for (int kh = 0; kh < a.kh; ++kh) {
      const int ih = oh * a.sh - a.pt + kh;
      if (ih < 0 || ih >= a.ih) continue;
      for (int kw = 0; kw < a.kw; ++kw) {
        const int iw = ow * a.sw - a.pl + kw;
        if (iw < 0 || iw >= a.iw) continue;
        fn(*reinterpret_cast<const v4i *>(base + ((int64_t)ih * a.iw + iw) * a.x_cs));
      }
    }
  }
}

// PoolingOpKernel INT8 max (core/pooling.cpp:155-157): MKL-DNN pooling_max skips
// padded positions.  Bytes compare as the upper halves of 16-bit words.
template <int K>
__global__ __launch_bounds__(256) void pool_max_kernel(PoolArgs a) {
  typedef short v2s __attribute__((ext_vector_type(2)));
  for (uint32_t i = xcd_block() * 256 + threadIdx.x; i < a.total; i += gridDim.x * 256) {
    uint32_t cg = i, ow = a.by_c16.split(cg), oh = a.by_ow.split(ow);
    const int b = (int)a.by_oh.split(oh);
    v2s best[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) best[k] = v2s{-32768, -32768};
    each_tap<K, true>(a, b, (int)oh, (int)ow, (int)cg, [&](v4i v) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const uint32_t word = (uint32_t)v[q];
        best[q * 2] = __builtin_elementwise_max(best[q * 2], __builtin_bit_cast(v2s, word << 8));
        best[q * 2 + 1] = __builtin_elementwise_max(best[q * 2 + 1], __builtin_bit_cast(v2s, word));
      }
    });
    v4i out;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      out[q] = (int)((__builtin_bit_cast(uint32_t, best[q * 2]) >> 8 & 0x00ff00ffu) |
                     (__builtin_bit_cast(uint32_t, best[q * 2 + 1]) & 0xff00ff00u));
    *reinterpret_cast<v4i *>(a.y + ((int64_t)(b * a.oh() + oh) * a.ow() + ow) * a.y_cs + cg * 16) = out;
  }
}

// PoolingOpKernel INT8 average, normal path (core/pooling.cpp:147-154): window
// sum with zero padding, then the float overload of
// applyMultiplierAndRShiftAndSaturateInt8 without qdm: float product, float
// quotient by a power of two, floor(f + 0.5), clamp.
template <int K>
__global__ __launch_bounds__(256) void pool_avg_kernel(PoolArgs a) {
  for (uint32_t i = xcd_block() * 256 + threadIdx.x; i < a.total; i += gridDim.x * 256) {
    uint32_t cg = i, ow = a.by_c16.split(cg), oh = a.by_ow.split(ow);
    const int b = (int)a.by_oh.split(oh);
    int32_t sum[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) sum[k] = 0;
    each_tap<K, false>(a, b, (int)oh, (int)ow, (int)cg, [&](v4i v) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int k = 0; k < 4; ++k) sum[q * 4 + k] += sb(v[q], k);
    });
    v4i out;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t w = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float prod = __fmul_rn((float)sum[q * 4 + k], a.mult);
        const float quo = __fmul_rn(prod, a.inv_pot);  // exact: power-of-two scaling
        w |= ((uint32_t)saturate_int8_f(quo) & 0xffu) << (8 * k);
      }
      out[q] = (int)w;
    }
    *reinterpret_cast<v4i *>(a.y + ((int64_t)(b * a.oh() + oh) * a.ow() + ow) * a.y_cs + cg * 16) = out;
  }
}

// Average pooling over windows of 16 to 64 positions: eight lanes share one (pixel, 16-channel group) output, each sums every
// eighth window position, and the partial sums meet by DPP, every lane finishing two channels.  Keeps enough loads in flight when
// there are few outputs (a 7x7 global pool has 49 taps per output and only n*c/16 outputs).  Bound by the chain of a wave that is
// alone on its SIMD, eight clocks an instruction: launch, one trip for up to eight positions, their adds, the requantisation.
// From a graph, against 48 wave shuffles and one lane of eight that finished 16 channels: 1 x 2048 x 7 x 7 4.42 -> 2.70 us, 64 x
// 1280 x 7 x 7 4.76 -> 2.90, 1 x 512 x 4 x 4 3.70 -> 2.32, 400 x 2048 x 7 x 7 (40 MB) 11.3 -> 8.4.
__global__ __launch_bounds__(256) void pool_avg_split_kernel(PoolArgs a, FastDiv by_kw) {
  constexpr int LANES = 8;
  const int64_t gid = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / LANES;
  const int sub = threadIdx.x % LANES;
  const bool live = gid < a.total;
  uint32_t cg = live ? (uint32_t)gid : 0, ow = a.by_c16.split(cg), oh = a.by_ow.split(ow);
  const int b = (int)a.by_oh.split(oh);
  int32_t sum[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) sum[k] = 0;
  const int taps = a.kh * a.kw;   // 64 at most, all of a lane's requested before any is added
  constexpr int MAXT = 64 / LANES;
  v4i v[MAXT];
#pragma unroll
  for (int u = 0; u < MAXT; ++u) {
    const int t = sub + u * LANES;
    uint32_t kw = (uint32_t)t;
    const int kh = (int)by_kw.split(kw);
    const int ih = (int)oh * a.sh - a.pt + kh, iw = (int)ow * a.sw - a.pl + (int)kw;
    const bool ok = (t < taps) & ((unsigned)ih < (unsigned)a.ih) & ((unsigned)iw < (unsigned)a.iw);
    v[u] = v4i{0, 0, 0, 0};
    if (ok)
      v[u] = *reinterpret_cast<const v4i *>(a.x + ((int64_t)(b * a.ih + ih) * a.iw + iw) * a.x_cs + cg * 16);
  }
#pragma unroll
  for (int u = 0; u < MAXT; ++u)
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int k = 0; k < 4; ++k) sum[q * 4 + k] = __builtin_amdgcn_sdot4(v[u][q], 1 << (8 * k), sum[q * 4 + k], false);
  // A lane keeps the half of the channels that it will finish and hands the other to the lane that keeps that one: mirrored
  // within the eight, two away, one away.  Lane `sub` ends with channels 2 * sub and 2 * sub + 1.
  auto halve = [&](auto n, auto ctrl, bool upper) {
    constexpr int N = decltype(n)::value;
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const int32_t keep = upper ? sum[N + k] : sum[k], give = upper ? sum[k] : sum[N + k];
      sum[k] = keep + __builtin_amdgcn_update_dpp(0, give, decltype(ctrl)::value, 0xf, 0xf, true);
    }
  };
  halve(std::integral_constant<int, 8>(), std::integral_constant<int, 0x141>(), sub & 4);   // row_half_mirror
  halve(std::integral_constant<int, 4>(), std::integral_constant<int, 0x4e>(), sub & 2);    // quad_perm 2, 3, 0, 1
  halve(std::integral_constant<int, 2>(), std::integral_constant<int, 0xb1>(), sub & 1);    // quad_perm 1, 0, 3, 2
  if (live) {
    uint32_t w = 0;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const float prod = __fmul_rn((float)sum[k], a.mult);
      const float quo = __fmul_rn(prod, a.inv_pot);
      w |= ((uint32_t)saturate_int8_f(quo) & 0xffu) << (8 * k);
    }
    *reinterpret_cast<uint16_t *>(a.y + ((int64_t)(b * a.oh() + oh) * a.ow() + ow) * a.y_cs + cg * 16 + 2 * sub) = (uint16_t)w;
  }
}

// Global average of a large map, few outputs with thousands of window positions each: a workgroup takes G 16-channel groups
// of an output pixel (lanes along the channels, so that a wave reads whole lines) and one slice of the window, 256 / G lanes
// deep, four positions in flight per lane; the lanes' sums meet in LDS.  With more than one slice the sums go to `parts`
// [output][slice][channel] and pool_avg_finish_kernel adds them.  A 75 x 75 window over 4 x 120 channels: 113 us with the
// kernel above (its eight lanes walk 700 positions each, one workgroup), 7 us with 32 slices.
template <int G>
__global__ __launch_bounds__(256) void pool_avg_window_kernel(PoolArgs a, FastDiv by_kw, int32_t *parts, int slices, int per_slice,
                                                              FastDiv by_slices, FastDiv by_blocks) {
  constexpr int P = 256 / G;
  __shared__ __attribute__((aligned(16))) int32_t lds[256 * 16];
  uint32_t slice = blockIdx.x, gb = by_slices.split(slice), pix = by_blocks.split(gb);
  uint32_t ow = pix, oh = a.by_ow.split(ow);
  const int b = (int)a.by_oh.split(oh);
  const int cl = threadIdx.x % G, row = threadIdx.x / G, cg = (int)gb * G + cl;
  int32_t sum[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) sum[k] = 0;
  const int end = min(((int)slice + 1) * per_slice, a.kh * a.kw);
  if (cg < a.c16()) {
    for (int t0 = (int)slice * per_slice + row; t0 < end; t0 += 4 * P) {
      v4i v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int t = t0 + u * P;
        uint32_t kw = (uint32_t)t;
        const int kh = (int)by_kw.split(kw);
        const int ih = (int)oh * a.sh - a.pt + kh, iw = (int)ow * a.sw - a.pl + (int)kw;
        v[u] = v4i{0, 0, 0, 0};
        if ((t < end) & ((unsigned)ih < (unsigned)a.ih) & ((unsigned)iw < (unsigned)a.iw))
          v[u] = *reinterpret_cast<const v4i *>(a.x + ((int64_t)(b * a.ih + ih) * a.iw + iw) * a.x_cs + cg * 16);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int k = 0; k < 4; ++k) sum[q * 4 + k] += sb(v[u][q], k);
    }
  }
  // P rows of G * 16 sums: each of the 16 / G parts adds 16 rows, then the first adds the parts
#pragma unroll
  for (int q = 0; q < 4; ++q)
    *reinterpret_cast<v4i *>(lds + (row * G + cl) * 16 + q * 4) = v4i{sum[q * 4], sum[q * 4 + 1], sum[q * 4 + 2], sum[q * 4 + 3]};
  __syncthreads();
  const int ch = threadIdx.x % (G * 16), part = threadIdx.x / (G * 16);
  int32_t s = 0;
#pragma unroll
  for (int r = 0; r < 16; ++r) s += lds[(part * 16 + r) * G * 16 + ch];
  if constexpr (G < 16) {
    __syncthreads();
    lds[threadIdx.x] = s;
    __syncthreads();
    if (part) return;
#pragma unroll
    for (int r = 1; r < 16 / G; ++r) s += lds[r * G * 16 + ch];
  }
  const int c = (int)gb * G * 16 + ch;
  if (c >= a.c16() * 16) return;
  if (parts)
    parts[((int64_t)pix * slices + slice) * (a.c16() * 16) + c] = s;
  else
    a.y[(int64_t)pix * a.y_cs + c] = (int8_t)saturate_int8_f(__fmul_rn(__fmul_rn((float)s, a.mult), a.inv_pot));
}

// adds the slices of pool_avg_window_kernel: 64 channels of an output pixel per workgroup, four threads per channel
struct FinishArgs {
  const int32_t *parts;
  int8_t *y;
  int slices, channels, y_cs;
  float mult, inv_pot;
};
__global__ __launch_bounds__(256) void pool_avg_finish_kernel(FinishArgs a) {
  __shared__ int32_t lds[256];
  const int c = blockIdx.x * 64 + (threadIdx.x & 63), part = threadIdx.x >> 6, all = a.channels;
  int32_t s = 0;
  if (c < all) {
#pragma unroll 8
    for (int k = part; k < a.slices; k += 4) s += a.parts[((int64_t)blockIdx.y * a.slices + k) * all + c];
  }
  lds[threadIdx.x] = s;
  __syncthreads();
  if (part || c >= all) return;
  s += lds[c % 64 + 64] + lds[c % 64 + 128] + lds[c % 64 + 192];
  a.y[(int64_t)blockIdx.y * a.y_cs + c] = (int8_t)saturate_int8_f(__fmul_rn(__fmul_rn((float)s, a.mult), a.inv_pot));
}

// more than 64 window positions for few outputs
int run_window(tpuhip_ctx *ctx, const PoolArgs &a) {
  const int c16 = a.c16();
  const int G = c16 >= 16 ? 16 : c16 > 4 ? 8 : c16 > 2 ? 4 : c16;
  const int gblocks = (c16 + G - 1) / G, taps = a.kh * a.kw;
  const int64_t pixels = a.total / c16, blocks = pixels * gblocks;
  // two workgroups per CU, while every lane keeps four positions; no slices where the grid of the second launch does not
  // reach or there is no memory, nor in a recorded launch: a graph may outlive this context's workspace, or replay beside
  // another one
  int64_t slices = std::min<int64_t>(std::min<int64_t>(2 * ctx->num_cu / blocks, taps / (4 * 256 / G)), 32);
  if (slices < 2 || pixels > 65535) slices = 1;
  if (slices > 1) {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    TPUHIP_CHECK_HIP(hipStreamIsCapturing(ctx->stream, &capture));
    const int rc = capture != hipStreamCaptureStatusNone
                       ? TPUHIP_ERR_NOMEM
                       : grow_workspace(ctx, (size_t)(pixels * slices * c16 * 16) * sizeof(int32_t));
    if (rc == TPUHIP_ERR_NOMEM) slices = 1;
    else if (rc) return rc;
  }
  int32_t *parts = slices > 1 ? (int32_t *)ctx->workspace : nullptr;
  const int per_slice = (int)((taps + slices - 1) / slices);
  auto *kernel = G == 16 ? pool_avg_window_kernel<16> : G == 8 ? pool_avg_window_kernel<8> : G == 4 ? pool_avg_window_kernel<4>
                 : G == 2 ? pool_avg_window_kernel<2> : pool_avg_window_kernel<1>;
  launch(ctx, kernel, dim3((unsigned)(blocks * slices)), dim3(256), a, FastDiv(a.kw), parts, (int)slices, per_slice,
         FastDiv(slices), FastDiv(gblocks));
  if (parts)
    launch(ctx, pool_avg_finish_kernel, dim3((unsigned)((c16 + 3) / 4), (unsigned)pixels), dim3(256),
           FinishArgs{parts, a.y, (int)slices, c16 * 16, a.y_cs, a.mult, a.inv_pot});
  TPUHIP_CHECK_HIP(hipGetLastError());
  return TPUHIP_OK;
}

int fill_args(const tpuhip_pool_desc *d, const void *x, void *y, PoolArgs *a) {
  TPUHIP_REQUIRE(d && x && y, "pool: NULL argument");
  TPUHIP_REQUIRE(d->n > 0 && d->c > 0 && d->ih > 0 && d->iw > 0 && d->oh > 0 && d->ow > 0 &&
                     d->kh > 0 && d->kw > 0 && d->sh > 0 && d->sw > 0,
                 "pool: non-positive dimension");
  TPUHIP_REQUIRE(d->pt >= 0 && d->pb >= 0 && d->pl >= 0 && d->pr >= 0, "pool: negative padding");
  TPUHIP_REQUIRE(d->x_cs % 16 == 0 && d->y_cs % 16 == 0 && d->x_cs >= d->c && d->y_cs >= d->c,
                 "pool: bad channel strides %d / %d for %d channels", d->x_cs, d->y_cs, d->c);
  // every window must contain at least one real input position
  TPUHIP_REQUIRE((d->oh - 1) * d->sh - d->pt < d->ih && (d->ow - 1) * d->sw - d->pl < d->iw &&
                     d->pt < d->kh && d->pl < d->kw,
                 "pool: an output window lies entirely in the padding");
  a->x = (const int8_t *)x;
  a->y = (int8_t *)y;
  a->ih = d->ih; a->iw = d->iw;
  a->kh = d->kh; a->kw = d->kw; a->sh = d->sh; a->sw = d->sw;
  a->pt = d->pt; a->pl = d->pl; a->x_cs = d->x_cs; a->y_cs = d->y_cs;
  a->mult = 0.f; a->inv_pot = 1.f;
  a->by_c16 = FastDiv((d->c + 15) / 16); a->by_ow = FastDiv(d->ow); a->by_oh = FastDiv(d->oh);
  const int64_t image = (int64_t)d->oh * d->ow * a->c16();
  TPUHIP_REQUIRE(image < (1ll << 31), "pool: an image of 2^31 output groups or more");
  return TPUHIP_OK;
}

// calls fn(args) for runs of images whose output groups a 31-bit index reaches
template <class F>
int each_part(PoolArgs a, int n, F fn) {
  const int64_t image = (int64_t)a.oh() * a.ow() * a.c16();
  const int most = (int)std::min<int64_t>(((1ll << 31) - 1) / image, n);
  for (int left = n; left > 0; left -= most) {
    a.total = (uint32_t)(image * std::min(left, most));
    if (int rc = fn(a)) return rc;
    a.x += (int64_t)most * a.ih * a.iw * a.x_cs;
    a.y += (int64_t)most * a.oh() * a.ow() * a.y_cs;
  }
  return TPUHIP_OK;
}

// the side of a square window, 0 otherwise
int square(const PoolArgs &a) { return a.kh == a.kw ? a.kh : 0; }

unsigned blocks_for(const PoolArgs &a) {
  // a multiple of 8 (see xcd_block)
  return 8u * (unsigned)std::max<int64_t>(1, std::min<int64_t>(((int64_t)a.total + 2047) / 2048, 1 << 13));
}

}  // namespace

extern "C" {

int tpuhip_pool_max_i8(tpuhip_ctx *ctx, const tpuhip_pool_desc *d, const void *x, void *y) {
  TPUHIP_REQUIRE(ctx, "pool_max: NULL context");
  PoolArgs a;
  if (int rc = fill_args(d, x, y, &a)) return rc;
  auto *kernel = square(a) == 3 ? pool_max_kernel<3> : square(a) == 2 ? pool_max_kernel<2> : pool_max_kernel<0>;
  return each_part(a, d->n, [&](const PoolArgs &part) -> int {
    launch(ctx, kernel, dim3(blocks_for(part)), dim3(256), part);
    TPUHIP_CHECK_HIP(hipGetLastError());
    return TPUHIP_OK;
  });
}

int tpuhip_pool_avg_i8(tpuhip_ctx *ctx, const tpuhip_pool_desc *d, const void *x, void *y,
                       uint32_t multiplier, uint32_t rshift) {
  TPUHIP_REQUIRE(ctx, "pool_avg: NULL context");
  TPUHIP_REQUIRE(rshift <= 30, "pool_avg: rshift %u outside [0,30]", rshift);
  PoolArgs a;
  if (int rc = fill_args(d, x, y, &a)) return rc;
  TPUHIP_REQUIRE((int64_t)d->kh * d->kw * 128 < (1 << 24), "pool_avg: window too large");
  a.mult = (float)multiplier;
  a.inv_pot = 1.0f / (float)(1 << rshift);
  auto *kernel = square(a) == 3 ? pool_avg_kernel<3> : square(a) == 2 ? pool_avg_kernel<2> : pool_avg_kernel<0>;
  return each_part(a, d->n, [&](const PoolArgs &part) -> int {
    // few outputs with many positions each: several lanes share one (65536 outputs fill the chip without)
    const int taps = part.kh * part.kw;
    if (taps > 64 && part.total < (1 << 16)) return run_window(ctx, part);
    if (taps >= 16 && part.total < (1 << 16))
      launch(ctx, pool_avg_split_kernel, dim3((unsigned)(((int64_t)part.total * 8 + 255) / 256)), dim3(256), part, FastDiv(part.kw));
    else
      launch(ctx, kernel, dim3(blocks_for(part)), dim3(256), part);
    TPUHIP_CHECK_HIP(hipGetLastError());
    return TPUHIP_OK;
  });
}

}  // extern "C"
