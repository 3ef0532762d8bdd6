// Two-input elementwise ops with broadcasting on int8 channels-last tensors:
// EltwiseMax / Min / Mul (core/eltwise.cpp:143-347) and BroadcastAdd / Mul / Sub
// (core/broadcast.cpp:45-154).  One lane = 16 channels of one output pixel; an
// operand dimension of 1 repeats along that dimension (a channel count of 1 repeats
// one byte over the 16 lanes of the group).
#include "common.hpp"

using namespace tpuhip;

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
constexpr int kThreads = 256;

// 112 bytes: a launch with more than that of arguments costs the host 0.5 us more (3.1 and 3.65 us back to back).
struct BinArgs {
  const int8_t *x0, *x1;
  int8_t *y;
  FastDiv by_groups, by_w, by_h;
  // pixels from one n, h, w of an operand to the next, 0 where it repeats; bytes per pixel, 0 where its channels repeat
  int n0, h0, w0, cs0;
  int n1, h1, w1, cs1;
  int c;
  int m0, m1;                // mul: m0 is the qdm multiplier
  uint32_t op_shift_relu;    // op | rshift << 8 | relu << 16
  uint32_t total;            // output pixels * 16-channel groups, below 2^31
};
static_assert(sizeof(BinArgs) <= 112, "see above");

__device__ __forceinline__ int32_t sb(int32_t word, int i) { return (int32_t)(int8_t)(word >> (8 * i)); }

__device__ __forceinline__ v4i load_operand(const int8_t *x, int64_t pix, int cs, int cs_y, int cg) {
  if (cs < 0) {   // one channel for all, at -cs bytes per pixel
    const int32_t s = (int32_t)((uint32_t)(uint8_t)x[pix * -cs] * 0x01010101u);
    return v4i{s, s, s, s};
  }
  return *reinterpret_cast<const v4i *>(x + pix * cs_y + cg * 16);
}

// A thread makes one 16-channel group; the op is known at compile time.  4 x 120 x 75 x 75, 8.6 MB (5.8 with a per-channel
// gate): 5.4 us with the op and the zeroing of pad channels decided per byte and 64-bit divisions for the indices, 3.3 now.
// PIXELWISE: neither operand repeats along n, h or w, so both read the output's pixel.
template <bool MUL, bool PIXELWISE>
__global__ __launch_bounds__(kThreads) void binary_kernel(BinArgs a) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= a.total) return;
  uint32_t cg = i;
  const uint32_t pix = a.by_groups.split(cg);
  int64_t p0 = pix, p1 = pix;
  if (!PIXELWISE) {
    uint32_t w = pix, h = a.by_w.split(w);
    const int n = (int)a.by_h.split(h);
    p0 = (int64_t)n * a.n0 + (int64_t)h * a.h0 + (int64_t)w * a.w0;
    p1 = (int64_t)n * a.n1 + (int64_t)h * a.h1 + (int64_t)w * a.w1;
  }
  const int cs = (int)a.by_groups.d * 16;
  const v4i v0 = load_operand(a.x0, p0, a.cs0, cs, (int)cg);
  const v4i v1 = load_operand(a.x1, p1, a.cs1, cs, (int)cg);
  const int op = (int)(a.op_shift_relu & 0xff), rshift = (int)(a.op_shift_relu >> 8 & 0xff);
  const int32_t floor0 = a.op_shift_relu >> 16 ? 0 : INT32_MIN;
  const int32_t rnd = rshift > 0 ? (1 << (rshift - 1)) : 0;
  const int32_t mask = (int32_t)((1u << rshift) - 1u);
  v4i out;
  auto make = [&](auto combine) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t word = 0;
#pragma unroll
      for (int b = 0; b < 4; ++b) word |= ((uint32_t)combine(sb(v0[q], b), sb(v1[q], b)) & 0xffu) << (8 * b);
      out[q] = (int)word;
    }
  };
  if constexpr (MUL) {
    make([&](int32_t x, int32_t y) { return requant_qdm(max(x * y, floor0), a.m0, rshift, mask, mask >> 1, -128); });
  } else {
    auto scaled = [&](int32_t v) { return clamp_i32((max(v, floor0) + rnd) >> rshift, -128, 127); };
    switch (op) {   // the same for all
      case TPUHIP_BIN_ADD: make([&](int32_t x, int32_t y) { return scaled(x * a.m0 + y * a.m1); }); break;
      case TPUHIP_BIN_SUB: make([&](int32_t x, int32_t y) { return scaled(x * a.m0 - y * a.m1); }); break;
      case TPUHIP_BIN_MAX: make([&](int32_t x, int32_t y) { return scaled(max(x * a.m0, y * a.m1)); }); break;
      default: make([&](int32_t x, int32_t y) { return scaled(min(x * a.m0, y * a.m1)); }); break;
    }
  }
  const int live = a.c - (int)cg * 16;   // pad channels are zero
  if (live < 16) {
#pragma unroll
    for (int q = 0; q < 4; ++q) out[q] &= live >= q * 4 + 4 ? -1 : live <= q * 4 ? 0 : (int)((1u << (8 * (live - q * 4))) - 1u);
  }
  *reinterpret_cast<v4i *>(a.y + (int64_t)i * 16) = out;
}

}  // namespace

extern "C" int tpuhip_binary_i8(tpuhip_ctx *ctx, const tpuhip_binary_desc *d, const void *x0,
                                const void *x1, void *y) {
  TPUHIP_REQUIRE(ctx && d && x0 && x1 && y, "binary: NULL argument");
  TPUHIP_REQUIRE(d->op >= TPUHIP_BIN_ADD && d->op <= TPUHIP_BIN_MUL, "binary: unknown op %d", d->op);
  TPUHIP_REQUIRE(d->n > 0 && d->c > 0 && d->h > 0 && d->w > 0, "binary: non-positive dimension");
  const int dims[2][4] = {{d->n0, d->c0, d->h0, d->w0}, {d->n1, d->c1, d->h1, d->w1}};
  const int out[4] = {d->n, d->c, d->h, d->w};
  for (int k = 0; k < 2; ++k)
    for (int j = 0; j < 4; ++j)
      TPUHIP_REQUIRE(dims[k][j] == out[j] || dims[k][j] == 1,
                     "binary: operand %d dimension %d is %d, neither 1 nor the output's %d", k, j,
                     dims[k][j], out[j]);
  TPUHIP_REQUIRE(d->y_cs >= d->c && d->y_cs % 16 == 0 && d->x0_cs >= d->c0 && d->x0_cs % 16 == 0 &&
                     d->x1_cs >= d->c1 && d->x1_cs % 16 == 0,
                 "binary: channel strides must be multiples of 16 covering the channels");
  TPUHIP_REQUIRE(d->c0 == 1 || d->x0_cs == d->y_cs, "binary: operand 0 channel stride differs from the output's");
  TPUHIP_REQUIRE(d->c1 == 1 || d->x1_cs == d->y_cs, "binary: operand 1 channel stride differs from the output's");
  TPUHIP_REQUIRE(d->rshift >= 0 && d->rshift <= 31, "binary: rshift %d outside [0,31]", d->rshift);
  if (d->op == TPUHIP_BIN_MUL) {
    TPUHIP_REQUIRE(d->rshift != 0 || d->multiplier != 0,
                   "binary: a product with rshift 0 and multiplier 0 has no int8 meaning "
                   "(the reference keeps the raw product)");
  } else {
    TPUHIP_REQUIRE(d->rshift <= 30, "binary: rshift %d outside [0,30]", d->rshift);
    TPUHIP_REQUIRE(d->m0 >= -128 && d->m0 <= 127 && d->m1 >= -128 && d->m1 <= 127,
                   "binary: multipliers must be int8");
  }
  TPUHIP_REQUIRE((int64_t)d->n * d->h * d->w < (1ll << 31), "binary: tensor too large");
  TPUHIP_CHECK_HIP(hipSetDevice(ctx->device));
  BinArgs a{};
  a.x0 = (const int8_t *)x0; a.x1 = (const int8_t *)x1; a.y = (int8_t *)y;
  const int groups = d->y_cs / 16;
  a.by_groups = FastDiv(groups); a.by_w = FastDiv(d->w); a.by_h = FastDiv(d->h);
  a.n0 = d->n0 == 1 ? 0 : d->h0 * d->w0; a.h0 = d->h0 == 1 ? 0 : d->w0; a.w0 = d->w0 == 1 ? 0 : 1;
  a.n1 = d->n1 == 1 ? 0 : d->h1 * d->w1; a.h1 = d->h1 == 1 ? 0 : d->w1; a.w1 = d->w1 == 1 ? 0 : 1;
  a.cs0 = d->c0 == 1 ? -d->x0_cs : 0;
  a.cs1 = d->c1 == 1 ? -d->x1_cs : 0;
  a.c = d->c;
  const bool mul = d->op == TPUHIP_BIN_MUL;
  a.m0 = mul ? d->multiplier : d->m0; a.m1 = d->m1;
  a.op_shift_relu = (uint32_t)d->op | (uint32_t)d->rshift << 8 | (d->do_relu ? 1u << 16 : 0u);
  const bool pixelwise = d->n0 == d->n && d->h0 == d->h && d->w0 == d->w && d->n1 == d->n &&
                         d->h1 == d->h && d->w1 == d->w;
  auto *kernel = mul ? (pixelwise ? binary_kernel<true, true> : binary_kernel<true, false>)
                     : (pixelwise ? binary_kernel<false, true> : binary_kernel<false, false>);
  // as many images a launch as a 31-bit index of groups reaches
  const int64_t image = (int64_t)d->h * d->w * groups;
  TPUHIP_REQUIRE(image < (1ll << 31), "binary: an image of 2^31 16-channel groups or more");
  const int most = (int)std::min<int64_t>(((1ll << 31) - 1) / image, d->n);
  for (int left = d->n; left > 0; left -= most) {
    const int images = std::min(left, most);
    a.total = (uint32_t)(image * images);
    launch(ctx, kernel, dim3((unsigned)ceil_div64(a.total, kThreads)), dim3(kThreads), a);
    TPUHIP_CHECK_HIP(hipGetLastError());
    a.x0 += (int64_t)most * a.n0 * (a.cs0 < 0 ? -a.cs0 : d->y_cs);
    a.x1 += (int64_t)most * a.n1 * (a.cs1 < 0 ? -a.cs1 : d->y_cs);
    a.y += image * 16 * most;
  }
  return TPUHIP_OK;
}
