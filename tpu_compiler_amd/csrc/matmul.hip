// Batched and transposed FullyConnected (core/fullyconnected.cpp:44-91; shapes by
// parseFullyConnectedParam, TPUOperationSupport.cpp:568-605) on channels-last device tensors.
// The reference permutes the input into [batch][m][k], runs one inner product per batch and
// permutes the result back; here the kernels find the operands through the tensors' 4-d views, and
// so need no permuted copies (any batch, either transpose, results of rank 3 or 4).  The plain
// [m,k] x [n,k] case runs on the conv path (tpuhip_fc_prepack).
#include "conv_epilogue.hpp"

#include <algorithm>
#include <cstring>
#include <vector>

using namespace tpuhip;

struct tpuhip_fc_batched_weights {
  tpuhip_fc_batched_desc d;
  int8_t *filter = nullptr;   // [batch][n][k], or its fragments (packed_filter)
  bool matrix = false;        // runs on fc_batched_mfma_kernel
  bool uniform = false;       // one (rshift, multiplier) for the whole batch
  bool fast = false;          // no sum can overflow the requantisation's rounding
  int32_t *params = nullptr;  // bias [batch][n] (zeros without one), then multiplier[batch], rshift[batch]
  int64_t total = 0;          // result elements
};

namespace {

struct FcbArgs {
  tpuhip_fc_batched_desc d;
  const int8_t *x, *w;
  const int32_t *bias, *mult, *rshift;
  int8_t *y;
  int64_t total;
};

// logical flat index of a 4-d view -> byte offset in the channels-last tensor
__device__ __forceinline__ int64_t view_offset(int64_t g, int C, int H, int W, int cs) {
  const int w = (int)(g % W);
  g /= W;
  const int h = (int)(g % H);
  g /= H;
  const int c = (int)(g % C);
  const int64_t n = g / C;
  return ((n * H + h) * W + w) * cs + c;
}

// One lane per result element: what is left for filters whose fragments would be nearly all padding (a batch of more than
// 2^15 products of a few elements each, see tpuhip_fc_batched_prepack).
__global__ __launch_bounds__(256) void fc_batched_kernel(FcbArgs a) {
  const tpuhip_fc_batched_desc &d = a.d;
  const int64_t mn = (int64_t)d.m * d.n;
  for (int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; f < a.total;
       f += (int64_t)gridDim.x * blockDim.x) {
    // the result's logical index: [batch_high][m][batch_low][n] when transposed, else [batch][m][n]
    int64_t r = f;
    const int nn = (int)(r % d.n);
    r /= d.n;
    int hb, lb, mm;
    if (d.output_transpose) {
      lb = (int)(r % d.batch_low);
      r /= d.batch_low;
      mm = (int)(r % d.m);
      hb = (int)(r / d.m);
    } else {
      mm = (int)(r % d.m);
      r /= d.m;
      lb = (int)(r % d.batch_low);
      hb = (int)(r / d.batch_low);
    }
    const int b = hb * d.batch_low + lb;
    // first element of the input row: [batch_high][m][batch_low][k] when transposed, else [batch][m][k]
    const int64_t g0 = d.input_transpose ? (((int64_t)hb * d.m + mm) * d.batch_low + lb) * d.k
                                         : ((int64_t)b * d.m + mm) * d.k;
    const int64_t x0 = view_offset(g0, d.x_c, d.x_h, d.x_w, d.x_cs);
    const int64_t xs = d.k > 1 ? view_offset(g0 + 1, d.x_c, d.x_h, d.x_w, d.x_cs) - x0 : 0;
    const int8_t *wr = a.w + ((int64_t)b * d.n + nn) * d.k;
    const int8_t *xr = a.x + x0;
    int32_t s = a.bias[(int64_t)b * d.n + nn];
    for (int t = 0; t < d.k; ++t) s += (int32_t)xr[(int64_t)t * xs] * (int32_t)wr[t];
    if (d.do_relu) s = max(s, 0);
    // (rshift, multiplier) of block f / (m*n) of the result as it lies after the output permute (:78-87)
    const int i = (int)(f / mn);
    const int32_t e = a.rshift[i];
    const int32_t mask = (int32_t)((1u << e) - 1u);
    a.y[view_offset(f, d.y_c, d.y_h, d.y_w, d.y_cs)] =
        (int8_t)requant_qdm(s, a.mult[i], e, mask, mask >> 1, -128);
  }
}

// ---------------------------------------------------------------------------
// The products on the matrix cores.  A workgroup takes 32 rows of a product and up to 256 of its columns, two blocks of 32
// per wave.  The rows' K elements go through LDS, 512 at a time; the filter comes straight from memory, packed as the
// fragments the instruction reads (1 KB runs, zeros past n and k, so that what LDS holds past k does not matter).
//
// In memory a [batch, m, k] or [batch_high, m, batch_low, k] tensor in channels-last form is [batch][k][m]: m is contiguous
// (XM).  It is read by dwords and transposed on the way into LDS, and the result, whose 32 x 32 block leaves the instruction
// with four consecutive m per lane and register, is stored 16 bytes at a time (YM).  Any other view (m between, as in a
// [batch_high, batch_low, m, k] tensor) is read and written byte by byte at the places that its index gives.
//
// Two steps of the filter, the bias and the pair (multiplier, shift) are requested before the rows are waited for; a block of 16
// outputs a lane is requantised with that pair in scalars where one serves all of it.
// Bound: launch and one trip to memory.  Replayed from a graph, before (a trip each for the rows, the second step and the
// parameters; one WG of five blocks; pairs looked up per output) and now: 32 products of 160 x 64 x 160 5.33 -> 3.56 us, 12 of 384 x
// 64 x 384 6.41 -> 4.18, 96 of 128 x 128 x 128 5.43 -> 4.22, 96 of 384 x 128 x 384 25.8 -> 16.3.
// ---------------------------------------------------------------------------
constexpr int kChunkSteps = 16;                  // K steps of 32 per pass through LDS
// Filter fragments in flight, before the rows are waited for.  Of one, two and four, two are within 3 % of the fastest in all of 22
// shapes: 32 products of 160 x 64 x 160 3.79, 3.75, 3.93 us, 96 of 384 x 128 x 384 18.1, 16.3, 15.9, 32 of 512 x 512 x 512 with rows
// and results byte by byte 59.7, 59.1, 64.6.
constexpr int kAhead = 2;
constexpr int kRowBytes = kChunkSteps * 32 + 16;  // 16 bytes apart from the next bank cycle: 16-byte reads by row do not collide

struct View {
  int cs, c;
  FastDiv by_c, by_h, by_w;
  // byte offset of logical flat index g
  __device__ __forceinline__ int64_t at(uint32_t g) const {
    uint32_t w = g, h = by_w.split(w), ch = by_h.split(h);
    const uint32_t n = by_c.split(ch);
    return (((int64_t)n * by_h.d + h) * by_w.d + w) * cs + ch;
  }
};

struct FcbMfmaArgs {
  const int8_t *x, *w;
  const int32_t *bias, *mult, *rshift;
  int8_t *y;
  View xv, yv;
  int m, k, n, low, steps, tiles, per_wg, relu, uniform, in_t, out_t;   // per_wg: blocks of columns of a workgroup
  FastDiv by_mtiles, by_nblocks, by_low, by_mn;
};

// SIMPLE: one multiplier and shift for all that a workgroup writes, and sums that cannot overflow the rounding.  The other form
// looks pairs up per output and is held to the registers that leave three waves on a SIMD (96 products of 200 x 33 x 70, a pair
// each: two 10.4 us, three 7.4, four, which spill, 8.9).
template <bool XM, bool YM, bool SIMPLE>
__global__ __launch_bounds__(256, SIMPLE ? 1 : 3) void fc_batched_mfma_kernel(FcbMfmaArgs a) {
  __shared__ __attribute__((aligned(16))) int8_t rows[32 * kRowBytes];
  __shared__ uint32_t base[32], stride[32];
  asm volatile("" ::"s"(a.x), "s"(a.w), "s"(a.bias), "s"(a.mult), "s"(a.rshift), "s"(a.y), "s"(a.xv.cs), "s"(a.yv.cs), "s"(a.m), "s"(a.k),
               "s"(a.n), "s"(a.low), "s"(a.steps), "s"(a.tiles), "s"(a.per_wg), "s"(a.by_mtiles.mul), "s"(a.by_nblocks.mul),
               "s"(a.by_low.mul));   // named here they arrive together
  uint32_t nb = blockIdx.x, mt = a.by_nblocks.split(nb), b = a.by_mtiles.split(mt);
  uint32_t lb = b;
  const uint32_t hb = a.by_low.split(lb);
  const int m0 = (int)mt * 32, wave = threadIdx.x >> 6, lane = threadIdx.x & 63, col = lane & 31, half = lane >> 5;
  const int t0 = (int)nb * a.per_wg + wave, t1 = t0 + 4;   // this wave's blocks of columns
  const bool have0 = wave < a.per_wg && t0 < a.tiles, have1 = wave + 4 < a.per_wg && t1 < a.tiles;
  const int8_t *w0 = a.w + (((int64_t)b * a.tiles + (have0 ? t0 : 0)) * a.steps * 64 + lane) * 16;
  const int8_t *w1 = a.w + (((int64_t)b * a.tiles + (have1 ? t1 : 0)) * a.steps * 64 + lane) * 16;
  v16i acc0 = {}, acc1 = {};
  v4i f0[kAhead] = {}, f1[kAhead] = {};
#pragma unroll
  for (int d = 0; d < kAhead; ++d) {
    if (have0 && d < a.steps) f0[d] = *reinterpret_cast<const v4i *>(w0 + d * 1024);
    if (have1 && d < a.steps) f1[d] = *reinterpret_cast<const v4i *>(w1 + d * 1024);
  }
  int32_t bias_of[2];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int nn = (t ? t1 : t0) * 32 + col;
    bias_of[t] = (t ? have1 : have0) && nn < a.n ? a.bias[(int64_t)b * a.n + nn] : 0;
  }
  const int32_t mult_b = a.mult[b], shift_b = a.rshift[b];
  if (!XM && threadIdx.x < 32) {
    // logical index of the row's first element, byte offset and the bytes from one element to the next
    const uint32_t mm = (uint32_t)min(m0 + (int)threadIdx.x, a.m - 1);
    const uint32_t g = (a.in_t ? (hb * a.m + mm) * a.low + lb : b * a.m + mm) * a.k;
    const int64_t at = a.xv.at(g);
    base[threadIdx.x] = (uint32_t)at;   // tensors of less than 2^31 bytes (prepack)
    stride[threadIdx.x] = a.k > 1 ? (uint32_t)(a.xv.at(g + 1) - at) : 0;
  }
  for (int s0 = 0; s0 < a.steps; s0 += kChunkSteps) {
    const int steps = min(kChunkSteps, a.steps - s0), k0 = s0 * 32;
    if (s0 || !XM) __syncthreads();
    if constexpr (XM) {
      for (int it = threadIdx.x; it < steps * 64; it += 256) {   // four k by four m
        const int mq = (it & 7) * 4, kq = (it >> 3) * 4, k = k0 + kq;
        const int8_t *p = a.x + ((int64_t)b * a.k + k) * a.xv.cs + m0 + mq;
        uint32_t v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          v[j] = k + j < a.k && m0 + mq < a.m ? *reinterpret_cast<const uint32_t *>(p + (int64_t)j * a.xv.cs) : 0;
        const uint32_t lo0 = __builtin_amdgcn_perm(v[1], v[0], 0x05010400u), hi0 = __builtin_amdgcn_perm(v[1], v[0], 0x07030602u),
                       lo1 = __builtin_amdgcn_perm(v[3], v[2], 0x05010400u), hi1 = __builtin_amdgcn_perm(v[3], v[2], 0x07030602u);
        uint32_t *to = reinterpret_cast<uint32_t *>(rows + mq * kRowBytes + kq);
        to[0] = __builtin_amdgcn_perm(lo1, lo0, 0x05040100u);
        to[kRowBytes / 4] = __builtin_amdgcn_perm(lo1, lo0, 0x07060302u);
        to[kRowBytes / 2] = __builtin_amdgcn_perm(hi1, hi0, 0x05040100u);
        to[kRowBytes / 4 * 3] = __builtin_amdgcn_perm(hi1, hi0, 0x07060302u);
      }
    } else {
      for (int it = threadIdx.x; it < steps * 256; it += 256) {   // four k of a row; lanes along k
        const int kq = (it % (steps * 8)) * 4, row = it / (steps * 8);
        const int8_t *p = a.x + base[row];
        uint32_t v = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (k0 + kq + j < a.k) v |= (uint32_t)(uint8_t)p[(uint64_t)(k0 + kq + j) * stride[row]] << (8 * j);
        *reinterpret_cast<uint32_t *>(rows + row * kRowBytes + kq) = v;
      }
    }
    __syncthreads();
    const int8_t *mine = rows + col * kRowBytes + half * 16;
    for (int s = 0; s < steps; s += kAhead) {
#pragma unroll
      for (int d = 0; d < kAhead; ++d) {
        if (s + d >= steps) break;
        const v4i fa = *reinterpret_cast<const v4i *>(mine + (s + d) * 32);
        acc0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa, f0[d], acc0, 0, 0, 0);
        if (have1) acc1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa, f1[d], acc1, 0, 0, 0);
        const int next = s0 + s + d + kAhead;   // (kChunkSteps is a multiple of kAhead: a step's slot is the same in every pass)
        if (next < a.steps) {
          if (have0) f0[d] = *reinterpret_cast<const v4i *>(w0 + (int64_t)next * 1024);
          if (have1) f1[d] = *reinterpret_cast<const v4i *>(w1 + (int64_t)next * 1024);
        }
      }
    }
  }
  // a lane holds, of column col, rows 8 * (i / 4) + 4 * half + i % 4
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const v16i &acc = t ? acc1 : acc0;
    const int nn = (t ? t1 : t0) * 32 + col;
    if (!(t ? have1 : have0)) continue;
    const int32_t bias = bias_of[t];
    int32_t mult = mult_b, e = shift_b;
    uint32_t word[4];
    if constexpr (SIMPLE) {
      const int32_t hpot = 1 << (e - 1);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        int32_t v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          int32_t s = acc[q * 4 + i] + bias;
          if (a.relu) s = max(s, 0);
          const int32_t x = srdhm(s, mult);
          v[i] = (x + hpot + (x >> 31)) >> e;
        }
        const uint32_t w = pack_sat4(v[0], v[1], v[2], v[3], -128);
        const int mm = m0 + 8 * q + 4 * half, live = a.m - mm;
        word[q] = live >= 4 ? w : live > 0 ? w & ((1u << (8 * live)) - 1u) : 0;
        if (!YM && nn < a.n) {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (i < live) {
              const uint32_t f = a.out_t ? ((hb * a.m + (uint32_t)(mm + i)) * a.low + lb) * a.n + nn : (b * a.m + (uint32_t)(mm + i)) * a.n + nn;
              a.y[a.yv.at(f)] = (int8_t)(w >> (8 * i));
            }
        }
      }
    } else
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      int32_t s = acc[i] + bias;
      if (a.relu) s = max(s, 0);
      if (a.out_t && !a.uniform) {
        // (rshift, multiplier) of block f / (m*n) of the result as it lies after the output permute (:78-87)
        const int mm = m0 + 8 * (i / 4) + 4 * half + i % 4;
        const uint32_t f = mm < a.m && nn < a.n ? ((uint32_t)mm * a.low + lb) * a.n + nn : 0;
        const uint32_t blk = hb * a.low + a.by_mn.div(f);
        mult = a.mult[blk];
        e = a.rshift[blk];
      }
      const int32_t mask = (int32_t)((1u << e) - 1u);
      const uint32_t r = (uint32_t)requant_qdm(s, mult, e, mask, mask >> 1, -128) & 0xffu;
      if (YM) {
        const uint32_t live = m0 + 8 * (i / 4) + 4 * half + i % 4 < a.m ? r : 0;
        word[i / 4] = i % 4 ? word[i / 4] | live << (8 * (i % 4)) : live;
      } else {
        const int mm = m0 + 8 * (i / 4) + 4 * half + i % 4;
        if (mm < a.m && nn < a.n) {
          const uint32_t f = a.out_t ? ((hb * a.m + (uint32_t)mm) * a.low + lb) * a.n + nn : (b * a.m + (uint32_t)mm) * a.n + nn;
          a.y[a.yv.at(f)] = (int8_t)r;
        }
      }
    }
    if constexpr (YM) {
      // the wave's halves exchange dwords: each then has 16 consecutive rows
      const auto p = __builtin_amdgcn_permlane32_swap(word[0], word[2], false, false);
      const auto q = __builtin_amdgcn_permlane32_swap(word[1], word[3], false, false);
      const int mm = m0 + half * 16;
      if (nn < a.n && mm < a.m)
        *reinterpret_cast<v4i *>(a.y + ((int64_t)b * a.n + nn) * a.yv.cs + mm) = v4i{(int)p[0], (int)p[1], (int)q[0], (int)q[1]};
    }
  }
}

// the filter's fragments: [batch][32 columns][32 of k][lane][16], zeros past n and k
std::vector<int8_t> packed_filter(const tpuhip_fc_batched_desc &d, const int8_t *filter) {
  const int64_t batch = (int64_t)d.batch_high * d.batch_low, tiles = (d.n + 31) / 32, steps = (d.k + 31) / 32;
  std::vector<int8_t> out((size_t)(batch * tiles * steps * 1024), 0);
  for (int64_t b = 0; b < batch; ++b)
    for (int64_t nn = 0; nn < d.n; ++nn) {
      const int8_t *row = filter + (b * d.n + nn) * d.k;
      int8_t *to = out.data() + (b * tiles + nn / 32) * steps * 1024 + nn % 32 * 16;
      for (int64_t k = 0; k < d.k; k += 16)
        std::memcpy(to + k / 32 * 1024 + k % 32 / 16 * 512, row + k, (size_t)std::min<int64_t>(16, d.k - k));
    }
  return out;
}

bool last_dim_is(int c, int h, int w, int want) {
  if (want == 1) return true;
  const int last = w > 1 ? w : h > 1 ? h : c;
  return last == want;
}

}  // namespace

extern "C" {

int tpuhip_fc_batched_prepack(tpuhip_ctx *ctx, const tpuhip_fc_batched_desc *desc, const int8_t *filter,
                              const int32_t *bias, const int32_t *multiplier, const int32_t *rshift,
                              tpuhip_fc_batched_weights **out) {
  TPUHIP_REQUIRE(ctx && desc && filter && multiplier && rshift && out, "tpuhip_fc_batched_prepack: NULL argument");
  const tpuhip_fc_batched_desc &d = *desc;
  TPUHIP_REQUIRE(d.batch_high >= 1 && d.batch_low >= 1 && d.m >= 1 && d.k >= 1 && d.n >= 1,
                 "fc_batched: batch_high, batch_low, m, k, n must be positive");
  const int64_t batch = (int64_t)d.batch_high * d.batch_low;
  TPUHIP_REQUIRE(batch * d.m * (int64_t)d.k < (1ll << 31) && batch * d.m * (int64_t)d.n < (1ll << 31) &&
                     batch * d.n * (int64_t)d.k < (1ll << 31),
                 "fc_batched: tensor of 2^31 elements or more");
  TPUHIP_REQUIRE(d.x_c >= 1 && d.x_h >= 1 && d.x_w >= 1 && d.y_c >= 1 && d.y_h >= 1 && d.y_w >= 1,
                 "fc_batched: 4-d views must be positive");
  TPUHIP_REQUIRE(d.x_cs >= d.x_c && d.y_cs >= d.y_c, "fc_batched: channel stride below the channel count");
  TPUHIP_REQUIRE((batch * d.m * d.k) % ((int64_t)d.x_c * d.x_h * d.x_w) == 0,
                 "fc_batched: the input's view (%d,%d,%d) does not divide batch*m*k", d.x_c, d.x_h, d.x_w);
  TPUHIP_REQUIRE((batch * d.m * d.n) % ((int64_t)d.y_c * d.y_h * d.y_w) == 0,
                 "fc_batched: the result's view (%d,%d,%d) does not divide batch*m*n", d.y_c, d.y_h, d.y_w);
  TPUHIP_REQUIRE(last_dim_is(d.x_c, d.x_h, d.x_w, d.k), "fc_batched: the input's last dim must be k = %d", d.k);
  TPUHIP_REQUIRE(last_dim_is(d.y_c, d.y_h, d.y_w, d.n), "fc_batched: the result's last dim must be n = %d", d.n);
  for (int64_t i = 0; i < batch; ++i)
    TPUHIP_REQUIRE(rshift[i] >= 0 && rshift[i] <= 31, "fc_batched: rshift[%lld] = %d outside [0,31]",
                   (long long)i, rshift[i]);
  TPUHIP_CHECK_HIP(hipSetDevice(ctx->device));
  auto *w = new tpuhip_fc_batched_weights;
  w->d = d;
  w->total = batch * d.m * d.n;
  // on the matrix cores unless padding the filter to 32 x 32 would blow it up beyond reason, or the grid (2^24 workgroups) or
  // the kernel's 31-bit byte offsets do not reach
  const int64_t padded = batch * round_up(d.n, 32) * round_up(d.k, 32);
  const int64_t groups = batch * ((d.m + 31) / 32) * ((d.n + 255) / 256);   // as many as of one block a wave stay below 4 a CU
  const int64_t x_bytes = batch * d.m * d.k / d.x_c * d.x_cs, y_bytes = batch * d.m * d.n / d.y_c * d.y_cs;
  w->matrix = padded <= std::max<int64_t>(32 << 20, 4 * batch * d.n * d.k) && groups < (1 << 24) && x_bytes < (1ll << 31) &&
              y_bytes < (1ll << 31);
  // RoundingDivideByPOT without its sign-dependent mask: shifts of 1 and more, and sums that with the rounding term fit 32 bits
  int64_t largest = 0;
  for (int64_t i = 0; bias && i < batch * d.n; ++i) largest = std::max<int64_t>(largest, std::abs((int64_t)bias[i]));
  w->fast = true;
  for (int64_t i = 0; i < batch; ++i)
    w->fast &= rshift[i] >= 1 && (int64_t)d.k * 128 * 128 + largest + 1 + (1ll << (rshift[i] - 1)) < (1ll << 31);
  w->uniform = std::count(multiplier, multiplier + batch, multiplier[0]) == batch && std::count(rshift, rshift + batch, rshift[0]) == batch;
  std::vector<int8_t> packed;
  if (w->matrix) {
    packed = packed_filter(d, filter);
    filter = packed.data();
  }
  const size_t fbytes = w->matrix ? packed.size() : (size_t)(batch * d.n * d.k);
  std::vector<int32_t> params((size_t)(batch * d.n + 2 * batch), 0);
  if (bias) std::copy(bias, bias + batch * d.n, params.begin());
  std::copy(multiplier, multiplier + batch, params.begin() + batch * d.n);
  std::copy(rshift, rshift + batch, params.begin() + batch * d.n + batch);
  hipError_t e = hipMalloc((void **)&w->filter, fbytes);
  if (e == hipSuccess) e = hipMalloc((void **)&w->params, params.size() * sizeof(int32_t));
  if (e == hipSuccess) e = hipMemcpy(w->filter, filter, fbytes, hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(w->params, params.data(), params.size() * sizeof(int32_t), hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    tpuhip_fc_batched_destroy(ctx, w);
    return set_error(TPUHIP_ERR_HIP, "fc_batched: uploading the weights failed: %s", hipGetErrorString(e));
  }
  *out = w;
  return TPUHIP_OK;
}

int tpuhip_fc_batched_destroy(tpuhip_ctx *ctx, tpuhip_fc_batched_weights *w) {
  (void)ctx;
  if (!w) return TPUHIP_OK;
  if (w->filter) (void)hipFree(w->filter);
  if (w->params) (void)hipFree(w->params);
  delete w;
  return TPUHIP_OK;
}

int tpuhip_fc_batched_i8(tpuhip_ctx *ctx, const tpuhip_fc_batched_weights *w, const void *x, void *y) {
  TPUHIP_REQUIRE(ctx && w && x && y, "tpuhip_fc_batched_i8: NULL argument");
  const tpuhip_fc_batched_desc &d = w->d;
  const int64_t batch = (int64_t)d.batch_high * d.batch_low;
  if (w->matrix) {
    FcbMfmaArgs a{};
    a.x = static_cast<const int8_t *>(x);
    a.w = w->filter;
    a.bias = w->params;
    a.mult = w->params + batch * d.n;
    a.rshift = a.mult + batch;
    a.y = static_cast<int8_t *>(y);
    a.xv = View{d.x_cs, d.x_c, FastDiv(d.x_c), FastDiv(d.x_h), FastDiv(d.x_w)};
    a.yv = View{d.y_cs, d.y_c, FastDiv(d.y_c), FastDiv(d.y_h), FastDiv(d.y_w)};
    a.m = d.m; a.k = d.k; a.n = d.n; a.low = d.batch_low;
    a.steps = (d.k + 31) / 32;
    a.tiles = (d.n + 31) / 32;
    a.relu = d.do_relu; a.uniform = w->uniform;
    a.in_t = d.input_transpose; a.out_t = d.output_transpose;
    a.by_mn = FastDiv((int64_t)d.m * d.n);
    // m contiguous: the view's channels are the rows and the rest is one product's (or one batch_high's) columns
    const bool xm = d.x_c == d.m && (int64_t)d.x_h * d.x_w == (d.input_transpose ? (int64_t)d.batch_low * d.k : d.k) && d.x_cs % 4 == 0 &&
                    (uintptr_t)x % 4 == 0;
    const bool ym = d.y_c == d.m && (int64_t)d.y_h * d.y_w == (d.output_transpose ? (int64_t)d.batch_low * d.n : d.n) && d.y_cs % 16 == 0 &&
                    (uintptr_t)y % 16 == 0;
    const bool simple = w->fast && (w->uniform || !d.output_transpose);
    // A wave takes two blocks of columns only where there are workgroups enough without that: 32 products of 160 x 64 x 160 are 160
    // of them so, one wave in four with two blocks, and 320 of three and two blocks without (3.83 and 3.75 us).  Enough are those
    // that a CU holds, two to four: with one block a wave and two, 96 of 160 x 64 x 160, 960 workgroups, 4.85 and 4.83 us where rows
    // come in dwords, 10.2 and 9.4 with pairs looked up, 23.6 and 20.2 byte by byte, where every workgroup gathers the rows anew;
    // 48 of 256 x 128 x 256 (768) 5.68 and 5.83, 8.7 and 10.8, 21.1 and 19.6.
    const int mtiles = (d.m + 31) / 32;
    const bool wide = batch * mtiles * ((a.tiles + 3) / 4) > (!xm ? 2 : simple ? 4 : 3) * (int64_t)ctx->num_cu;
    const int nblocks = wide ? (a.tiles + 7) / 8 : (a.tiles + 3) / 4;
    a.per_wg = (a.tiles + nblocks - 1) / nblocks;
    a.by_mtiles = FastDiv(mtiles); a.by_nblocks = FastDiv(nblocks); a.by_low = FastDiv(d.batch_low);
    auto *kernel = xm   ? ym ? simple ? fc_batched_mfma_kernel<true, true, true> : fc_batched_mfma_kernel<true, true, false>
                             : simple ? fc_batched_mfma_kernel<true, false, true> : fc_batched_mfma_kernel<true, false, false>
                   : ym ? simple ? fc_batched_mfma_kernel<false, true, true> : fc_batched_mfma_kernel<false, true, false>
                        : simple ? fc_batched_mfma_kernel<false, false, true> : fc_batched_mfma_kernel<false, false, false>;
    launch(ctx, kernel, dim3((unsigned)(batch * mtiles * nblocks)), dim3(256), a);
    TPUHIP_CHECK_HIP(hipGetLastError());
    return TPUHIP_OK;
  }
  FcbArgs a;
  a.d = w->d;
  a.x = static_cast<const int8_t *>(x);
  a.w = w->filter;
  a.bias = w->params;
  a.mult = w->params + batch * w->d.n;
  a.rshift = a.mult + batch;
  a.y = static_cast<int8_t *>(y);
  a.total = w->total;
  const unsigned blocks = (unsigned)std::min<int64_t>(ceil_div64(a.total, 256), (int64_t)ctx->num_cu * 32);
  launch(ctx, fc_batched_kernel, dim3(blocks), dim3(256), a);
  TPUHIP_CHECK_HIP(hipGetLastError());
  return TPUHIP_OK;
}

}  // extern "C"
