// Bandwidth-bound INT8 ops for gfx950: eltwise add, 256-entry table ops
// (leaky-ReLU / clip / LUT activations), ReLU, nearest upsample, concat and the
// NCHW <-> channels-last conversions at the API edge.  All kernels move 16
// bytes per lane per access where the layout allows it; none uses MFMA.
#include "common.hpp"

#include <cstring>

#include <algorithm>
#include <cmath>
#include <type_traits>

using namespace tpuhip;

typedef int v4i __attribute__((ext_vector_type(4)));

namespace {

constexpr int kThreads = 256;

inline unsigned grid_for(int64_t items, int per_block = kThreads, int64_t cap = 1 << 16) {
  return (unsigned)std::max<int64_t>(1, std::min<int64_t>(ceil_div64(items, per_block), cap));
}

__device__ __forceinline__ int32_t sb(int32_t word, int i) {
  return (int32_t)(int8_t)(word >> (8 * i));
}

// ---------------------------------------------------------------------------
// eltwise add (core/eltwise.cpp:52-85).  The reference forms sum_i x_i * m_i and
// sum / 2^r in float; both are exact for |sum| < 2^24 (at most 8 inputs of
// 128 * 128), so the integer form floor((sum + 2^(r-1)) / 2^r) is identical.
// ---------------------------------------------------------------------------
template <int NIN>
struct EltArgs {
  const int8_t *x[NIN];
  int8_t *y;
  int32_t m[NIN];
  int rshift;
  int relu;
  int64_t n16;   // number of 16-byte groups
};

// one group a thread (two of them one after the other: 4.4 us on 4 x 120 x 75 x 75, now 3.4)
template <int NIN>
__global__ __launch_bounds__(kThreads) void eltwise_add_kernel(EltArgs<NIN> a) {
  const int32_t rnd = a.rshift > 0 ? (1 << (a.rshift - 1)) : 0;
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < a.n16; i += (int64_t)gridDim.x * kThreads) {
    v4i in[NIN];
#pragma unroll
    for (int k = 0; k < NIN; ++k) in[k] = reinterpret_cast<const v4i *>(a.x[k])[i];
    v4i out;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t word = 0;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        int32_t s = 0;
#pragma unroll
        for (int k = 0; k < NIN; ++k) s += sb(in[k][q], b) * a.m[k];
        if (a.relu) s = max(s, 0);
        s = clamp_i32((s + rnd) >> a.rshift, -128, 127);
        word |= ((uint32_t)s & 0xffu) << (8 * b);
      }
      out[q] = (int)word;
    }
    reinterpret_cast<v4i *>(a.y)[i] = out;
  }
}

// ---------------------------------------------------------------------------
// one 256-entry table per channel (PRelu's per-channel slope, core/activation.cpp:185-224):
// y[pixel][c] = tables[c][(unsigned char)x[pixel][c]].  One lane = 16 channels of a pixel;
// the tables (c * 256 bytes) stay in the caches.  Pad channels are written as zero.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kThreads) void lut_per_channel_kernel(const int8_t *x, int8_t *y,
                                                                   const uint8_t *tables,
                                                                   int64_t total, int c, int cs) {
  const int c16 = cs >> 4;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int cg = (int)(i % c16);
    const v4i in = reinterpret_cast<const v4i *>(x)[i];
    v4i out;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t word = 0;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const int ch = cg * 16 + q * 4 + b;
        const uint32_t idx = ((uint32_t)in[q] >> (8 * b)) & 255u;
        const uint32_t r = ch < c ? tables[(size_t)ch * 256 + idx] : 0u;
        word |= r << (8 * b);
      }
      out[q] = (int)word;
    }
    reinterpret_cast<v4i *>(y)[i] = out;
  }
}

// ---------------------------------------------------------------------------
// table ops: y = table[(unsigned char)x] (core/activation.cpp:47-53).  The table
// arrives by value in the kernel arguments and is spread into LDS once per
// workgroup; pad channels are forced to zero.
// ---------------------------------------------------------------------------
struct LutArgs {
  const int8_t *x;
  int8_t *y;
  int64_t pixels;
  int c, x_cs, y_cs;  // channels, strides
  int coff;           // channel offset into y (concat)
  int use_table;
  FastDiv by_groups;  // 16-byte groups per pixel
};

// the 64 words of a table, one per thread, out of the kernel arguments (requested first, parked behind the data's request)
__device__ __forceinline__ uint32_t table_word(const Table256 &t) { return threadIdx.x < 64 ? t.w[threadIdx.x] : 0; }
__device__ __forceinline__ void park_table(uint32_t word, uint32_t *lds) {
  if (threadIdx.x < 64) lds[threadIdx.x] = word;
  __syncthreads();
}
// four bytes through a table in LDS; bytes from `valid` on are zero
__device__ __forceinline__ uint32_t look_up4(uint32_t w, const uint8_t *tab, int valid) {
  const uint32_t o = (uint32_t)tab[w & 255u] | ((uint32_t)tab[(w >> 8) & 255u] << 8) | ((uint32_t)tab[(w >> 16) & 255u] << 16) |
                     ((uint32_t)tab[w >> 24] << 24);
  return o & (valid >= 4 ? 0xffffffffu : valid <= 0 ? 0u : (1u << (8 * valid)) - 1u);
}

// A table that follows from numbers, made by the kernel: thread v & 255 computes the entry of input v.  (Its 256 bytes as an
// argument cost a launch 0.5 us and the host's loop 0.2 us or more.)  The float overload of
// applyMultiplierAndRShiftAndSaturateInt8: product, quotient by a power of two, floor(f + 0.5), clamp.
__device__ __forceinline__ int32_t rescaled(int32_t v, float m, float inv_pot) {
  return saturate_int8_f(__fmul_rn(__fmul_rn((float)v, m), inv_pot));
}
struct LeakyRule {
  float m_pos, inv_pos, m_neg, inv_neg;   // m_pos 0: positive inputs stay
};
__device__ __forceinline__ void park_leaky(const LeakyRule &r, uint32_t *lds) {
  const int32_t v = (int32_t)(int8_t)threadIdx.x;
  const int32_t o = v <= 0 ? rescaled(v, r.m_neg, r.inv_neg) : r.m_pos != 0.f ? rescaled(v, r.m_pos, r.inv_pos) : v;
  reinterpret_cast<int8_t *>(lds)[threadIdx.x] = (int8_t)o;
  __syncthreads();
}

__global__ __launch_bounds__(kThreads) void leaky_vec_kernel(LutArgs a, LeakyRule rule) {
  __shared__ uint32_t tab[64];
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const bool live = i < a.pixels * a.by_groups.d;
  uint32_t r = (uint32_t)i;
  const int64_t pix = a.by_groups.split(r);
  const int cg = (int)r;
  v4i v = {0, 0, 0, 0};
  if (live) v = *reinterpret_cast<const v4i *>(a.x + pix * a.x_cs + cg * 16);
  park_leaky(rule, tab);
#pragma unroll
  for (int q = 0; q < 4; ++q) v[q] = (int)look_up4((uint32_t)v[q], reinterpret_cast<const uint8_t *>(tab), a.c - cg * 16 - q * 4);
  if (live) *reinterpret_cast<v4i *>(a.y + pix * a.y_cs + cg * 16) = v;
}

// vector form: groups of 16 channels, strides multiple of 16, coff multiple of 16.  One group per thread: 4 x 120 x 75 x 75 in
// 3.1 us (8.2 with four groups after one another in a quarter of the threads and a table spread by 64 selects).
__global__ __launch_bounds__(kThreads) void lut_vec_kernel(LutArgs a, Table256 t) {
  __shared__ uint32_t tab[64];
  const uint32_t word = a.use_table ? table_word(t) : 0;
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const bool live = i < a.pixels * a.by_groups.d;
  uint32_t r = (uint32_t)i;
  const int64_t pix = a.by_groups.split(r);
  const int cg = (int)r;
  v4i v = {0, 0, 0, 0};
  if (live) v = *reinterpret_cast<const v4i *>(a.x + pix * a.x_cs + cg * 16);
  if (a.use_table) {
    park_table(word, tab);
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = (int)look_up4((uint32_t)v[q], reinterpret_cast<const uint8_t *>(tab), a.c - cg * 16 - q * 4);
  }
  if (live) *reinterpret_cast<v4i *>(a.y + pix * a.y_cs + a.coff + cg * 16) = v;
}

// byte form for channel offsets / counts that are not multiples of 16
__global__ __launch_bounds__(kThreads) void lut_byte_kernel(LutArgs a, Table256 t) {
  __shared__ uint32_t tab[64];
  park_table(a.use_table ? table_word(t) : 0, tab);
  const int64_t total = a.pixels * a.c;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t pix = i / a.c;
    const int ch = (int)(i - pix * a.c);
    uint8_t v = (uint8_t)a.x[pix * a.x_cs + ch];
    if (a.use_table) v = reinterpret_cast<const uint8_t *>(tab)[v];
    a.y[pix * a.y_cs + a.coff + ch] = (int8_t)v;
  }
}

// Concat of up to kConcatMax inputs as one launch, each input with a table of its own or none.
constexpr int kConcatMax = 6;

// along the channels: a thread makes 16 channels of an output pixel.  A dword that lies inside one input is one load at any
// alignment; one that straddles two is put together from bytes.  (Inputs off the 16-channel grid went byte by byte, a
// launch each and one for the pad channels: 4 x (120 + 120) x 75 x 75 in 22 us, now 5.4, with tables 6.3.)
template <int N>
struct ConcatChannelArgs {
  const int8_t *x[N];
  int8_t *y;
  int start[N + 1];            // first output channel of each input; start[N] = output channels
  int cs[N];
  int y_cs;
  FastDiv by_groups;           // groups written per pixel
  uint32_t total;
};
// requantisation and ReLU of each input: tables made by the kernel
template <int N>
struct ConcatRules {
  float m[N], inv_pot[N];      // m 0 with inv_pot 0: values stay
  int relu;
};
template <int N>
__device__ __forceinline__ void park_rules(const ConcatRules<N> &r, uint32_t *tab) {
  const int32_t v = (int32_t)(int8_t)threadIdx.x;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    int32_t o = r.inv_pot[k] != 0.f ? rescaled(v, r.m[k], r.inv_pot[k]) : v;
    if (r.relu) o = max(o, 0);
    reinterpret_cast<int8_t *>(tab + k * 64)[threadIdx.x] = (int8_t)o;
  }
  __syncthreads();
}
struct NoRules {};

// Two inputs have kernels of their own: their arguments stay below the 112 bytes up to which a launch is 0.5 us cheaper.
template <int N, class Rules>
__global__ __launch_bounds__(kThreads) void concat_channels_kernel(ConcatChannelArgs<N> a, Rules rules) {
  constexpr bool kTables = !std::is_same<Rules, NoRules>::value;
  __shared__ uint32_t tab[kTables ? N * 64 : 1];
  if constexpr (kTables) park_rules<N>(rules, tab);
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= a.total) return;
  uint32_t r = i;
  const int64_t pix = a.by_groups.split(r);
  const int c0 = (int)r * 16;
  v4i out;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int c = c0 + q * 4;
    const int8_t *src = a.x[0];
    int k = 0, first = 0, last = a.start[1], cs = a.cs[0];
#pragma unroll
    for (int j = 1; j < N; ++j)
      if (c >= a.start[j]) { k = j; src = a.x[j]; first = a.start[j]; last = a.start[j + 1]; cs = a.cs[j]; }
    uint32_t w = 0;
    if (c + 4 <= last) {
      __builtin_memcpy(&w, src + pix * cs + (c - first), 4);
      if constexpr (kTables) w = look_up4(w, reinterpret_cast<const uint8_t *>(tab + k * 64), 4);
    } else {
      for (int b = 0; b < 4; ++b) {
        const int cb = c + b;
        if (cb >= a.start[N]) break;   // pad channels are zero
        const int8_t *from = a.x[0];
        int kb = 0, at = 0, bcs = a.cs[0];
#pragma unroll
        for (int j = 1; j < N; ++j)
          if (cb >= a.start[j]) { kb = j; from = a.x[j]; at = a.start[j]; bcs = a.cs[j]; }
        uint32_t v = (uint8_t)from[pix * bcs + (cb - at)];
        if constexpr (kTables) v = reinterpret_cast<const uint8_t *>(tab + kb * 64)[v];
        w |= v << (8 * b);
      }
    }
    out[q] = (int)w;
  }
  *reinterpret_cast<v4i *>(a.y + pix * a.y_cs + c0) = out;
}

// along n, h or w: in channels-last memory these are "for each outer index, the inputs' chunks one after the other" (outer =
// image row for w, image for h, nothing for n), chunks of whole pixels.  A thread moves one 16-byte group.
struct ConcatArgs {
  const int8_t *x[kConcatMax];
  int8_t *y;
  int64_t outer;                 // outer indices
  int64_t stride[kConcatMax];    // bytes from one outer index to the next in each input
  int64_t y_stride;              // ... in the output
  int64_t start[kConcatMax + 1]; // first 16-byte group of each input's chunk within an output chunk; start[n] = groups per chunk
  int n, c;
  FastDiv by_groups, by_c16;     // groups per outer index, per pixel
};

template <class Rules>
__global__ __launch_bounds__(kThreads) void concat_chunks_kernel(ConcatArgs a, Rules rules) {
  constexpr bool kTables = !std::is_same<Rules, NoRules>::value;
  __shared__ uint32_t tab[kTables ? kConcatMax * 64 : 1];
  if constexpr (kTables) park_rules<kConcatMax>(rules, tab);
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= a.outer * a.start[a.n]) return;
  uint32_t g = (uint32_t)i;
  const int64_t o = a.by_groups.split(g);
  // which input the group comes from: selects, so that no array is indexed by a lane's value
  const int8_t *src = a.x[0];
  int64_t stride = a.stride[0], first = 0;
  int k = 0;
#pragma unroll
  for (int j = 1; j < kConcatMax; ++j)
    if (a.n > j && g >= a.start[j]) { src = a.x[j]; stride = a.stride[j]; first = a.start[j]; k = j; }
  v4i v = *reinterpret_cast<const v4i *>(src + o * stride + (g - first) * 16);
  if constexpr (kTables) {
    uint32_t cg = g;   // chunks are whole pixels, so the group's place in its pixel follows from g alone
    a.by_c16.split(cg);
#pragma unroll
    for (int q = 0; q < 4; ++q)
      v[q] = (int)look_up4((uint32_t)v[q], reinterpret_cast<const uint8_t *>(tab + k * 64), a.c - (int)cg * 16 - q * 4);
  }
  *reinterpret_cast<v4i *>(a.y + o * a.y_stride + (int64_t)g * 16) = v;
}

// zero the channels [c0, c1) of every pixel
__global__ __launch_bounds__(kThreads) void zero_channels_kernel(int8_t *y, int64_t pixels, int cs,
                                                                 int c0, int c1) {
  const int w = c1 - c0;
  const int64_t total = pixels * w;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t pix = i / w;
    y[pix * cs + c0 + (int)(i - pix * w)] = 0;
  }
}

__global__ __launch_bounds__(kThreads) void relu_kernel(const v4i *x, v4i *y, int64_t n16) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16;
       i += (int64_t)gridDim.x * blockDim.x) {
    v4i v = x[i];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      uint32_t w = (uint32_t)v[q];
      // a byte with its sign bit set becomes 0
      uint32_t neg = (w & 0x80808080u) >> 7;   // 1 per negative byte
      uint32_t mask = neg * 0xffu;             // 0xff per negative byte
      v[q] = (int)(w & ~mask);
    }
    y[i] = v;
  }
}

// ---------------------------------------------------------------------------
// nearest upsample (core/upsample.cpp:20-41), channels-last: a thread reads one 16-byte group of an input pixel and
// writes it to the sh x sw output pixels it becomes.
// ---------------------------------------------------------------------------
struct UpsampleArgs {
  const int8_t *x;
  int8_t *y;
  FastDiv by_groups, by_iw;   // 16-byte groups per pixel, input columns
  int sh, sw, ow, x_cs, y_cs;
  int64_t total;
};
__global__ __launch_bounds__(kThreads) void upsample_kernel(UpsampleArgs a) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= a.total) return;
  uint32_t cg = (uint32_t)i;
  uint32_t pix = a.by_groups.split(cg);
  const v4i v = *reinterpret_cast<const v4i *>(a.x + (int64_t)pix * a.x_cs + cg * 16);
  uint32_t w = pix;
  const uint32_t row = a.by_iw.split(w);   // image * input rows + input row: output rows follow each other the same way
  int8_t *to = a.y + ((int64_t)row * a.sh * a.ow + (int64_t)w * a.sw) * a.y_cs + cg * 16;
  for (int r = 0; r < a.sh; ++r, to += (int64_t)a.ow * a.y_cs)
    for (int s = 0; s < a.sw; ++s) *reinterpret_cast<v4i *>(to + (int64_t)s * a.y_cs) = v;
}

// ---------------------------------------------------------------------------
// layout conversion through an LDS tile: reads are contiguous along W (NCHW
// side), writes contiguous along C (channels-last side) and vice versa.
// ---------------------------------------------------------------------------
template <typename SRC>
__global__ __launch_bounds__(kThreads) void nchw_to_nhwc_kernel(const SRC *src, int8_t *dst, int c,
                                                                int64_t hw, int cs) {
  // block: 64 spatial positions x 64 channels of one image
  __shared__ int8_t tile[64][65];
  const int n = blockIdx.z;
  const int64_t s0 = (int64_t)blockIdx.x * 64;
  const int c0 = blockIdx.y * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;  // 4 rows of 64
  for (int r = ty; r < 64; r += 4) {
    const int ch = c0 + r;
    const int64_t s = s0 + tx;
    int8_t v = 0;
    if (ch < c && s < hw) v = (int8_t)src[((int64_t)n * c + ch) * hw + s];
    tile[r][tx] = v;
  }
  __syncthreads();
  for (int r = ty; r < 64; r += 4) {
    const int64_t s = s0 + r;
    const int ch = c0 + tx;
    if (s < hw && ch < cs) dst[((int64_t)n * hw + s) * cs + ch] = tile[tx][r];
  }
}

template <typename DST>
__global__ __launch_bounds__(kThreads) void nhwc_to_nchw_kernel(const int8_t *src, DST *dst, int c,
                                                                int64_t hw, int cs) {
  __shared__ int8_t tile[64][65];
  const int n = blockIdx.z;
  const int64_t s0 = (int64_t)blockIdx.x * 64;
  const int c0 = blockIdx.y * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int r = ty; r < 64; r += 4) {
    const int64_t s = s0 + r;
    const int ch = c0 + tx;
    int8_t v = 0;
    if (s < hw && ch < c) v = src[((int64_t)n * hw + s) * cs + ch];
    tile[r][tx] = v;
  }
  __syncthreads();
  for (int r = ty; r < 64; r += 4) {
    const int ch = c0 + r;
    const int64_t s = s0 + tx;
    if (ch < c && s < hw) dst[((int64_t)n * c + ch) * hw + s] = (DST)tile[tx][r];
  }
}

// The int8 conversions move dwords: four pixels of four channels at a time, transposed in registers.  NCHW rows start at
// any byte, so that side is accessed unaligned; where it lies in pinned host memory the bus sees whole runs of 128 bytes
// (byte accesses: 64).  hw pixels, tile of 64 channels x 128 pixels, LDS rows of one pixel's 16 dwords + 1.
__device__ __forceinline__ void transpose4x4(const uint32_t (&r)[4], uint32_t (&t)[4]) {
  const uint32_t lo01 = __builtin_amdgcn_perm(r[1], r[0], 0x05010400u), hi01 = __builtin_amdgcn_perm(r[1], r[0], 0x07030602u);
  const uint32_t lo23 = __builtin_amdgcn_perm(r[3], r[2], 0x05010400u), hi23 = __builtin_amdgcn_perm(r[3], r[2], 0x07030602u);
  t[0] = __builtin_amdgcn_perm(lo23, lo01, 0x05040100u);
  t[1] = __builtin_amdgcn_perm(lo23, lo01, 0x07060302u);
  t[2] = __builtin_amdgcn_perm(hi23, hi01, 0x05040100u);
  t[3] = __builtin_amdgcn_perm(hi23, hi01, 0x07060302u);
}
// up to `left` bytes at p (any alignment); the rest of the dword is zero
__device__ __forceinline__ uint32_t load_run(const int8_t *p, int64_t left) {
  uint32_t v = 0;
  if (left >= 4) {
    __builtin_memcpy(&v, p, 4);
  } else {
    for (int k = 0; k < 4; ++k)
      if (k < left) v |= (uint32_t)(uint8_t)p[k] << (8 * k);
  }
  return v;
}
__device__ __forceinline__ void store_run(int8_t *p, uint32_t v, int64_t left) {
  if (left >= 4) {
    __builtin_memcpy(p, &v, 4);
  } else {
    for (int k = 0; k < 4; ++k)
      if (k < left) p[k] = (int8_t)(v >> (8 * k));
  }
}
constexpr int kTransPix = 128, kTransRow = 17;

__global__ __launch_bounds__(kThreads) void nchw_to_nhwc_i8_kernel(const int8_t *src, int8_t *dst, int c, int64_t hw, int cs) {
  __shared__ uint32_t tile[kTransPix * kTransRow];
  const int64_t s0 = (int64_t)blockIdx.x * kTransPix;
  const int c0 = blockIdx.y * 64, n = blockIdx.z;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int pq = threadIdx.x & 31, cq = (threadIdx.x >> 5) + u * 8;
    const int64_t s = s0 + pq * 4;
    uint32_t r[4], t[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ch = c0 + cq * 4 + i;
      r[i] = ch < c && s < hw ? load_run(src + ((int64_t)n * c + ch) * hw + s, hw - s) : 0u;
    }
    transpose4x4(r, t);
#pragma unroll
    for (int j = 0; j < 4; ++j) tile[(pq * 4 + j) * kTransRow + cq] = t[j];
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kTransPix / 16; ++u) {
    const int cq = threadIdx.x & 15, p = (threadIdx.x >> 4) + u * 16;
    if (s0 + p < hw && c0 + cq * 4 < cs)
      *reinterpret_cast<uint32_t *>(dst + ((int64_t)n * hw + s0 + p) * cs + c0 + cq * 4) = tile[p * kTransRow + cq];
  }
}

// one tile of one image: pixels from s0, channels from c0
__device__ __forceinline__ void dense_tile(uint32_t *tile, const int8_t *src, int8_t *dst, int c, int64_t hw, int cs, int n, int64_t s0,
                                           int c0) {
#pragma unroll
  for (int u = 0; u < kTransPix / 16; ++u) {
    const int cq = threadIdx.x & 15, p = (threadIdx.x >> 4) + u * 16;
    uint32_t v = 0;
    if (s0 + p < hw && c0 + cq * 4 < cs)
      v = *reinterpret_cast<const uint32_t *>(src + ((int64_t)n * hw + s0 + p) * cs + c0 + cq * 4);
    tile[p * kTransRow + cq] = v;
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int pq = threadIdx.x & 31, cq = (threadIdx.x >> 5) + u * 8;
    const int64_t s = s0 + pq * 4;
    uint32_t r[4], t[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) r[j] = tile[(pq * 4 + j) * kTransRow + cq];
    transpose4x4(r, t);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int ch = c0 + cq * 4 + i;
      if (ch < c && s < hw) store_run(dst + ((int64_t)n * c + ch) * hw + s, t[i], hw - s);
    }
  }
}

__global__ __launch_bounds__(kThreads) void nhwc_to_nchw_i8_kernel(const int8_t *src, int8_t *dst, int c, int64_t hw, int cs) {
  __shared__ uint32_t tile[kTransPix * kTransRow];
  dense_tile(tile, src, dst, c, hw, cs, blockIdx.z, (int64_t)blockIdx.x * kTransPix, blockIdx.y * 64);
}

// Several tensors in one launch: a workgroup finds the one its tile belongs to, then the tile (pixels, then channels, then
// images).  A launch per tensor of half a megabyte is 6.6 us of which the bytes are 0.2, in turn with the transfers of those
// before it: the 34 tensors (18.5 MB) of a backbone's dump took 224 us of the stream, now 14, and the dump 880 us, now 705-720.
constexpr int kDenseMost = 48;
template <int N>
struct DenseList {
  DenseItem item[N];
  uint32_t end[N];     // workgroups up to and with each tensor's
  uint32_t by_pix[N], by_chan[N];   // tiles of a plane, of the channels
};
template <int N>
__global__ __launch_bounds__(kThreads) void dense_list_kernel(DenseList<N> l) {
  __shared__ uint32_t tile[kTransPix * kTransRow];
  int k = 0;
  while (blockIdx.x >= l.end[k]) ++k;   // the last end is the grid's
  const DenseItem it = l.item[k];
  uint32_t b = blockIdx.x - (k ? l.end[k - 1] : 0u);
  const uint32_t px = b % l.by_pix[k];
  b /= l.by_pix[k];
  dense_tile(tile, it.src, it.dst, it.c, it.hw, it.cs, b / l.by_chan[k], (int64_t)px * kTransPix, b % l.by_chan[k] * 64);
}

// at most four channels (images): a lane makes four pixels from one dword of each plane and writes their channel rows,
// one dword (cs 4) or 16 bytes (cs 16) each.  64 images of 3 x 224 x 224 from a 64-channel tile: 61 of 64 rows idle
__global__ __launch_bounds__(kThreads) void image_to_nhwc_i8_kernel(const int8_t *src, int8_t *dst, int c, int64_t hw, int cs) {
  const int64_t s = ((int64_t)blockIdx.x * kThreads + threadIdx.x) * 4;
  const int n = blockIdx.z;
  if (s >= hw) return;
  uint32_t r[4], t[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = i < c ? load_run(src + ((int64_t)n * c + i) * hw + s, hw - s) : 0u;
  transpose4x4(r, t);
  int8_t *to = dst + ((int64_t)n * hw + s) * cs;
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (s + j < hw) {
      if (cs == 4) *reinterpret_cast<uint32_t *>(to + j * 4) = t[j];
      else *reinterpret_cast<v4i *>(to + j * 16) = v4i{(int)t[j], 0, 0, 0};
    }
}

// one pixel per image (vectors): both sides are rows of channels, only their pitch differs; 16 bytes per lane, the
// dense side unaligned
template <bool TO_DENSE>
__global__ __launch_bounds__(kThreads) void vector_rows_i8_kernel(const int8_t *src, int8_t *dst, int64_t rows, int c, int cs) {
  const int groups = TO_DENSE ? (c + 15) >> 4 : cs >> 4;
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  const int64_t row = i / groups;
  if (row >= rows) return;
  const int c0 = (int)(i - row * groups) * 16;
  if (TO_DENSE) {
    const v4i v = *reinterpret_cast<const v4i *>(src + row * cs + c0);
    int8_t *to = dst + row * c + c0;
    if (c0 + 16 <= c) {
      __builtin_memcpy(to, &v, 16);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) store_run(to + q * 4, (uint32_t)v[q], (int64_t)c - c0 - q * 4);
    }
  } else {
    const int8_t *from = src + row * c + c0;
    v4i v = {0, 0, 0, 0};
    if (c0 + 16 <= c) {
      __builtin_memcpy(&v, from, 16);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (c0 + q * 4 < c) v[q] = (int)load_run(from + q * 4, (int64_t)c - c0 - q * 4);
    }
    *reinterpret_cast<v4i *>(dst + row * cs + c0) = v;
  }
}

int check_layout_args(const void *a, const void *b, int n, int c, int h, int w, int cs) {
  TPUHIP_REQUIRE(a && b, "layout: NULL pointer");
  TPUHIP_REQUIRE(n > 0 && c > 0 && h > 0 && w > 0, "layout: non-positive dimension");
  TPUHIP_REQUIRE(cs >= c && (cs % 16 == 0 || cs == 4), "layout: channel stride %d must be 4 or a multiple of 16, >= %d",
                 cs, c);
  TPUHIP_REQUIRE(n <= 65535 && (c + 63) / 64 <= 65535, "layout: too many images / channels");
  return TPUHIP_OK;
}

template <typename SRC>
int to_nhwc(tpuhip_ctx *ctx, const void *src, void *dst, int n, int c, int h, int w, int cs) {
  TPUHIP_REQUIRE(ctx, "layout: NULL context");
  if (int rc = check_layout_args(src, dst, n, c, h, w, cs)) return rc;
  const int64_t hw = (int64_t)h * w;
  if constexpr (sizeof(SRC) == 1) {
    // vectors, images, everything else
    const auto *from = (const int8_t *)src;
    if (hw == 1 && cs % 16 == 0)
      launch(ctx, (vector_rows_i8_kernel<false>), dim3((unsigned)ceil_div64((int64_t)n * (cs / 16), kThreads)), dim3(kThreads), from,
             (int8_t *)dst, (int64_t)n, c, cs);
    else if (c <= 4 && cs <= 16)
      launch(ctx, image_to_nhwc_i8_kernel, dim3((unsigned)ceil_div64(hw, kThreads * 4), 1, (unsigned)n), dim3(kThreads), from,
             (int8_t *)dst, c, hw, cs);
    else
      launch(ctx, nchw_to_nhwc_i8_kernel, dim3((unsigned)ceil_div64(hw, kTransPix), (unsigned)((cs + 63) / 64), (unsigned)n),
             dim3(kThreads), from, (int8_t *)dst, c, hw, cs);
  } else {
    dim3 grid((unsigned)ceil_div64(hw, 64), (unsigned)((cs + 63) / 64), (unsigned)n);
    launch(ctx, (nchw_to_nhwc_kernel<SRC>), grid, dim3(kThreads), (const SRC *)src, (int8_t *)dst, c, hw, cs);
  }
  TPUHIP_CHECK_HIP(hipGetLastError());
  return TPUHIP_OK;
}

template <typename DST>
int to_nchw(tpuhip_ctx *ctx, const void *src, void *dst, int n, int c, int h, int w, int cs) {
  TPUHIP_REQUIRE(ctx, "layout: NULL context");
  if (int rc = check_layout_args(src, dst, n, c, h, w, cs)) return rc;
  const int64_t hw = (int64_t)h * w;
  if constexpr (sizeof(DST) == 1) {
    if (hw == 1 && cs % 16 == 0)
      launch(ctx, (vector_rows_i8_kernel<true>), dim3((unsigned)ceil_div64((int64_t)n * ((c + 15) / 16), kThreads)), dim3(kThreads),
             (const int8_t *)src, (int8_t *)dst, (int64_t)n, c, cs);
    else
      launch(ctx, nhwc_to_nchw_i8_kernel, dim3((unsigned)ceil_div64(hw, kTransPix), (unsigned)((c + 63) / 64), (unsigned)n),
             dim3(kThreads), (const int8_t *)src, (int8_t *)dst, c, hw, cs);
  } else {
    dim3 grid((unsigned)ceil_div64(hw, 64), (unsigned)((c + 63) / 64), (unsigned)n);
    launch(ctx, (nhwc_to_nchw_kernel<DST>), grid, dim3(kThreads), (const int8_t *)src, (DST *)dst, c, hw, cs);
  }
  TPUHIP_CHECK_HIP(hipGetLastError());
  return TPUHIP_OK;
}

}  // namespace

int tpuhip::lay_out_dense(tpuhip_ctx *ctx, const DenseItem *items, size_t n) {
  constexpr int64_t kMostTiles = 1 << 22;
  constexpr int kFew = 4;   // the longer list is 2.9 KB of arguments
  DenseList<kDenseMost> l;
  int count = 0;
  int64_t blocks = 0;
  auto issue = [&] {
    if (count > kFew) {
      launch(ctx, dense_list_kernel<kDenseMost>, dim3((unsigned)blocks), dim3(kThreads), l);
    } else if (count) {
      DenseList<kFew> few{};
      for (int k = 0; k < count; ++k) {
        few.item[k] = l.item[k];
        few.end[k] = l.end[k];
        few.by_pix[k] = l.by_pix[k];
        few.by_chan[k] = l.by_chan[k];
      }
      launch(ctx, dense_list_kernel<kFew>, dim3((unsigned)blocks), dim3(kThreads), few);
    }
    count = 0;
    blocks = 0;
    return hipGetLastError();
  };
  for (size_t i = 0; i < n; ++i) {
    const DenseItem &it = items[i];
    if (int rc = check_layout_args(it.src, it.dst, it.n, it.c, it.h, it.w, it.cs)) return rc;
    const int64_t by_pix = ceil_div64(it.hw, kTransPix), by_chan = (it.c + 63) / 64, mine = by_pix * by_chan * it.n;
    // one tensor alone: a list of four is 240 bytes of arguments, and above 112 a launch costs the host 0.5 us more (65 536 elements
    // as floats 21.8 us, 23.1 by a list); rows of channels have a kernel of their own; so many tiles, a launch of their own
    if (n == 1 || it.hw == 1 || mine > kMostTiles) {
      if (int rc = to_nchw<int8_t>(ctx, it.src, it.dst, it.n, it.c, it.h, it.w, it.cs)) return rc;
      continue;
    }
    if (count == kDenseMost || blocks + mine > kMostTiles) TPUHIP_CHECK_HIP(issue());
    l.item[count] = it;
    l.by_pix[count] = (uint32_t)by_pix;
    l.by_chan[count] = (uint32_t)by_chan;
    l.end[count++] = (uint32_t)(blocks += mine);
  }
  TPUHIP_CHECK_HIP(issue());
  return TPUHIP_OK;
}

namespace {

// host: saturateInt8 of v * multiplier / 2^rshift evaluated in float32 the way
// applyMultiplierAndRShiftAndSaturateInt8's float overload does
// (QuantizationArithmetic.cpp:518-528, :301-334)
int8_t host_mult_rshift_sat8(float v, uint32_t rshift, uint32_t multiplier) {
#pragma clang fp contract(off)
  const float quo = v * (float)multiplier * (1.0f / (float)(1 << rshift));   // a power of two: the quotient, exactly
  // floor of a clamped number: the bounds are integers.  (No libm call and no branch, so that the loops over the 256 inputs
  // become vector code: a table takes 0.2 us of the host, 2 before.)
  const double s = std::min(std::max((double)quo + 0.5, -128.0), 127.0);
  const int t = (int)s;
  return (int8_t)(t - (s < (double)t));
}

Table256 pack_table(const int8_t *t) {
  Table256 r;
  for (int i = 0; i < 64; ++i)
    r.w[i] = (uint32_t)(uint8_t)t[4 * i] | ((uint32_t)(uint8_t)t[4 * i + 1] << 8) |
             ((uint32_t)(uint8_t)t[4 * i + 2] << 16) | ((uint32_t)(uint8_t)t[4 * i + 3] << 24);
  return r;
}

int launch_lut(tpuhip_ctx *ctx, const void *x, void *y, const int8_t *table, int64_t pixels, int c,
               int x_cs, int y_cs, int coff) {
  LutArgs a{};
  a.x = (const int8_t *)x;
  a.y = (int8_t *)y;
  a.pixels = pixels;
  a.c = c;
  a.x_cs = x_cs;
  a.y_cs = y_cs;
  a.coff = coff;
  a.use_table = table != nullptr;
  Table256 t{};
  if (table) t = pack_table(table);
  const bool vec = (x_cs % 16 == 0) && (y_cs % 16 == 0) && (coff % 16 == 0) &&
                   (c % 16 == 0 || (coff + round_up(c, 16) <= y_cs));
  if (vec) {
    a.by_groups = FastDiv((c + 15) / 16);
    const int64_t most = ((1ll << 31) - 1) / a.by_groups.d;   // as many pixels as the 31-bit index reaches
    for (int64_t p0 = 0; p0 < pixels; p0 += most, a.x += most * x_cs, a.y += most * y_cs) {
      a.pixels = std::min(most, pixels - p0);
      launch(ctx, lut_vec_kernel, dim3((unsigned)ceil_div64(a.pixels * a.by_groups.d, kThreads)), dim3(kThreads), a, t);
    }
  } else {
    launch(ctx, lut_byte_kernel, dim3(grid_for(pixels * c, kThreads * 8)), dim3(kThreads), a, t);
  }
  TPUHIP_CHECK_HIP(hipGetLastError());
  return TPUHIP_OK;
}

// INT8 LRN across channels (core/lrn.cpp:104-166).  A lane produces four consecutive channels
// of a pixel; the window of local_size channels around each is summed from the squares table
// (indexed by the input byte), rescaled to an index into the power table, and that entry
// scales the input.  All integers: the reference's float arithmetic is exact for them.
struct LrnArgs {
  const int8_t *x;
  int8_t *y;
  int64_t total;   // pixels * (cs / 4)
  int c, cs, local_size, sum_rshift, lrn_rshift, quant0, quant1;
  Table256 sqr, power;
};

__global__ __launch_bounds__(kThreads) void lrn_kernel(LrnArgs a) {
  __shared__ uint32_t tsq[64], tpw[64];
  if (threadIdx.x < 64) {
    tsq[threadIdx.x] = a.sqr.w[threadIdx.x];
    tpw[threadIdx.x] = a.power.w[threadIdx.x];
  }
  __syncthreads();
  const uint8_t *sq = reinterpret_cast<const uint8_t *>(tsq);
  const uint8_t *pw = reinterpret_cast<const uint8_t *>(tpw);
  const int c4 = a.cs >> 2, pre_pad = (a.local_size - 1) / 2;
  const int rnd_s = a.sum_rshift > 0 ? 1 << (a.sum_rshift - 1) : 0;
  const int rnd_l = a.lrn_rshift > 0 ? 1 << (a.lrn_rshift - 1) : 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < a.total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int cq = (int)(i % c4);
    const int64_t pix = i / c4;
    const int8_t *row = a.x + pix * a.cs;
    uint32_t word = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int ch = cq * 4 + b;
      if (ch >= a.c) continue;   // pad channels stay zero
      int s = 0;
      const int lo = max(ch - pre_pad, 0), hi = min(ch - pre_pad + a.local_size, a.c);
      for (int k = lo; k < hi; ++k) s += sq[(uint8_t)row[k]];
      const int t = min(max((s * a.quant0 + rnd_s) >> a.sum_rshift, 0), 255);
      const int m = (int)pw[t] * (int)row[ch] * a.quant1;
      const int o = min(max((m + rnd_l) >> a.lrn_rshift, -128), 127);
      word |= (uint32_t)(uint8_t)(int8_t)o << (8 * b);
    }
    *reinterpret_cast<uint32_t *>(a.y + pix * a.cs + cq * 4) = word;
  }
}

}  // namespace

extern "C" {

int tpuhip_nchw_to_nhwc_i8(tpuhip_ctx *ctx, const void *s, void *d, int n, int c, int h, int w,
                           int cs) {
  return to_nhwc<int8_t>(ctx, s, d, n, c, h, w, cs);
}
int tpuhip_nchw_f32_to_nhwc_i8(tpuhip_ctx *ctx, const void *s, void *d, int n, int c, int h, int w,
                               int cs) {
  return to_nhwc<float>(ctx, s, d, n, c, h, w, cs);
}
int tpuhip_nhwc_to_nchw_i8(tpuhip_ctx *ctx, const void *s, void *d, int n, int c, int h, int w,
                           int cs) {
  return to_nchw<int8_t>(ctx, s, d, n, c, h, w, cs);
}
int tpuhip_nhwc_i8_to_nchw_f32(tpuhip_ctx *ctx, const void *s, void *d, int n, int c, int h, int w,
                               int cs) {
  return to_nchw<float>(ctx, s, d, n, c, h, w, cs);
}

int tpuhip_eltwise_add_i8(tpuhip_ctx *ctx, const void *const *xs, int nin,
                          const int8_t *multiplier, int rshift, int do_relu, void *y,
                          size_t bytes) {
  TPUHIP_REQUIRE(ctx && xs && multiplier && y, "eltwise_add: NULL argument");
  TPUHIP_REQUIRE(nin >= 1 && nin <= 8, "eltwise_add: %d inputs (1..8 supported)", nin);
  TPUHIP_REQUIRE(rshift >= 0 && rshift <= 30, "eltwise_add: rshift %d outside [0,30]", rshift);
  TPUHIP_REQUIRE(bytes % 16 == 0, "eltwise_add: byte count %zu not a multiple of 16", bytes);
  if (bytes == 0) return TPUHIP_OK;
  for (int i = 0; i < nin; ++i) TPUHIP_REQUIRE(xs[i], "eltwise_add: input %d is NULL", i);
  auto run = [&](auto count) {
    constexpr int NIN = decltype(count)::value;
    EltArgs<NIN> a{};
    for (int i = 0; i < NIN; ++i) {
      a.x[i] = (const int8_t *)xs[i];
      a.m[i] = multiplier[i];
    }
    a.y = (int8_t *)y;
    a.rshift = rshift;
    a.relu = do_relu ? 1 : 0;
    a.n16 = (int64_t)(bytes / 16);
    launch(ctx, eltwise_add_kernel<NIN>, dim3(grid_for(a.n16, kThreads, 1 << 20)), dim3(kThreads), a);
  };
  switch (nin) {
    case 1: run(std::integral_constant<int, 1>()); break;
    case 2: run(std::integral_constant<int, 2>()); break;
    case 3: run(std::integral_constant<int, 3>()); break;
    case 4: run(std::integral_constant<int, 4>()); break;
    case 5: run(std::integral_constant<int, 5>()); break;
    case 6: run(std::integral_constant<int, 6>()); break;
    case 7: run(std::integral_constant<int, 7>()); break;
    default: run(std::integral_constant<int, 8>()); break;
  }
  TPUHIP_CHECK_HIP(hipGetLastError());
  return TPUHIP_OK;
}

int tpuhip_lut_i8(tpuhip_ctx *ctx, const void *x, void *y, const int8_t *table256, size_t pixels,
                  int c, int cs) {
  TPUHIP_REQUIRE(ctx && x && y && table256, "lut: NULL argument");
  TPUHIP_REQUIRE(c > 0 && cs >= c && cs % 16 == 0, "lut: bad channels %d / stride %d", c, cs);
  if (pixels == 0) return TPUHIP_OK;
  return launch_lut(ctx, x, y, table256, (int64_t)pixels, c, cs, cs, 0);
}

int tpuhip_lrn_i8(tpuhip_ctx *ctx, const void *x, void *y, size_t pixels, int c, int cs, int local_size,
                  const uint8_t *sqr_lut256, const uint8_t *power_lut256, int sum_rshift, int lrn_rshift,
                  int quant0, int quant1) {
  TPUHIP_REQUIRE(ctx && x && y && sqr_lut256 && power_lut256, "lrn: NULL argument");
  TPUHIP_REQUIRE(c > 0 && cs >= c && cs % 16 == 0, "lrn: bad channels %d / stride %d", c, cs);
  TPUHIP_REQUIRE(local_size >= 1 && local_size <= 64, "lrn: local_size %d outside [1,64]", local_size);
  TPUHIP_REQUIRE(sum_rshift >= 0 && sum_rshift <= 23 && lrn_rshift >= 0 && lrn_rshift <= 23,
                 "lrn: shifts %d / %d outside [0,23]", sum_rshift, lrn_rshift);
  // the reference computes in float; these bounds keep every intermediate an exact integer
  // multiple of a power of two below 2^24, so the integer form used here gives the same bytes
  // (the running sum holds one more term than the window while the head is added before the
  // tail is subtracted; the rounding term is half a unit of the shifted result)
  TPUHIP_REQUIRE(quant0 >= 0 && (int64_t)255 * quant0 * (local_size + 1) + (1ll << sum_rshift) < (1 << 24),
                 "lrn: quant_data0 %d too large for exact float sums", quant0);
  TPUHIP_REQUIRE(quant1 >= 0 && (int64_t)255 * 128 * quant1 + (1ll << lrn_rshift) < (1 << 24),
                 "lrn: quant_data1 %d too large for exact float products", quant1);
  if (pixels == 0) return TPUHIP_OK;
  TPUHIP_CHECK_HIP(hipSetDevice(ctx->device));
  LrnArgs a{};
  a.x = (const int8_t *)x;
  a.y = (int8_t *)y;
  a.total = (int64_t)pixels * (cs / 4);
  a.c = c; a.cs = cs; a.local_size = local_size;
  a.sum_rshift = sum_rshift; a.lrn_rshift = lrn_rshift; a.quant0 = quant0; a.quant1 = quant1;
  memcpy(a.sqr.w, sqr_lut256, 256);
  memcpy(a.power.w, power_lut256, 256);
  launch(ctx, lrn_kernel, dim3(grid_for(a.total, kThreads * 2)), dim3(kThreads), a);
  TPUHIP_CHECK_HIP(hipGetLastError());
  return TPUHIP_OK;
}

int tpuhip_lut_per_channel_i8(tpuhip_ctx *ctx, const void *x, void *y, const void *tables,
                              size_t pixels, int c, int cs) {
  TPUHIP_REQUIRE(ctx && x && y && tables, "lut_per_channel: NULL argument");
  TPUHIP_REQUIRE(c > 0 && cs >= c && cs % 16 == 0, "lut_per_channel: bad channels %d / stride %d", c, cs);
  if (pixels == 0) return TPUHIP_OK;
  TPUHIP_CHECK_HIP(hipSetDevice(ctx->device));
  const int64_t total = (int64_t)pixels * (cs / 16);
  launch(ctx, lut_per_channel_kernel, dim3(grid_for(total, kThreads * 2)), dim3(kThreads),
         (const int8_t *)x, (int8_t *)y, (const uint8_t *)tables, total, c, cs);
  TPUHIP_CHECK_HIP(hipGetLastError());
  return TPUHIP_OK;
}

int tpuhip_prelu_tables(const float *slope, int c, uint32_t rshift_pos, uint32_t multiplier_pos,
                        uint32_t rshift_neg, int8_t *tables) {
  TPUHIP_REQUIRE(slope && tables && c > 0, "prelu_tables: bad argument");
  TPUHIP_REQUIRE(rshift_pos <= 30 && rshift_neg <= 30, "prelu: rshift outside [0,30]");
  // PReluOpKernel::invoke (core/activation.cpp:185-224) for each channel and each of the 256 inputs
  for (int ch = 0; ch < c; ++ch)
    for (int v = -128; v <= 127; ++v) {
      int8_t out;
      if (v > 0) {
        out = host_mult_rshift_sat8((float)v, rshift_pos, multiplier_pos);
      } else {
        volatile float prod = slope[ch] * (float)v;
        volatile float quo = prod / (float)(1 << rshift_neg);
        double s = std::floor((double)quo + 0.5);
        s = s > 127.0 ? 127.0 : s < -128.0 ? -128.0 : s;
        out = (int8_t)(int)s;
      }
      tables[(size_t)ch * 256 + (uint8_t)(int8_t)v] = out;
    }
  return TPUHIP_OK;
}

int tpuhip_leaky_relu_table(uint32_t rshift_pos, uint32_t multiplier_pos, uint32_t rshift_neg,
                            uint32_t multiplier_neg, int8_t *table256) {
  TPUHIP_REQUIRE(table256, "leaky_relu_table: NULL table");
  TPUHIP_REQUIRE(rshift_pos <= 30 && rshift_neg <= 30, "leaky_relu: rshift outside [0,30]");
  // LeakyReluOpKernel::invoke (core/activation.cpp:126-153) for each of the 256 inputs;
  // entry index = two's-complement byte of the input
  for (int v = -128; v <= 127; ++v) {
    int8_t out;
    if (v > 0)
      out = multiplier_pos != 0 ? host_mult_rshift_sat8((float)v, rshift_pos, multiplier_pos)
                                : (int8_t)v;
    else
      out = host_mult_rshift_sat8((float)v, rshift_neg, multiplier_neg);
    table256[(uint8_t)(int8_t)v] = out;
  }
  return TPUHIP_OK;
}

int tpuhip_clip_table(float minv, float maxv, uint32_t rshift, uint32_t multiplier,
                      int8_t *table256) {
  TPUHIP_REQUIRE(table256, "clip_table: NULL table");
  TPUHIP_REQUIRE(rshift <= 30, "clip: rshift outside [0,30]");
  for (int v = -128; v <= 127; ++v) {
    const float c = std::max(minv, std::min((float)v, maxv));
    table256[(uint8_t)(int8_t)v] = host_mult_rshift_sat8(c, rshift, multiplier);
  }
  return TPUHIP_OK;
}

int tpuhip_leaky_relu_i8(tpuhip_ctx *ctx, const void *x, void *y, size_t pixels, int c, int cs,
                         uint32_t rshift_pos, uint32_t multiplier_pos, uint32_t rshift_neg,
                         uint32_t multiplier_neg) {
  TPUHIP_REQUIRE(rshift_pos <= 30 && rshift_neg <= 30, "leaky_relu: rshift outside [0,30]");
  TPUHIP_REQUIRE(ctx && x && y, "leaky_relu: NULL argument");
  TPUHIP_REQUIRE(c > 0 && cs >= c && cs % 16 == 0, "leaky_relu: bad channels %d / stride %d", c, cs);
  if (pixels == 0) return TPUHIP_OK;
  const int groups = (c + 15) / 16;
  if ((int64_t)pixels * groups >= (1ll << 31)) {
    int8_t table[256];
    if (int rc = tpuhip_leaky_relu_table(rshift_pos, multiplier_pos, rshift_neg, multiplier_neg, table)) return rc;
    return tpuhip_lut_i8(ctx, x, y, table, pixels, c, cs);
  }
  LutArgs a{};
  a.x = (const int8_t *)x;
  a.y = (int8_t *)y;
  a.pixels = (int64_t)pixels;
  a.c = c;
  a.x_cs = a.y_cs = cs;
  a.by_groups = FastDiv(groups);
  launch(ctx, leaky_vec_kernel, dim3((unsigned)ceil_div64((int64_t)pixels * groups, kThreads)), dim3(kThreads), a,
         LeakyRule{(float)multiplier_pos, 1.0f / (float)(1 << rshift_pos), (float)multiplier_neg, 1.0f / (float)(1 << rshift_neg)});
  TPUHIP_CHECK_HIP(hipGetLastError());
  return TPUHIP_OK;
}

int tpuhip_relu_i8(tpuhip_ctx *ctx, const void *x, void *y, size_t bytes) {
  TPUHIP_REQUIRE(ctx && x && y, "relu: NULL argument");
  TPUHIP_REQUIRE(bytes % 16 == 0, "relu: byte count %zu not a multiple of 16", bytes);
  if (bytes == 0) return TPUHIP_OK;
  const int64_t n16 = (int64_t)(bytes / 16);
  launch(ctx, relu_kernel, dim3(grid_for(n16, kThreads * 2)), dim3(kThreads), (const v4i *)x, (v4i *)y, n16);
  TPUHIP_CHECK_HIP(hipGetLastError());
  return TPUHIP_OK;
}

int tpuhip_upsample_nearest_i8(tpuhip_ctx *ctx, const void *x, void *y, int n, int c, int ih,
                               int iw, int scale_h, int scale_w, int x_cs, int y_cs) {
  TPUHIP_REQUIRE(ctx && x && y, "upsample: NULL argument");
  TPUHIP_REQUIRE(n > 0 && c > 0 && ih > 0 && iw > 0 && scale_h > 0 && scale_w > 0,
                 "upsample: non-positive dimension");
  TPUHIP_REQUIRE(x_cs % 16 == 0 && y_cs % 16 == 0 && x_cs >= c && y_cs >= c,
                 "upsample: bad channel strides %d / %d for %d channels", x_cs, y_cs, c);
  const int c16 = (c + 15) / 16;
  UpsampleArgs a{};
  a.x = (const int8_t *)x;
  a.y = (int8_t *)y;
  a.by_groups = FastDiv(c16);
  a.by_iw = FastDiv(iw);
  a.sh = scale_h; a.sw = scale_w; a.ow = iw * scale_w;
  a.x_cs = x_cs; a.y_cs = y_cs;
  const int64_t rows = (int64_t)n * ih, row_groups = (int64_t)iw * c16;
  const int64_t most = std::max<int64_t>(((1ll << 31) - 1) / row_groups, 1);   // as many rows as the 31-bit index reaches
  for (int64_t r0 = 0; r0 < rows; r0 += most) {
    a.total = std::min(most, rows - r0) * row_groups;
    launch(ctx, upsample_kernel, dim3((unsigned)ceil_div64(a.total, kThreads)), dim3(kThreads), a);
    a.x += most * iw * x_cs;
    a.y += most * scale_h * a.ow * y_cs;
  }
  TPUHIP_CHECK_HIP(hipGetLastError());
  return TPUHIP_OK;
}

int tpuhip_concat_i8(tpuhip_ctx *ctx, const void *const *xs, int nin, const int *in_dims,
                     const int *in_cs, int axis, const uint32_t *rshift,
                     const uint32_t *multiplier, int do_relu, void *y, int y_cs) {
  TPUHIP_REQUIRE(ctx && xs && in_dims && in_cs && y, "concat: NULL argument");
  TPUHIP_REQUIRE(nin >= 1, "concat: no inputs");
  TPUHIP_REQUIRE(axis >= 0 && axis <= 3, "concat: axis %d outside 0..3", axis);
  const bool need_quant = rshift != nullptr && multiplier != nullptr;
  int out_dims[4] = {in_dims[0], in_dims[1], in_dims[2], in_dims[3]};
  out_dims[axis] = 0;
  for (int i = 0; i < nin; ++i) {
    TPUHIP_REQUIRE(xs[i], "concat: input %d is NULL", i);
    for (int k = 0; k < 4; ++k) {
      TPUHIP_REQUIRE(in_dims[4 * i + k] > 0, "concat: input %d has a non-positive dimension", i);
      if (k != axis)
        TPUHIP_REQUIRE(in_dims[4 * i + k] == in_dims[k], "concat: input %d differs on axis %d", i, k);
    }
    TPUHIP_REQUIRE(in_cs[i] >= in_dims[4 * i + 1] && in_cs[i] % 16 == 0,
                   "concat: bad channel stride of input %d", i);
    if (need_quant) TPUHIP_REQUIRE(rshift[i] <= 30, "concat: rshift[%d] outside [0,30]", i);
    out_dims[axis] += in_dims[4 * i + axis];
  }
  const int N = out_dims[0], Cc = out_dims[1], H = out_dims[2], W = out_dims[3];
  TPUHIP_REQUIRE(y_cs >= Cc && y_cs % 16 == 0, "concat: bad output channel stride %d", y_cs);

  // Each input goes through a 256-entry table: requant (unless m == 1, r == 0) then ReLU
  // -- both pure functions of the int8 input (core/concat.cpp:66-88); the identity is no table.
  auto table_of = [&](int i, int8_t *table) {
    bool identity = true;
    for (int v = -128; v <= 127; ++v) {
      int8_t o = (int8_t)v;
      if (need_quant && !(multiplier[i] == 1 && rshift[i] == 0))
        o = host_mult_rshift_sat8((float)v, rshift[i], multiplier[i]);
      if (do_relu && o < 0) o = 0;
      if (o != (int8_t)v) identity = false;
      table[(uint8_t)(int8_t)v] = o;
    }
    return !identity;
  };
  // One launch for all inputs where the kernels' index arithmetic reaches: along the channels always; along n, h or w when
  // all tensors have the channel stride of their channel count (a chunk is then a run of whole pixels, pad channels included,
  // which are zero in every input).
  bool one = nin <= kConcatMax && (int64_t)N * H * W * (y_cs / 16) < (1ll << 31);
  for (int i = 0; i < nin && one && axis != 1; ++i) one = in_cs[i] == y_cs && y_cs == round_up(Cc, 16);
  if (one) {
    TPUHIP_CHECK_HIP(hipSetDevice(ctx->device));
    const bool rules = need_quant || do_relu;
    auto fill_rules = [&](auto &r, int n) {
      for (int i = 0; i < n; ++i) {
        const bool stays = i >= nin || !need_quant || (multiplier[i] == 1 && rshift[i] == 0);
        r.m[i] = stays ? 0.f : (float)multiplier[i];
        r.inv_pot[i] = stays ? 0.f : 1.0f / (float)(1 << rshift[i]);
      }
      r.relu = do_relu ? 1 : 0;
    };
    if (axis == 1) {
      auto run = [&](auto count) {
        constexpr int M = decltype(count)::value;
        ConcatChannelArgs<M> a{};
        a.y = (int8_t *)y;
        a.y_cs = y_cs;
        for (int i = 0; i < M; ++i) {   // inputs that are not there start where the channels end
          a.x[i] = (const int8_t *)xs[std::min(i, nin - 1)];
          a.cs[i] = in_cs[std::min(i, nin - 1)];
          a.start[i + 1] = a.start[i] + (i < nin ? in_dims[4 * i + 1] : 0);
        }
        // the output's stride may be wider than its channels: the pad groups are written as zero
        a.by_groups = FastDiv(y_cs / 16);
        a.total = (uint32_t)((int64_t)N * H * W * (y_cs / 16));
        const dim3 grid((unsigned)ceil_div64(a.total, kThreads));
        if (!rules) {
          launch(ctx, concat_channels_kernel<M, NoRules>, grid, dim3(kThreads), a, NoRules());
          return;
        }
        ConcatRules<M> r{};
        fill_rules(r, M);
        launch(ctx, concat_channels_kernel<M, ConcatRules<M>>, grid, dim3(kThreads), a, r);
      };
      static_assert(sizeof(ConcatChannelArgs<2>) + sizeof(ConcatRules<2>) <= 112, "see the kernel");
      if (nin <= 2) run(std::integral_constant<int, 2>());
      else run(std::integral_constant<int, kConcatMax>());
    } else {
      ConcatArgs a{};
      a.y = (int8_t *)y;
      a.n = nin;
      a.c = Cc;
      // bytes of one step along the axis, and of everything inside one outer index of the output
      const int64_t unit = axis == 3 ? y_cs : axis == 2 ? (int64_t)W * y_cs : (int64_t)H * W * y_cs;
      a.outer = axis == 3 ? (int64_t)N * H : axis == 2 ? N : 1;
      a.y_stride = unit * out_dims[axis];
      for (int i = 0; i < nin; ++i) {
        a.x[i] = (const int8_t *)xs[i];
        a.stride[i] = unit * in_dims[4 * i + axis];
        a.start[i + 1] = a.start[i] + unit * in_dims[4 * i + axis] / 16;
      }
      a.by_groups = FastDiv(a.start[nin]);
      a.by_c16 = FastDiv(y_cs / 16);
      const dim3 grid((unsigned)ceil_div64(a.outer * a.start[nin], kThreads));
      if (rules) {
        ConcatRules<kConcatMax> r{};
        fill_rules(r, kConcatMax);
        launch(ctx, concat_chunks_kernel<ConcatRules<kConcatMax>>, grid, dim3(kThreads), a, r);
      } else {
        launch(ctx, concat_chunks_kernel<NoRules>, grid, dim3(kThreads), a, NoRules());
      }
    }
    TPUHIP_CHECK_HIP(hipGetLastError());
    return TPUHIP_OK;
  }

  int offset = 0;  // running offset along the concat axis
  for (int i = 0; i < nin; ++i) {
    const int *dm = in_dims + 4 * i;
    int8_t table[256];
    const bool identity = !table_of(i, table);
    const int8_t *tab = identity ? nullptr : table;
    const int8_t *src = (const int8_t *)xs[i];
    int8_t *dst = (int8_t *)y;
    int rc = TPUHIP_OK;
    if (axis == 1) {
      rc = launch_lut(ctx, src, dst, tab, (int64_t)N * H * W, dm[1], in_cs[i], y_cs, offset);
    } else if (axis == 0) {
      rc = launch_lut(ctx, src, dst + (int64_t)offset * H * W * y_cs, tab, (int64_t)dm[0] * H * W,
                      Cc, in_cs[i], y_cs, 0);
    } else if (axis == 2) {
      for (int b = 0; b < N && !rc; ++b)
        rc = launch_lut(ctx, src + (int64_t)b * dm[2] * W * in_cs[i],
                        dst + ((int64_t)b * H + offset) * W * y_cs, tab, (int64_t)dm[2] * W, Cc,
                        in_cs[i], y_cs, 0);
    } else {
      for (int b = 0; b < N * H && !rc; ++b)
        rc = launch_lut(ctx, src + (int64_t)b * dm[3] * in_cs[i],
                        dst + ((int64_t)b * W + offset) * y_cs, tab, dm[3], Cc, in_cs[i], y_cs, 0);
    }
    if (rc) return rc;
    offset += dm[axis];
  }
  // channel concat that ends off a 16 boundary: clear the pad channels
  if (axis == 1 && Cc % 16 != 0) {
    const int c1 = std::min(round_up(Cc, 16), y_cs);
    const int64_t total = (int64_t)N * H * W * (c1 - Cc);
    launch(ctx, zero_channels_kernel, dim3(grid_for(total)), dim3(kThreads), (int8_t *)y, (int64_t)N * H * W, y_cs, Cc, c1);
    TPUHIP_CHECK_HIP(hipGetLastError());
  }
  return TPUHIP_OK;
}

}  // extern "C"
