// Convolutions that are no plain implicit GEMM -- groups, zeros inserted between the input's pixels -- as one
// (core/conv.cpp:11-104; core/deconv.cpp for the transposed form, which reaches the kernels as inserted zeros).
//
//   * Inserted zeros.  With S = ins + 1, an output row oh meets real input rows only through the taps kh for which
//     oh * sh - pt + kh * dh is a multiple of S.  Rows that are congruent modulo P = S / gcd(S, sh) meet the same taps at
//     the same distance, so a layer is P_h * P_w convs ("phases") over the input as it lies in memory, each with its own
//     list of (dy, dx) taps, and no multiplication by an inserted zero is left (three quarters of all, doubling a map).
//   * Groups.  A block of 32 output channels reads the input channels of the groups it covers, one contiguous range; the
//     filter of that range is packed with zeros where output and input channel belong to different groups.  32 groups of
//     4 x 4 channels keep an eighth of the matrix pipe's work, which is idle otherwise.
//
// A wave owns TM x 32 output channels x TN x 32 pixels of a phase and feeds the MFMAs straight from memory in fragment
// layout, without LDS for the operands and without barriers: filter fragments are packed as 1 KB runs, an activation
// fragment is one 16-byte load per lane at the position that the table entry of its (tap, 16 channels) names; a position
// outside the image reads zeros through the buffer descriptor.  The table of a phase (two entries per 32-byte K slice,
// one for each half of the wave) sits in LDS.  D slices are in flight per wave.
//
// Bound: the trip to memory at the start (few slices per wave: 9 for 3x3 with 32 channels per block) and the vector L1 at
// 32 bytes per pixel row.  One lane per output element with byte loads, which this replaces, is bound by its serial loads:
// 4 x 128 x 45 x 53, transposed 4x4 stride 2 -> 90 x 106: 8290 us, here 16; 32 groups 3x3: 41 us, here 7.  (8 x 256 x 60 x 60
// transposed: 97 us, 0.6 POP/s.)  Six or eight slices in flight are no faster.
//
// That vector L1 bound is what transposed convs of many channels meet: the 64 lanes of an activation load lie in 32 or 64
// different places, and every phase and channel block loads them again.  They have a kernel of their own,
// conv_gather_patch_kernel, that keeps the input rows of all phases in LDS; patch_plan() says which layers.
#include "conv_gather.hpp"

#include <algorithm>
#include <climits>
#include <cstring>
#include <numeric>
#include <vector>

#include "conv_epilogue.hpp"

namespace tpuhip {

namespace {

struct GatherPhase {
  int oh0, ow0;        // first output row / column
  int qh, qw;          // rows and columns of the phase
  int iy0, ix0;        // input row / column that tap (0, 0) of output (oh0, ow0) stands at
  int slices;          // 32-byte K slices
  uint32_t w;          // byte offset of the phase's packed filter
  uint32_t magic_qw;   // ceil(2^32 / qw); 0 for one column
};

}  // namespace

struct GatherPlan {
  tpuhip_conv_desc d;
  int8_t *w = nullptr;          // packed filters, then a table of max_entries per phase, then the phases
  uint32_t w_bytes = 0;
  uint32_t tab_at = 0, phase_at = 0;
  int n_phases = 0, max_entries = 0, max_pixels = 0;
  int ph = 1, pw = 1, step_h = 1, step_w = 1;   // output rows / columns between two of a phase, input ones between them
  int blocks = 0;               // 32-channel blocks
  int tm = 1;                   // blocks per wave
  // the patch kernel (rows > 0)
  int rows = 0, tiles = 0, waves = 0, groups = 0;   // output rows of a phase per tile, tiles per image, 64-pixel groups per phase
  int row_min = 0, span = 0, col_min = 0, cols = 0; // first input row and column that output (0, 0) reads, rows above each other, columns
  int prow = 0;                                     // bytes of a patch position
  unsigned lds = 0;
};

namespace {

constexpr int64_t kPatchLds = 160 * 1024;
constexpr int kMaxEntries = 2048;   // table entries of a phase, of all phases in the patch kernel (16 and 8 KB of LDS)

struct GatherArgs {   // up to 112 bytes: a launch with more of arguments costs the host 0.5 us more
  const int8_t *x, *w;
  int8_t *y;
  const int32_t *bias, *planes;   // planes: multiplier, rshift and 2^(rshift-1), nparam entries each
  int nparam;
  uint32_t tab_at, phase_at, x_bytes, w_bytes;
  int n, ih, iw, x_cs, oh, ow, y_cs, ocw;
  uint16_t ph, pw, step_h, step_w;
  int ocg, icg;      // channels per group; grouped layers only: the first channel a block reads is that of its first group
  uint16_t entries;  // table entries per phase
  uint8_t relu, relu_first;
};
static_assert(sizeof(GatherArgs) <= 112, "see above");

// one 16-byte chunk of requantised channels per lane and pixel
template <bool FAST>
__device__ __forceinline__ int32_t requant_one(int32_t v, int32_t mult, int32_t rshift, int32_t hpot) {
  const int32_t x = srdhm(v, mult);
  if (FAST) return (x + hpot + (x >> 31)) >> rshift;
  const int32_t mask = (int32_t)((1u << rshift) - 1u);
  return rdbp(x, rshift, mask, mask >> 1);
}

template <int TM, int TN, bool FAST>
__global__ __launch_bounds__(256) void conv_gather_kernel(GatherArgs a) {
  extern __shared__ __attribute__((aligned(16))) int8_t gather_lds[];
  int32_t *sparam = reinterpret_cast<int32_t *>(gather_lds);              // [multiplier, rshift, 2^(rshift-1)][TM * 32]
  int2 *stab = reinterpret_cast<int2 *>(gather_lds + 3 * TM * 32 * 4);
  constexpr int D = 4;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 31, half = lane >> 5;
  const int blk0 = blockIdx.y * TM;
  // the phase, its table and the channels' parameters in one trip to memory
  const int2 *tab = reinterpret_cast<const int2 *>(a.w + a.tab_at) + blockIdx.z * a.entries;
  const GatherPhase p = reinterpret_cast<const GatherPhase *>(a.w + a.phase_at)[blockIdx.z];
  int32_t param = 0;
  if (threadIdx.x < 3 * TM * 32)
    param = a.planes[(int)(threadIdx.x / (TM * 32)) * a.nparam + blk0 * 32 + (int)(threadIdx.x % (TM * 32))];
  for (int i = threadIdx.x; i < a.entries; i += 256) stab[i] = tab[i];
  if (threadIdx.x < 3 * TM * 32) sparam[threadIdx.x] = param;
  __syncthreads();
  const int npix = a.n * p.qh * p.qw;
  const int pix0 = ((int)blockIdx.x * 4 + wave) * (TN * 32);
  if (pix0 >= npix) return;

  const __amdgpu_buffer_rsrc_t xrsrc = __builtin_amdgcn_make_buffer_rsrc((void *)a.x, 0, a.x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t wrsrc = __builtin_amdgcn_make_buffer_rsrc((void *)a.w, 0, a.w_bytes, 0x00020000);
  const int cbase = a.icg ? (blk0 * 32 / a.ocg * a.icg) & ~15 : 0;

  int iy[TN], ix[TN], off[TN], out[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int q = min(pix0 + j * 32 + col, npix - 1);
    const int qw = q % p.qw, t = q / p.qw;
    const int qh = t % p.qh, n = t / p.qh;
    iy[j] = qh * a.step_h + p.iy0;
    ix[j] = qw * a.step_w + p.ix0;
    off[j] = ((n * a.ih + iy[j]) * a.iw + ix[j]) * a.x_cs + cbase;
    out[j] = (n * a.oh + p.oh0 + qh * a.ph) * a.ow + p.ow0 + qw * a.pw;
  }
  uint32_t woff[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i)
    woff[i] = p.w + (uint32_t)((blk0 + i) * p.slices) * 1024u + (uint32_t)lane * 16u;

  v4i af[D][TM], bf[D][TN];
  auto load = [&](int slot, int s) {
    const bool in_k = s < p.slices;
    const int2 e = stab[min(2 * s + half, max(2 * p.slices - 1, 0))];
    const int dy = e.y >> 16, dx = (int)(short)(e.y & 0xffff);
#pragma unroll
    for (int i = 0; i < TM; ++i) af[slot][i] = buffer_load16(wrsrc, in_k ? woff[i] + (uint32_t)s * 1024u : kOobOffset);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const bool ok = in_k & ((unsigned)(iy[j] + dy) < (unsigned)a.ih) & ((unsigned)(ix[j] + dx) < (unsigned)a.iw);
      bf[slot][j] = buffer_load16(xrsrc, ok ? (uint32_t)(off[j] + e.x) : kOobOffset);
    }
  };
  v16i acc[TM][TN];
  const int oc0 = blk0 * 32 + half * 16 * TM;   // a lane's TM * 16 channels are consecutive
#pragma unroll
  for (int d = 0; d < D; ++d) load(d, d);
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const v4i b = *reinterpret_cast<const v4i *>(a.bias + oc0 + i * 16 + q * 4);
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[i][j][q * 4 + e] = b[e];
    }
  for (int s0 = 0; s0 < p.slices; s0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      // slices past the end are zeros in both operands
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[d][i], bf[d][j], acc[i][j], 0, 0, 0);
      load(d, s0 + D + d);
    }
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int oc = oc0 + i * 16;
    if (oc >= a.ocw) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      v4i o;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int32_t *at = sparam + (oc - blk0 * 32) + q * 4;
        const v4i m = *reinterpret_cast<const v4i *>(at);
        const v4i r = *reinterpret_cast<const v4i *>(at + TM * 32);
        const v4i h = *reinterpret_cast<const v4i *>(at + 2 * TM * 32);
        int32_t v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          int32_t s = acc[i][j][q * 4 + e];
          if (a.relu_first) s = max(s, 0);
          v[e] = requant_one<FAST>(s, m[e], r[e], h[e]);
        }
        o[q] = (int)pack_sat4(v[0], v[1], v[2], v[3], a.relu ? 0 : -128);
      }
      if (pix0 + j * 32 + col < npix) *reinterpret_cast<v4i *>(a.y + (int64_t)out[j] * a.y_cs + oc) = o;
    }
  }
}

// ---------------------------------------------------------------------------
// Layers of several phases from a patch in LDS.  A workgroup computes 32 channels of some rows of every phase of one image: the
// input rows that the phases' taps reach, with their borders as zeros, are fetched once, in memory order, and a fragment of any
// tap is one LDS read per lane at the offset that the (phase's) table names.  A wave owns one phase's 32 channels x 64 pixels;
// filter fragments come straight from memory, D slices ahead, and waves of one phase find each other's in the vector L1.  A
// position takes an odd number of 16 bytes in LDS, so that a fragment's lanes spread over the banks.
// What bounds it: 4 x 128 x 45 x 53, 4x4 to 90 x 106, of 7.7 us 2.4 are the launch, 1.1 its MFMAs, the rest the trip of the patch
// into LDS and of the result out; 8 x 256 x 60 x 60 the filter, which every workgroup reads again.  The compiler moves the
// loads of D slices to the end of the loop, to be waited for at once (9.3 us), unless the schedule is held after every MFMA.
// Four blocks of 32 pixels per wave instead of two: 8 x 128 x 60 x 60 17.0 us against 17.9, but 4 x 256 x 30 x 30 9.7 against 8.4.
// Against the kernel above: 4 x 128 x 45 x 53 13.5 -> 7.7 us, 1 x 128 x 14 x 14 5.6 -> 4.1, 3 x 160 x 25 x 49 9.1 -> 6.4,
// 8 x 256 x 60 x 60 90 -> 50, 8 x 64 x 60 x 60 10.1 -> 8.5; 3x3 of 4 x 128 x 30 x 30 6.1 -> 4.6; 2x2 of 8 x 256 x 60 x 60 38 -> 28.
// ---------------------------------------------------------------------------
struct GatherPatchArgs {
  const int8_t *x, *w;
  int8_t *y;
  const int32_t *bias, *planes;
  int nparam;
  uint32_t tab_at, phase_at, w_bytes;
  uint32_t magic_row, magic_c16;        // ceil(2^32 / 16-byte chunks of a patch row), ceil(2^32 / those of a position); 0 for one
  uint16_t ih, iw, x_cs, oh, ow, y_cs, ocw, cols, prow;
  int16_t row_min, col_min;
  uint16_t rows, span, tiles, blocks, per_xcd, n_tiles, entries, phases;
  uint8_t groups, ph, pw, step_h, step_w, relu, relu_first;
};
static_assert(sizeof(GatherPatchArgs) <= 112, "see above");

__device__ __forceinline__ int div_by(uint32_t v, uint32_t magic) { return magic ? (int)__umulhi(v, magic) : (int)v; }

template <bool FAST>
__global__ __launch_bounds__(1024) void conv_gather_patch_kernel(GatherPatchArgs a) {
  extern __shared__ __attribute__((aligned(16))) int8_t gather_lds[];
  constexpr int D = 8, NB = 2;
  int32_t *const sparam = reinterpret_cast<int32_t *>(gather_lds);              // [multiplier, rshift, 2^(rshift-1)][32]
  int32_t *const stab = sparam + 3 * 32;
  int8_t *const patch = gather_lds + 3 * 32 * 4 + (int)a.phases * a.entries * 4;
  const int tid = threadIdx.x, nt = blockDim.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = nt >> 6;
  const int col = lane & 31, half = lane >> 5;
  const int logical = (int)(blockIdx.x & 7) * a.per_xcd + (int)(blockIdx.x >> 3);
  if (logical >= a.n_tiles) return;
  const int tile = logical / a.blocks, blk = logical - tile * a.blocks;
  const int img = tile / a.tiles, r0 = (tile - img * a.tiles) * a.rows;

  // ---- the patch: every chunk of it is loaded, one outside the image as zeros
  const int c16 = a.x_cs >> 4, row_chunks = a.cols * c16;
  const int total = ((a.rows - 1) * a.step_h + a.span) * row_chunks;
  const __amdgpu_buffer_rsrc_t xrsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void *)(a.x + (size_t)img * a.ih * a.iw * a.x_cs), 0, (uint32_t)a.ih * a.iw * a.x_cs, 0x00020000);
  const __amdgpu_buffer_rsrc_t wrsrc = __builtin_amdgcn_make_buffer_rsrc((void *)a.w, 0, a.w_bytes, 0x00020000);
  const int y_first = r0 * a.step_h + a.row_min;
  constexpr int NP = 4;
  auto fetch = [&](int q, v4i &v, int &at) {
    const int row = div_by((uint32_t)q, a.magic_row), in_row = q - row * row_chunks;
    const int pos = div_by((uint32_t)in_row, a.magic_c16), ch = in_row - pos * c16;
    const int iy = y_first + row, ix = a.col_min + pos;
    const bool ok = (q < total) & ((unsigned)iy < (unsigned)a.ih) & ((unsigned)ix < (unsigned)a.iw);
    v = buffer_load16(xrsrc, ok ? (uint32_t)((iy * a.iw + ix) * c16 + ch) * 16u : kOobOffset);
    at = (row * a.cols + pos) * a.prow + ch * 16;
  };
  v4i pv[NP];
  int pat[NP];
#pragma unroll
  for (int u = 0; u < NP; ++u) fetch(tid + u * nt, pv[u], pat[u]);
  int32_t param = 0;   // (a workgroup has two waves at least: one per phase)
  if (tid < 96) param = a.planes[(tid >> 5) * a.nparam + blk * 32 + (tid & 31)];
  const int32_t *tab = reinterpret_cast<const int32_t *>(a.w + a.tab_at);
  const GatherPhase *phases = reinterpret_cast<const GatherPhase *>(a.w + a.phase_at);

  for (int i = tid; i < (int)a.phases * a.entries; i += nt) stab[i] = tab[i];
  if (tid < 96) sparam[tid] = param;

  // ---- the wave's phase and pixels; its first filter fragments are on their way while the patch arrives
  const int ph = wave / a.groups, grp = wave - ph * a.groups;
  const GatherPhase p = phases[ph];
  const uint32_t lane16 = (uint32_t)lane * 16u;
  int wslice = p.slices ? (int)p.w + blk * p.slices * 1024 : 0;   // (the scalar offset is not range-checked)
  const int wlast = wslice + max(p.slices - 1, 0) * 1024;
  v4i af[D];
  auto load_A = [&](v4i &dst) {   // one slice after the other; past the last it is repeated and never used
    dst = (v4i)__builtin_amdgcn_raw_buffer_load_b128(wrsrc, lane16, wslice, 0);
    wslice = min(wslice + 1024, wlast);
  };
#pragma unroll
  for (int d = 0; d < D; ++d) load_A(af[d]);
#pragma unroll
  for (int u = 0; u < NP; ++u)
    if (tid + u * nt < total) *reinterpret_cast<v4i *>(patch + pat[u]) = pv[u];
  for (int q = tid + NP * nt; q < total; q += NP * nt) {
#pragma unroll
    for (int u = 0; u < NP; ++u) fetch(q + u * nt, pv[u], pat[u]);
#pragma unroll
    for (int u = 0; u < NP; ++u)
      if (q + u * nt < total) *reinterpret_cast<v4i *>(patch + pat[u]) = pv[u];
  }
  const int npix = min((int)a.rows, p.qh - r0) * p.qw;
  int base[NB], out[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int q = max(min(grp * NB * 32 + j * 32 + col, npix - 1), 0);
    const int qh = div_by((uint32_t)q, p.magic_qw), qw = q - qh * p.qw;
    base[j] = (qh * a.step_h * a.cols + qw * a.step_w) * a.prow;
    out[j] = (img * a.oh + p.oh0 + (r0 + qh) * a.ph) * a.ow + p.ow0 + qw * a.pw;
  }
  const int oc0 = blk * 32 + half * 16;
  v16i acc[NB];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const v4i b = *reinterpret_cast<const v4i *>(a.bias + oc0 + q * 4);
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[j][q * 4 + e] = b[e];
  }
  __syncthreads();
  if (grp * NB * 32 >= npix) return;

  // what is not an MFMA stands behind one: the next slice's pixel fragments, the filter fragment D slices ahead
  const int32_t *const my = stab + ph * a.entries + half;
  v4i bf[2][NB];
  int next = my[2];
  {
    const int at = my[0];
#pragma unroll
    for (int j = 0; j < NB; ++j) bf[0][j] = *reinterpret_cast<const v4i *>(patch + base[j] + at);
  }
  int s0 = 0;
  auto slice = [&](auto dc, bool request) {
    constexpr int d = decltype(dc)::value;
    const int after = my[2 * (s0 + d + 2)];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      acc[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[d], bf[d & 1][j], acc[j], 0, 0, 0);
      bf[(d + 1) & 1][j] = *reinterpret_cast<const v4i *>(patch + base[j] + next);
      if (request && j == NB - 1) load_A(af[d]);
      __builtin_amdgcn_sched_barrier(0);
    }
    next = after;
  };
  for (; s0 + D <= p.slices; s0 += D) static_for<D>([&](auto dc) { slice(dc, true); });
  static_for<D - 1>([&](auto dc) {
    if (s0 + decltype(dc)::value < p.slices) slice(dc, false);
  });

  if (oc0 >= a.ocw) return;
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    v4i o;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int32_t *at = sparam + half * 16 + q * 4;
      const v4i m = *reinterpret_cast<const v4i *>(at);
      const v4i r = *reinterpret_cast<const v4i *>(at + 32);
      const v4i h = *reinterpret_cast<const v4i *>(at + 64);
      int32_t v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        int32_t s = acc[j][q * 4 + e];
        if (a.relu_first) s = max(s, 0);
        v[e] = requant_one<FAST>(s, m[e], r[e], h[e]);
      }
      o[q] = (int)pack_sat4(v[0], v[1], v[2], v[3], a.relu ? 0 : -128);
    }
    if (grp * NB * 32 + j * 32 + col < npix) *reinterpret_cast<v4i *>(a.y + (int64_t)out[j] * a.y_cs + oc0) = o;
  }
}

uint32_t magic_of(int d) { return d == 1 ? 0u : (uint32_t)(((1ull << 32) + d - 1) / d); }

int floor_div(int a, int b) { return a >= 0 ? a / b : -((-a + b - 1) / b); }

// The patch kernel's tiles, where the layer is the patch kernel's; rows stays 0 elsewhere.  It needs several phases, at most
// 16 waves of 64 pixels for one row of all of them, and their patch in LDS.  Fewer than eight slices are in flight at once
// without it, and nothing is shared: 64 -> 64 channels, 2x2 on 2 x 40 x 40 3.8 us, in the patch kernel 4.0.
// From eight slices on, of 2482 layers (profiles/conv_transposed_kernels.txt: 2 to 16 phases, 32 to 512 channels to 24 to 256):
//   * four phases and fewer: faster in the patch kernel (4x4, 128 -> 128 on 8 x 45 x 53 14.7 us, without 23.2; 2x2, 352 -> 24 on
//     250 x 250 10.5 and 25.2), but for two kinds.  A layer of a single block of 32 channels and few outputs has less to fetch
//     without the patch, whose first row waits for the last (4x4, 64 -> 24 on 45 x 53 4.4 us, 5.0 with it; eight images of it 7.1
//     and 6.3) -- not where positions lie 128 bytes apart or a multiple, which the gathering loads are slower from (128 -> 24
//     on 45 x 53 5.8 and 5.7, 192 -> 24 5.7 and 6.2).
//     And where the chip is filled many times over, a patch's way into LDS is paid by every block of channels and no wait is
//     left to save: fewer than twelve slices of fewer than 128 channels (4x4, 64 -> 128 on 8 x 100 x 90 35.0 us, 39.4 with it);
//   * more phases: a workgroup has a wave for each, so that its tiles hold a few pixels, which the same many rows of patch are
//     fetched for.  6x6 to three times the size, 64 -> 64 on 16 x 60 x 60 31.1 us, 39.1 with it.  The patch is faster on many
//     outputs and from 128 channels (128 -> 64: 54.2 us, 44.7 with it) or 16 slices on.
// By that line (few: 144 outputs x blocks a CU; many: 1800) the layers take 0.4 % longer than with the faster kernel each, at
// most 1.34 times; all in the patch kernel 2.0 % and 1.63, none 22 % and 3.6.
// The rows of a tile: fewest groups of 64 pixels on the busiest CU, a tile's start counted as one more.  (4 x 128 x 45 x 53:
// three rows 8.0 us, one 8.9, two 9.7, four 9.3; 4 x 256 x 30 x 30: one 12.2, two and four 8.8.)
void patch_plan(int num_cu, const tpuhip_conv_desc &d, GatherPlan *g) {
  const int sh = d.ins_h + 1, sw = d.ins_w + 1;
  const int ph = sh / std::gcd(sh, d.sh), pw = sw / std::gcd(sw, d.sw);
  const int step_h = ph * d.sh / sh, step_w = pw * d.sw / sw;
  // one phase of results -- no zeros that matter, or a result of one row or column across them -- shares its patch with none (and
  // would leave the kernel a workgroup of one wave, which does not fetch all of its block's parameters)
  const int nh = std::min(ph, d.oh), nw = std::min(pw, d.ow);
  if (d.g != 1 || nh * nw == 1 || ph * pw > 64 || d.x_cs % 16 || d.x_cs > 4096 || step_h > 255 || step_w > 255) return;
  for (int v : {d.ih, d.iw, d.oh, d.ow, d.kh * d.dh, d.kw * d.dw, d.pt, d.pl})
    if (v >= 30000) return;
  if (d.y_cs > 65535 || (int64_t)d.ih * d.iw * d.x_cs >= (1ll << 31) - 1 || (int64_t)d.n * d.oh * d.ow >= (1ll << 31)) return;
  // what the taps of all phases reach
  int row_min = INT_MAX, row_max = INT_MIN, col_min = INT_MAX, col_max = INT_MIN, taps_max = 0;
  const int qh = (d.oh + ph - 1) / ph, qw = (d.ow + pw - 1) / pw;
  for (int a = 0; a < nh; ++a)
    for (int b = 0; b < nw; ++b) {
      int taps = 0;
      for (int kh = 0; kh < d.kh; ++kh)
        for (int kw = 0; kw < d.kw; ++kw) {
          const int y = a * d.sh - d.pt + kh * d.dh, x = b * d.sw - d.pl + kw * d.dw;
          const int iy = floor_div(y, sh), ix = floor_div(x, sw);
          if (iy * sh != y || ix * sw != x) continue;
          row_min = std::min(row_min, iy); row_max = std::max(row_max, iy);
          col_min = std::min(col_min, ix); col_max = std::max(col_max, ix);
          ++taps;
        }
      taps_max = std::max(taps_max, taps);
    }
  if (!taps_max || row_min < -30000 || col_min < -30000) return;
  const int n16 = (round_up(d.ic, 16)) / 16, slices = (taps_max * n16 + 1) / 2;
  const int entries = 2 * (round_up(slices, 4) + 4), phases = nh * nw;
  if (entries * phases > kMaxEntries || slices < 8) return;
  const int blocks = (d.oc + 31) / 32;
  const int64_t work = (int64_t)d.n * d.oh * d.ow * blocks;
  const bool few = work < 144 * (int64_t)num_cu, many = work > 1800 * (int64_t)num_cu;
  if (phases <= 4 ? (few && blocks == 1 && d.x_cs % 128) || (many && slices < 12 && d.x_cs < 128)
                  : few || (slices < 16 && d.x_cs < 128))
    return;
  const int prow = d.x_cs + (d.x_cs % 32 ? 0 : 16);   // an odd number of 16 bytes: the lanes of a fragment spread over the banks
  const int64_t cols = (int64_t)(qw - 1) * step_w + col_max - col_min + 1, span = row_max - row_min + 1;
  int64_t best = INT64_MAX;
  for (int rows = 1; rows <= qh; ++rows) {
    const int64_t lds = 3 * 32 * 4 + (int64_t)phases * entries * 4 + ((rows - 1) * (int64_t)step_h + span) * cols * prow;
    const int groups = (rows * qw + 63) / 64, tiles = (qh + rows - 1) / rows;
    const int64_t wgs = (int64_t)d.n * tiles * blocks;
    if (lds > kPatchLds || groups * phases > 16) break;
    if (wgs >= 65536 || tiles >= 65536 || cols > 30000) continue;
    const int64_t cost = (wgs + num_cu - 1) / num_cu * (groups * phases + 1);
    if (cost >= best) continue;
    best = cost;
    g->rows = rows;
    g->tiles = tiles;
    g->groups = groups;
    g->waves = groups * phases;
    g->lds = (unsigned)lds;
  }
  if (!g->rows) return;
  g->row_min = row_min;
  g->span = (int)span;
  g->col_min = col_min;
  g->cols = (int)cols;
  g->prow = prow;
  g->max_entries = entries;
}

// A layer's plan, phases and tables, and its packed filter; filter NULL: all but the bytes of the filter.
struct GatherLayer {
  GatherPlan plan;
  std::vector<GatherPhase> phases;
  std::vector<std::vector<int2>> tabs;
  std::vector<int8_t> w;
};

// false: not the gather kernels' layer.  patch: whether it may go to the patch kernel
bool gather_layer(int num_cu, const tpuhip_conv_desc &d, const int8_t *filter, bool patch, GatherLayer *out) {
  const int icg = d.ic / d.g, ocg = d.oc / d.g;
  const int sh = d.ins_h + 1, sw = d.ins_w + 1;
  const int ph = sh / std::gcd(sh, d.sh), pw = sw / std::gcd(sw, d.sw);
  *out = GatherLayer();
  GatherPlan &geo = out->plan;
  if (patch) patch_plan(num_cu, d, &geo);
  // without groups all blocks read the same input channels: two of them per wave halve the activation loads
  const int tm = d.g == 1 && d.oc > 32 && !geo.rows ? 2 : 1;
  const int blocks = round_up(d.oc, 32 * tm) / 32;
  // 16-channel groups that a block reads: from the first channel of its first group, down to a multiple of 16
  int n16 = 0;
  for (int b = 0; b < blocks; ++b) {
    if (b * 32 >= d.oc) break;
    const int first = (b * 32 / ocg * icg) & ~15;
    const int last = (std::min(b * 32 + 31, d.oc - 1) / ocg + 1) * icg;
    n16 = std::max(n16, (last - first + 15) / 16);
  }
  // where it does not apply: a table entry holds its tap as two 16-bit distances, a phase's table fits its share of LDS,
  // and every packed filter byte is addressed with 32 bits
  if (d.x_cs % 16 || ph * pw > 256 || (int64_t)d.kh * d.dh >= 30000 || (int64_t)d.kw * d.dw >= 30000 || d.ih >= 30000 ||
      d.iw >= 30000 || d.sh >= 256 || d.sw >= 256 || (int64_t)d.kh * d.kw * n16 + 2 > kMaxEntries ||
      (int64_t)blocks * ((int64_t)d.kh * d.kw * n16 + 2 * ph * pw) * 512 >= (1ll << 30))
    return false;

  auto &phases = out->phases;
  auto &tabs = out->tabs;
  auto &w = out->w;
  size_t w_bytes = 0;
  int max_entries = 0, max_pixels = 0;
  struct Tap { int kh, kw, dy, dx; };
  for (int a = 0; a < std::min(ph, d.oh); ++a)
    for (int b = 0; b < std::min(pw, d.ow); ++b) {
      GatherPhase p{};
      p.oh0 = a;
      p.ow0 = b;
      p.qh = (d.oh - a + ph - 1) / ph;
      p.qw = (d.ow - b + pw - 1) / pw;
      // position of tap (kh, kw) of the phase's first output, in the input with its zeros: divisible or no tap
      const int y0 = a * d.sh - d.pt, x0 = b * d.sw - d.pl;
      p.iy0 = floor_div(y0, sh);
      p.ix0 = floor_div(x0, sw);
      std::vector<Tap> taps;
      for (int kh = 0; kh < d.kh; ++kh)
        for (int kw = 0; kw < d.kw; ++kw) {
          const int y = y0 + kh * d.dh, x = x0 + kw * d.dw;
          if (floor_div(y, sh) * sh != y || floor_div(x, sw) * sw != x) continue;
          taps.push_back({kh, kw, floor_div(y, sh) - p.iy0, floor_div(x, sw) - p.ix0});
        }
      const int entries = (int)taps.size() * n16;
      p.slices = (entries + 1) / 2;
      p.magic_qw = magic_of(p.qw);
      p.w = (uint32_t)w_bytes;
      std::vector<int2> tab;
      for (int e = 0; e < 2 * p.slices; ++e) {
        // the second half of an odd last slice: zeros in the filter, and the last real tap's position, which the patch holds
        // whatever taps the phase has
        const Tap t = taps[std::min(e, entries - 1) / n16];
        int2 v;
        v.x = (int)(((int64_t)t.dy * d.iw + t.dx) * d.x_cs) + (e < entries ? e % n16 : 0) * 16;
        v.y = (int)(((uint32_t)t.dy << 16) | ((uint32_t)t.dx & 0xffffu));
        tab.push_back(v);
      }
      tabs.push_back(std::move(tab));
      w_bytes += (size_t)blocks * p.slices * 1024;
      if (filter) w.resize(w_bytes, 0);
      for (int blk = 0; blk < blocks && filter; ++blk) {
        const int c_first = d.g == 1 ? 0 : (blk * 32 / ocg * icg) & ~15;
        for (int row = 0; row < 32; ++row) {
          const int oc = blk / tm * tm * 32 + mfma_row_to_oc(blk % tm * 32 + row, tm);
          if (oc >= d.oc) continue;
          const int g = oc / ocg;
          for (int e = 0; e < entries; ++e) {
            const Tap &t = taps[e / n16];
            int8_t *to = w.data() + p.w + ((size_t)(blk * p.slices + e / 2) * 64 + row + 32 * (e & 1)) * 16;
            for (int k = 0; k < 16; ++k) {
              const int c = c_first + (e % n16) * 16 + k - g * icg;   // channel within the group
              if (c >= 0 && c < icg) to[k] = filter[(((size_t)oc * icg + c) * d.kh + t.kh) * d.kw + t.kw];
            }
          }
        }
      }
      max_entries = std::max(max_entries, 2 * p.slices);
      max_pixels = std::max(max_pixels, d.n * p.qh * p.qw);
      phases.push_back(p);
    }
  if (geo.rows) {
    // table entries of the patch kernel: LDS bytes, a number for all phases that covers its look ahead
    max_entries = geo.max_entries;
    for (size_t i = 0; i < tabs.size(); ++i) {
      std::vector<int2> t(geo.max_entries / 2, int2{0, 0});
      for (size_t e = 0; e < tabs[i].size(); ++e) {
        const int dy = tabs[i][e].y >> 16, dx = (int16_t)(tabs[i][e].y & 0xffff);
        const int c = tabs[i][e].x - (int)(((int64_t)dy * d.iw + dx) * d.x_cs);
        const int at = ((phases[i].iy0 + dy - geo.row_min) * geo.cols + phases[i].ix0 + dx - geo.col_min) * geo.prow + c;
        (e & 1 ? t[e / 2].y : t[e / 2].x) = at;
      }
      tabs[i] = std::move(t);
    }
  }
  geo.d = d;
  geo.n_phases = (int)phases.size();
  geo.max_entries = max_entries;
  geo.max_pixels = max_pixels;
  geo.ph = ph;
  geo.pw = pw;
  geo.step_h = ph * d.sh / sh;
  geo.step_w = pw * d.sw / sw;
  geo.blocks = blocks;
  geo.tm = tm;
  geo.w_bytes = (uint32_t)std::max<size_t>(w_bytes, 16);
  return true;
}

}  // namespace

int gather_prepack(tpuhip_ctx *ctx, const tpuhip_conv_desc &d, const int8_t *filter, GatherPlan **out) {
  *out = nullptr;
  GatherLayer l;
  if (!gather_layer(ctx->num_cu, d, filter, true, &l)) return TPUHIP_OK;
  if (l.plan.lds > 64 * 1024)
    for (const void *kernel : {(const void *)conv_gather_patch_kernel<true>, (const void *)conv_gather_patch_kernel<false>})
      if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kPatchLds) != hipSuccess) {
        (void)hipGetLastError();
        (void)gather_layer(ctx->num_cu, d, filter, false, &l);
        break;
      }
  auto *plan = new GatherPlan(l.plan);
  const size_t tab_bytes = (size_t)plan->max_entries * (plan->rows ? sizeof(int) : sizeof(int2));
  const size_t tab_at = plan->w_bytes, phase_at = tab_at + std::max<size_t>(l.tabs.size() * tab_bytes, 16);
  std::vector<int8_t> image(phase_at + l.phases.size() * sizeof(GatherPhase), 0);
  if (!l.w.empty()) memcpy(image.data(), l.w.data(), l.w.size());
  for (size_t i = 0; i < l.tabs.size(); ++i)
    if (!l.tabs[i].empty()) memcpy(image.data() + tab_at + i * tab_bytes, l.tabs[i].data(), l.tabs[i].size() * sizeof(int2));
  memcpy(image.data() + phase_at, l.phases.data(), l.phases.size() * sizeof(GatherPhase));
  plan->tab_at = (uint32_t)tab_at;
  plan->phase_at = (uint32_t)phase_at;
  int rc = tpuhip_malloc(ctx, image.size(), (void **)&plan->w);
  if (!rc) rc = stage_upload(ctx, plan->w, image.data(), image.size());
  if (rc) {
    gather_destroy(ctx, plan);
    return rc;
  }
  *out = plan;
  return TPUHIP_OK;
}

int gather_form(const tpuhip_conv_desc &d, int num_cu, int *reach) {
  GatherLayer l;
  if (!gather_layer(num_cu, d, nullptr, true, &l)) return 0;
  const GatherPlan &g = l.plan;
  if (!g.rows) return 1;
  const int patch = 3 * 32 * 4 + g.n_phases * g.max_entries * 4;
  int64_t low = 0, high = 0;
  for (size_t i = 0; i < l.phases.size(); ++i) {
    const GatherPhase &p = l.phases[i];
    const int64_t last = ((int64_t)(std::min(g.rows, p.qh) - 1) * g.step_h * g.cols + (int64_t)(p.qw - 1) * g.step_w) * g.prow;
    for (const int2 &e : l.tabs[i])
      for (int at : {e.x, e.y}) {
        low = std::min<int64_t>(low, at);
        high = std::max<int64_t>(high, last + at);
      }
  }
  if (reach) {
    const int64_t r[5] = {patch, patch + low, patch + high + 16, (int64_t)g.lds, g.waves * 64};
    for (int i = 0; i < 5; ++i) reach[i] = (int)std::clamp<int64_t>(r[i], INT_MIN, INT_MAX);
  }
  return 2;
}

void gather_destroy(tpuhip_ctx *ctx, GatherPlan *plan) {
  if (!plan) return;
  if (plan->w) (void)tpuhip_free(ctx, plan->w);
  delete plan;
}

int gather_run(tpuhip_ctx *ctx, const GatherPlan *plan, const void *x, void *y, const int32_t *bias, const int32_t *planes,
               int nparam, bool fast) {
  const tpuhip_conv_desc &d = plan->d;
  if (plan->rows) {
    GatherPatchArgs a{};
    a.x = (const int8_t *)x;
    a.w = plan->w;
    a.y = (int8_t *)y;
    a.bias = bias;
    a.planes = planes;
    a.nparam = nparam;
    a.tab_at = plan->tab_at;
    a.phase_at = plan->phase_at;
    a.w_bytes = plan->w_bytes;
    a.magic_row = magic_of(plan->cols * (d.x_cs / 16));
    a.magic_c16 = magic_of(d.x_cs / 16);
    a.ih = (uint16_t)d.ih; a.iw = (uint16_t)d.iw; a.x_cs = (uint16_t)d.x_cs;
    a.oh = (uint16_t)d.oh; a.ow = (uint16_t)d.ow; a.y_cs = (uint16_t)d.y_cs; a.ocw = (uint16_t)round_up(d.oc, 16);
    a.cols = (uint16_t)plan->cols; a.prow = (uint16_t)plan->prow;
    a.row_min = (int16_t)plan->row_min; a.col_min = (int16_t)plan->col_min;
    a.rows = (uint16_t)plan->rows; a.span = (uint16_t)plan->span;
    a.tiles = (uint16_t)plan->tiles; a.blocks = (uint16_t)plan->blocks;
    const int n_tiles = d.n * plan->tiles * plan->blocks, per_xcd = (n_tiles + 7) / 8;
    a.n_tiles = (uint16_t)n_tiles; a.per_xcd = (uint16_t)per_xcd;
    a.entries = (uint16_t)plan->max_entries; a.phases = (uint16_t)plan->n_phases; a.groups = (uint8_t)plan->groups;
    a.ph = (uint8_t)plan->ph; a.pw = (uint8_t)plan->pw; a.step_h = (uint8_t)plan->step_h; a.step_w = (uint8_t)plan->step_w;
    a.relu = d.do_relu && !d.relu_first;
    a.relu_first = (d.do_relu && d.relu_first) ? 1 : 0;
    const dim3 grid((unsigned)(per_xcd * 8)), block((unsigned)(plan->waves * 64));
    auto go = [&](auto kernel) {
      if (ctx->prof_start)
        hipExtLaunchKernelGGL(kernel, grid, block, plan->lds, ctx->stream, ctx->prof_start, ctx->prof_stop, 0, a);
      else
        hipLaunchKernelGGL(kernel, grid, block, plan->lds, ctx->stream, a);
    };
    fast ? go(conv_gather_patch_kernel<true>) : go(conv_gather_patch_kernel<false>);
    TPUHIP_CHECK_HIP(hipGetLastError());
    return TPUHIP_OK;
  }
  GatherArgs a{};
  a.x = (const int8_t *)x;
  a.y = (int8_t *)y;
  a.w = plan->w;
  a.tab_at = plan->tab_at;
  a.phase_at = plan->phase_at;
  a.entries = (uint16_t)plan->max_entries;
  a.bias = bias;
  a.planes = planes;
  a.nparam = nparam;
  a.x_bytes = (uint32_t)((int64_t)d.n * d.ih * d.iw * d.x_cs);
  a.w_bytes = plan->w_bytes;
  a.n = d.n; a.ih = d.ih; a.iw = d.iw; a.x_cs = d.x_cs;
  a.oh = d.oh; a.ow = d.ow; a.y_cs = d.y_cs; a.ocw = round_up(d.oc, 16);
  a.ph = (uint16_t)plan->ph; a.pw = (uint16_t)plan->pw;
  a.step_h = (uint16_t)plan->step_h; a.step_w = (uint16_t)plan->step_w;
  a.ocg = d.oc / d.g;
  a.icg = d.g > 1 ? d.ic / d.g : 0;
  a.relu = d.do_relu && !d.relu_first;
  a.relu_first = (d.do_relu && d.relu_first) ? 1 : 0;
  // 64 pixels per wave where that still gives every SIMD two waves, else 32
  const int groups = plan->blocks / plan->tm;
  const int64_t waves = (int64_t)((plan->max_pixels + 63) / 64) * groups * plan->n_phases;
  const bool wide = waves >= (int64_t)ctx->num_cu * 8;
  const int per_wg = wide ? 256 : 128;
  const dim3 grid((unsigned)((plan->max_pixels + per_wg - 1) / per_wg), (unsigned)groups, (unsigned)plan->n_phases), block(256);
  const unsigned lds = (unsigned)(3 * plan->tm * 32 * 4 + std::max(plan->max_entries, 1) * sizeof(int2));
  auto go = [&](auto kernel) {
    if (ctx->prof_start)
      hipExtLaunchKernelGGL(kernel, grid, block, lds, ctx->stream, ctx->prof_start, ctx->prof_stop, 0, a);
    else
      hipLaunchKernelGGL(kernel, grid, block, lds, ctx->stream, a);
  };
  if (plan->tm == 2) {
    if (wide) fast ? go(conv_gather_kernel<2, 2, true>) : go(conv_gather_kernel<2, 2, false>);
    else fast ? go(conv_gather_kernel<2, 1, true>) : go(conv_gather_kernel<2, 1, false>);
  } else {
    if (wide) fast ? go(conv_gather_kernel<1, 2, true>) : go(conv_gather_kernel<1, 2, false>);
    else fast ? go(conv_gather_kernel<1, 1, true>) : go(conv_gather_kernel<1, 1, false>);
  }
  TPUHIP_CHECK_HIP(hipGetLastError());
  return TPUHIP_OK;
}

}  // namespace tpuhip
