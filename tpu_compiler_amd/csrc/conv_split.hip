// Convs of few outputs, one image of a network from 56 x 56 down: K split over the waves of a workgroup, blocks of 16 channels x
// 16 pixels on v_mfma_i32_16x16x64_i8.
//
// Such a layer is a chain -- launch, arguments, operands, one meeting of the partial sums, requantisation, store -- whose
// longest link is the operands' way into a CU, some 24 bytes a clock.  With blocks of 32 x 32 a 3x3 layer of 512 channels on
// 7 x 7 is 32 workgroups that fetch 295 KB each, 5.1 of its 6.7 us; blocks of 16 x 16 are four times as many that fetch half of
// it.  Where the window overlaps itself the input comes once, as a patch in LDS that holds what the tile's rows (or part of a row)
// reach, and only the filter comes in fragments: 16 channels x 52 outputs of 512 -> 1024 on 13 x 13 fetch 120 KB, where im2col
// fetches 313.
//
// A workgroup of KW x PW waves owns 16 * OB channels of PW * NB blocks of pixels; wave (k, g) multiplies slices k, k + KW, ... of
// 64 bytes of K for the NB blocks of pixel group g.  The filter is packed fragment by fragment (1 KB loads), patch_depth() or
// kDepth slices of a wave in flight before anything is waited for.  The partial sums meet in LDS behind one barrier; every block is finished by one
// wave, four channels of a pixel per lane.
//
// Replayed from a graph (a launch of nothing is 1.7 us there), against the best of the other forms: 3x3 of 512 channels on 7 x 7
// 6.7 -> 3.9 us, 256 on 14 x 14 4.8 -> 3.35, 64 on 56 x 56 3.2 -> 2.8, 256 -> 512 on 26 x 26 6.8 -> 5.3, 512 -> 1024 on 13 x 13
// 7.1 -> 4.8, at stride 2 from 26 x 26 7.1 -> 5.6; 1x1 2048 -> 512 on 7 x 7 4.5 -> 3.1, 1024 -> 256 on 14 x 14 3.4 -> 2.6; 5x5 at
// stride 2, 128 channels on 4 x 45 x 53, 8.9 -> 5.7.  What is left of the large ones is the same link: 112 KB per CU at 26 x 26 are
// 1.9 us.
#include "conv_split.hpp"

#include "conv_epilogue.hpp"

#include <algorithm>

namespace {

constexpr int kLdsBytes = 160 * 1024;
constexpr int kDepth = 4;        // gather form: slices in flight
constexpr int kPatchLoads = 8;   // patch form: 16-byte loads of a thread in flight
// Patch form: slices of the filter in flight per wave.  Eight waves: three.  All of a wave's at once, up to nine, take the registers
// of another workgroup and are waited for together: of 56 layers, over all variants, three are 9 % faster in the mean than all of
// up to three, five and nine, the fastest variants 5.5 % (512 -> 1024 on 13 x 13: 4.93, 4.85 and 5.22 us with two, three and nine,
// and where the filter comes from beyond the L2s 5.37 and 6.14 with three and nine; 512 on 7 x 7 4.05, 3.91, 3.95, 4.72 and 4.85);
// four are 3 % slower than three.  Four waves have half as much in flight with as many, which is too little where the filter comes
// from afar: 512 on 7 x 7 5.68, 4.79 and 4.80 us with three, six and nine, 256 on 14 x 14 3.62, 3.62 and 3.51.  Six where a slice
// straddles taps (337 channels on 17 x 36: nine 8 % slower).
constexpr int patch_depth(int waves, bool uni) { return waves > 4 ? 3 : uni ? 9 : 6; }

// x / d for x * d < 2^32, d = 1 too, without a branch: magic = floor((2^32 - 1) / d)
__device__ __forceinline__ uint32_t div_by(uint32_t x, uint32_t magic) { return __umulhi(x + 1, magic); }

template <bool FAST>
__device__ __forceinline__ int32_t requant_one(int32_t v, int32_t mult, int32_t shift, int32_t hpot) {
  const int32_t x = srdhm(v, mult);
  if (FAST) return (x + hpot + (x >> 31)) >> shift;
  const int32_t mask = (int32_t)((1u << shift) - 1u);
  return rdbp(x, shift, mask, mask >> 1);
}

// UNI: the channels are a multiple of 64, a slice lies within one tap.
template <int KW, int PW, int NB, int OB, bool FAST, bool UNI, bool PATCH, bool POST>
__device__ __forceinline__ void split_body(const SplitArgs &a, const SplitPost *post) {
  // named here, the arguments leave the scalar cache together instead of one by one where they are first needed
  asm volatile("" ::"s"(a.x), "s"(a.w), "s"(a.bias), "s"(a.x_bytes), "s"(a.n_tiles), "s"(a.n_pix), "s"(a.shape), "s"(a.magic_tile),
               "s"(a.magic_img), "s"(a.magic_row), "s"(a.magic_c16), "s"(a.magic_kw), "s"(a.magic_pw), "s"((int)a.per_img), "s"((int)a.ih),
               "s"(a.x_cs), "s"((int)a.sh), "s"((int)a.dh), "s"((int)a.slices_pad_relu), "s"((int)a.oc));
  extern __shared__ v4i lds[];   // the patch, [group][wave of K][block][lane] sums, the table's 256 bytes
  constexpr int T = KW * PW * 64, B = NB * OB, FIN = (B + KW - 1) / KW;   // FIN: blocks that a wave finishes
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wave % KW, wg = wave / KW;
  const uint32_t tiles_per_xcd = (a.n_tiles + 7) >> 3;
  const uint32_t wt = (blockIdx.x & 7) * tiles_per_xcd + (blockIdx.x >> 3);
  if (wt >= a.n_tiles) return;                 // uniform over the workgroup
  const uint32_t n_oc = (a.oc + 16 * OB - 1) / (16 * OB);
  uint32_t pix_tile, oc_tile;
  const uint32_t major = div_by(wt, a.magic_tile);
  if (a.n_pix) {
    oc_tile = major;
    pix_tile = wt - major * a.n_pix;
  } else {
    pix_tile = major;
    oc_tile = wt - major * n_oc;
  }
  const int oc0 = (int)oc_tile * (16 * OB);
  const int slices = a.slices_pad_relu >> 4, groups = 4 * slices - (a.slices_pad_relu >> 2 & 3);   // groups of 16 bytes of K
  const int px = lane & 15, chunk = lane >> 4;
  const __amdgpu_buffer_rsrc_t xrsrc = __builtin_amdgcn_make_buffer_rsrc((void *)a.x, 0, a.x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t wrsrc =
      __builtin_amdgcn_make_buffer_rsrc((void *)a.w, 0, (uint32_t)(n_oc * OB * slices) * 1024u, 0x00020000);

  // the lane's pixel of every block: where its input begins (gather: byte offset, rows and columns for the borders; patch:
  // byte of LDS), and where its output goes
  uint32_t at[NB];
  int ih0[NB], iw0[NB];
  bool out_ok[FIN];
  uint32_t out_base = 0, img = 0;
  int oh0 = 0, ow0 = 0, rows = 0, cols = 0;
  const int pitch = (a.c16 | 1) * 16;          // of a position in LDS: an odd number of 16 bytes, for 16 positions on all banks
  const int th = a.shape & 255, tw = a.shape >> 8 & 255, ph = a.shape >> 16;
  const int pw = (tw - 1) * a.sw + (a.kw - 1) * a.dw + 1;
  if (PATCH) {
    img = div_by(pix_tile, a.magic_img);
    const uint32_t in_img = pix_tile - img * a.per_img, trow = div_by(in_img, a.magic_row);
    oh0 = (int)trow * th;
    ow0 = (int)(in_img - trow * a.per_row) * tw;
    rows = min(th, a.oh - oh0);
    cols = min(tw, a.ow - ow0);
    out_base = (img * a.oh + oh0) * a.ow + ow0;
  }
  auto row_of = [&](uint32_t slot) { return (slot + 1) * a.by_tw >> 16; };   // slots < 256, floor(2^16 - 1 / tw): exact
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const uint32_t slot = (uint32_t)(wg * NB + j) * 16 + px;
    if (PATCH) {
      const uint32_t r = row_of(slot), c = slot - r * tw;
      const bool ok = (int)r < rows && (int)c < cols;
      at[j] = (ok ? (r * a.sh * pw + c * a.sw) * pitch : 0) + (UNI ? chunk * 16 : 0);
    } else {
      const uint32_t pix = pix_tile * (PW * NB * 16) + slot;
      const uint32_t q = div_by(pix, a.magic_row), c = pix - q * a.ow, n = div_by(q, a.magic_img), r = q - n * a.oh;
      ih0[j] = (int)(r * a.sh) - a.pt;
      iw0[j] = (int)(c * a.sw) - a.pl;
      at[j] = (uint32_t)(((int)(n * a.ih) + ih0[j]) * a.iw + iw0[j]) * a.x_cs + (UNI ? chunk * 16 : 0);
      if (pix >= a.shape) ih0[j] = -(1 << 29);
    }
  }
  const uint32_t woff = (uint32_t)lane * 16u;
  const uint32_t wbase = (uint32_t)(oc_tile * OB * slices) * 1024u;
  constexpr int D = PATCH ? patch_depth(KW * PW, UNI) : kDepth;
  v4i af[D][OB], bf[PATCH ? 1 : D][NB];
  auto load_filter = [&](int slot, int s) {
#pragma unroll
    for (int o = 0; o < OB; ++o)
      af[slot][o] = (v4i)__builtin_amdgcn_raw_buffer_load_b128(wrsrc, s < slices ? woff : kOobOffset, (o * slices + s) * 1024 + wbase, 0);
  };
  auto load_input = [&](int slot, int s) {
    const bool in_k = s < slices;
    const uint32_t kg = (uint32_t)(4 * s + (UNI ? 0 : chunk));
    const uint32_t tap = div_by(kg, a.magic_c16), cgrp = kg - tap * a.c16, tkh = div_by(tap, a.magic_kw), tkw = tap - tkh * a.kw;
    const int dh_off = in_k ? (int)(tkh * a.dh) : 1 << 28, dw_off = (int)(tkw * a.dw);
    const int tap_off = ((int)(tkh * a.dh) * a.iw + dw_off) * (int)a.x_cs + (int)cgrp * 16;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int ih = ih0[j] + dh_off, iw = iw0[j] + dw_off;
      const bool ok = ((unsigned)ih < (unsigned)a.ih) & ((unsigned)iw < (unsigned)a.iw);
      bf[slot][j] = buffer_load16(xrsrc, ok ? at[j] + (uint32_t)tap_off : kOobOffset);
    }
  };

  // ---- operands on their way
  const int patch_chunks = PATCH ? ph * pw * a.c16 : 0;
  v4i pv[kPatchLoads];
  uint32_t pto[kPatchLoads];
  const int prow0 = oh0 * a.sh - a.pt, pcol0 = ow0 * a.sw - a.pl;
  auto fetch_patch = [&](int q0) {
#pragma unroll
    for (int u = 0; u < kPatchLoads; ++u) {
      if (q0 + u * T >= patch_chunks) break;
      const uint32_t q = (uint32_t)(q0 + u * T + tid);
      const uint32_t pos = div_by(q, a.magic_c16), c = q - pos * a.c16, r = div_by(pos, a.magic_pw), col = pos - r * pw;
      const int ih = prow0 + (int)r, iw = pcol0 + (int)col;
      const bool ok = (int)q < patch_chunks && (unsigned)ih < (unsigned)a.ih && (unsigned)iw < (unsigned)a.iw;
      pto[u] = pos * pitch + c * 16;
      pv[u] = buffer_load16(xrsrc, ok ? (uint32_t)(((int)(img * a.ih) + ih) * a.iw + iw) * a.x_cs + c * 16 : kOobOffset);
    }
  };
  auto park_patch = [&](int q0) {
#pragma unroll
    for (int u = 0; u < kPatchLoads; ++u)
      if (q0 + u * T + tid < patch_chunks) *reinterpret_cast<v4i *>(reinterpret_cast<char *>(lds) + pto[u]) = pv[u];
  };
  if (PATCH) fetch_patch(0);
#pragma unroll
  for (int d = 0; d < D; ++d) {
    if (!PATCH && wk + d * KW >= slices) break;
    load_filter(d, wk + d * KW);
    if (!PATCH) load_input(d, wk + d * KW);
  }

  // ---- what finishing takes besides the sums
  const bool second = POST && post->split_oc > 0 && oc0 >= post->split_oc;
  int8_t *const y = second ? post->y2 : a.y;
  const int y_cs = second ? post->y2_cs : a.y_cs, oc_shift = second ? post->split_oc : 0;
  const int lo = second ? post->lo2 : (a.slices_pad_relu & 3) == 1 ? 0 : -128;
  v4i bias[FIN], mult[FIN], shift[FIN], hpot[FIN];
  uint32_t src[FIN];
  int64_t off[FIN];
  const int nparam = param_entries(a.oc);
#pragma unroll
  for (int f = 0; f < FIN; ++f) {
    const int b = wk + f * KW, oc = oc0 + (b / NB) * 16 + chunk * 4;   // block b: channels b / NB, pixels b % NB
    const uint32_t slot = (uint32_t)(wg * NB + b % NB) * 16 + px;
    bool ok = b < B && oc < ((a.oc + 15) & ~15);
    uint32_t pix;
    if (PATCH) {
      const uint32_t r = row_of(slot), c = slot - r * tw;
      ok = ok && (int)r < rows && (int)c < cols;
      pix = out_base + r * a.ow + c;
    } else {
      pix = pix_tile * (PW * NB * 16) + slot;
      ok = ok && pix < a.shape;
    }
    out_ok[f] = ok;
    off[f] = (int64_t)pix * y_cs + (oc - oc_shift);
    src[f] = 0;
    if (b < B) {
      bias[f] = *reinterpret_cast<const v4i *>(a.bias + oc);
      mult[f] = *reinterpret_cast<const v4i *>(a.bias + nparam + oc);
      shift[f] = *reinterpret_cast<const v4i *>(a.bias + 2 * nparam + oc);
      hpot[f] = *reinterpret_cast<const v4i *>(a.bias + 3 * nparam + oc);
      if (POST && ok && post->add_dst) src[f] = *reinterpret_cast<const uint32_t *>(post->add_src + off[f]);
    }
  }
  v4i *const sums = lds + (PATCH ? ph * pw * (a.c16 | 1) : 0);
  uint8_t *const lut = reinterpret_cast<uint8_t *>(sums + KW * PW * B * 64);
  uint32_t lutv = 0;
  if (POST && post->has_lut && tid < 64) lutv = post->lut.w[tid];

  if (PATCH) {
    for (int q0 = 0;;) {
      park_patch(q0);
      q0 += kPatchLoads * T;
      if (q0 >= patch_chunks) break;
      fetch_patch(q0);
    }
    __syncthreads();
  }

  // ---- multiply
  v4i acc[OB][NB];
#pragma unroll
  for (int o = 0; o < OB; ++o)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[o][j] = v4i{0, 0, 0, 0};
  const int mine = (slices - wk + KW - 1) / KW;
  auto multiply = [&](int slot, int s) {
    v4i b[NB];
    if (PATCH) {
      // past the end the filter is zeros
      const uint32_t kg = UNI ? 4u * (uint32_t)min(s, slices - 1) : (uint32_t)min(4 * s + chunk, groups - 1);
      const uint32_t tap = div_by(kg, a.magic_c16), cgrp = kg - tap * a.c16, tkh = div_by(tap, a.magic_kw), tkw = tap - tkh * a.kw;
      const char *from = reinterpret_cast<const char *>(lds) + (tkh * a.dh * pw + tkw * a.dw) * pitch + cgrp * 16;
#pragma unroll
      for (int j = 0; j < NB; ++j) b[j] = *reinterpret_cast<const v4i *>(from + at[j]);
    } else {
#pragma unroll
      for (int j = 0; j < NB; ++j) b[j] = bf[slot][j];
    }
#pragma unroll
    for (int o = 0; o < OB; ++o)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[o][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[slot][o], b[j], acc[o][j], 0, 0, 0);
  };
  int i0 = 0;
#pragma nounroll
  for (; i0 + D < mine; i0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      multiply(d, wk + (i0 + d) * KW);
      load_filter(d, wk + (i0 + D + d) * KW);
      if (!PATCH) load_input(d, wk + (i0 + D + d) * KW);
    }
  }
#pragma unroll
  for (int d = 0; d < D; ++d) {
    if (!PATCH && i0 + d >= mine) break;
    multiply(d, wk + (i0 + d) * KW);   // patch form: slices past the end are zeros
  }

  // ---- the sums meet
  if (POST && post->has_lut && tid < 64) reinterpret_cast<uint32_t *>(lut)[tid] = lutv;
#pragma unroll
  for (int o = 0; o < OB; ++o)
#pragma unroll
    for (int j = 0; j < NB; ++j) sums[(wave * B + o * NB + j) * 64 + lane] = acc[o][j];
  __syncthreads();
#pragma unroll
  for (int f = 0; f < FIN; ++f) {
    const int b = wk + f * KW;
    if (b >= B) return;
    v4i t = bias[f];
#pragma unroll
    for (int k = 0; k < KW; ++k) t += sums[((wg * KW + k) * B + b) * 64 + lane];
    if (a.slices_pad_relu & 2) {
#pragma unroll
      for (int e = 0; e < 4; ++e) t[e] = max(t[e], 0);
    }
    uint32_t o = pack_sat4(requant_one<FAST>(t[0], mult[f][0], shift[f][0], hpot[f][0]),
                           requant_one<FAST>(t[1], mult[f][1], shift[f][1], hpot[f][1]),
                           requant_one<FAST>(t[2], mult[f][2], shift[f][2], hpot[f][2]),
                           requant_one<FAST>(t[3], mult[f][3], shift[f][3], hpot[f][3]), lo);
    if (!out_ok[f]) continue;
    if (!POST) {
      *reinterpret_cast<uint32_t *>(y + off[f]) = o;
      continue;
    }
    if (post->store_y) *reinterpret_cast<uint32_t *>(y + off[f]) = o;
    if (post->has_lut) {
      const uint32_t r = (uint32_t)lut[o & 255u] | ((uint32_t)lut[(o >> 8) & 255u] << 8) | ((uint32_t)lut[(o >> 16) & 255u] << 16) |
                         ((uint32_t)lut[o >> 24] << 24);
      const int valid = a.oc - (oc0 + (b / NB) * 16 + chunk * 4);   // channels of this dword that exist
      o = r & (valid >= 4 ? 0xffffffffu : valid <= 0 ? 0u : (1u << (8 * valid)) - 1u);
      if (post->lut_dst) *reinterpret_cast<uint32_t *>(post->lut_dst + off[f]) = o;
    }
    if (post->add_dst) {
      const v4i z = fused_add_chunk(v4i{(int)o, 0, 0, 0}, v4i{(int)src[f], 0, 0, 0}, post->add_m_src, post->add_m_conv, post->add_rshift,
                                    post->add_relu, post->add_pk);
      *reinterpret_cast<uint32_t *>(post->add_dst + off[f]) = (uint32_t)z[0];
    }
  }
}

template <int KW, int PW, int NB, int OB, bool FAST, bool UNI, bool PATCH>
__global__ __launch_bounds__(KW * PW * 64) void conv_split_kernel(SplitArgs a) {
  split_body<KW, PW, NB, OB, FAST, UNI, PATCH, false>(a, nullptr);
}
template <int KW, int PW, int NB, int OB, bool FAST, bool UNI, bool PATCH>
__global__ __launch_bounds__(KW * PW * 64) void conv_split_post_kernel(SplitPost p) {
  split_body<KW, PW, NB, OB, FAST, UNI, PATCH, true>(p.a, &p);
}

// FullyConnected of few rows (a classifier) the same way, from the filter in fragments of 32 channels that fc_prepack() makes: 16
// rows of a fragment are 256 contiguous bytes of it, channels 0-7 and 16-23 of the block of 32, or the others.  A workgroup of
// four or eight waves per 16 * OB channels x 16 * NB rows; K split over the waves, four slices of 64 bytes in flight each.
// Bound: launch, one trip to memory, one meeting in LDS; from 64 rows on the operands' way into a CU (98 KB each at 100 x 2048 x
// 1000).  Replayed from a graph, against sixteen waves per block of 32 x 32, two barriers and one wave that finished 16 channels a
// lane: 1 x 2048 x 1000 3.63 -> 2.35 us, 32 rows 4.92 -> 3.18, 100 rows 5.11 -> 4.25, 16 x 8192 x 4096 10.2 -> 6.9, 256 x 1024 x
// 4096 8.11 -> 7.1.
template <int KW, int NB, int OB, bool FAST>
__global__ __launch_bounds__(KW * 64) void fc_split_kernel(FcArgs a) {
  constexpr int B = NB * OB, D = kDepth;
  static_assert(B <= KW, "a wave finishes one block");
  __shared__ v4i sums[KW * B * 64];
  asm volatile("" ::"s"(a.x), "s"(a.w), "s"(a.bias), "s"(a.x_bytes), "s"(a.w_bytes), "s"(a.rows), "s"(a.oc), "s"(a.x_cs), "s"(a.slices),
               "s"(a.nparam));
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int oc_tile = blockIdx.x, row0 = blockIdx.y * (NB * 16);
  const int first = OB == 2 ? oc_tile * 32 : (oc_tile >> 1) * 32 + (oc_tile & 1) * 8;   // its first channel
  if (first >= ((a.oc + 15) & ~15)) return;    // uniform over the workgroup
  const int px = lane & 15, chunk = lane >> 4;
  const __amdgpu_buffer_rsrc_t xrsrc = __builtin_amdgcn_make_buffer_rsrc((void *)a.x, 0, a.x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t wrsrc = __builtin_amdgcn_make_buffer_rsrc((void *)a.w, 0, a.w_bytes, 0x00020000);
  const uint32_t wbase = (uint32_t)(first >> 5) * (uint32_t)a.slices * 2048u + (OB == 2 ? 0u : (uint32_t)(oc_tile & 1) * 256u);
  const uint32_t woff = (uint32_t)(chunk >> 1) * 1024u + (uint32_t)(px + 32 * (chunk & 1)) * 16u;
  uint32_t xoff[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int row = row0 + j * 16 + px;
    xoff[j] = row < a.rows ? (uint32_t)row * (uint32_t)a.x_cs + chunk * 16 : kOobOffset;
  }
  v4i af[D][OB], bf[D][NB];
  auto load = [&](int slot, int s) {
    const bool in_k = s < a.slices;
#pragma unroll
    for (int o = 0; o < OB; ++o)
      af[slot][o] = (v4i)__builtin_amdgcn_raw_buffer_load_b128(wrsrc, in_k ? woff : kOobOffset, wbase + s * 2048 + o * 256, 0);
#pragma unroll
    for (int j = 0; j < NB; ++j) bf[slot][j] = (v4i)__builtin_amdgcn_raw_buffer_load_b128(xrsrc, in_k ? xoff[j] : kOobOffset, s * 64, 0);
  };
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (wave + d * KW < a.slices) load(d, wave + d * KW);   // (256 x 1024 x 4096, two slices a wave: 9.0 us with loads of nothing)

  // block b: channels of half b / NB, rows of block b % NB
  const int oc = first + (wave / NB) * 8 + (chunk & 1) * 16 + (chunk >> 1) * 4, row = row0 + (wave % NB) * 16 + px;
  v4i bias = {0, 0, 0, 0}, mult = bias, shift = bias, hpot = bias;
  if (wave < B) {
    bias = *reinterpret_cast<const v4i *>(a.bias + oc);
    mult = *reinterpret_cast<const v4i *>(a.bias + a.nparam + oc);
    shift = *reinterpret_cast<const v4i *>(a.bias + 2 * a.nparam + oc);
    hpot = *reinterpret_cast<const v4i *>(a.bias + 3 * a.nparam + oc);
  }
  v4i acc[OB][NB];
#pragma unroll
  for (int o = 0; o < OB; ++o)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[o][j] = v4i{0, 0, 0, 0};
  auto multiply = [&](int slot) {
#pragma unroll
    for (int o = 0; o < OB; ++o)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[o][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(af[slot][o], bf[slot][j], acc[o][j], 0, 0, 0);
  };
  const int mine = (a.slices - wave + KW - 1) / KW;
  int last = 0;                                // first slice of the wave's last round
#pragma nounroll
  for (; last + D < mine; last += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      multiply(d);
      load(d, wave + (last + D + d) * KW);
    }
  }
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (d < mine - last) multiply(d);
#pragma unroll
  for (int o = 0; o < OB; ++o)
#pragma unroll
    for (int j = 0; j < NB; ++j) sums[(wave * B + o * NB + j) * 64 + lane] = acc[o][j];
  __syncthreads();
  if (wave >= B) return;
  v4i t = bias;
#pragma unroll
  for (int k = 0; k < KW; ++k) t += sums[(k * B + wave) * 64 + lane];
  if (a.relu_first) {
#pragma unroll
    for (int e = 0; e < 4; ++e) t[e] = max(t[e], 0);
  }
  const uint32_t o = pack_sat4(requant_one<FAST>(t[0], mult[0], shift[0], hpot[0]), requant_one<FAST>(t[1], mult[1], shift[1], hpot[1]),
                               requant_one<FAST>(t[2], mult[2], shift[2], hpot[2]), requant_one<FAST>(t[3], mult[3], shift[3], hpot[3]), a.lo);
  if (row < a.rows && oc < ((a.oc + 15) & ~15)) *reinterpret_cast<uint32_t *>(a.y + (int64_t)row * a.y_cs + oc) = o;
}

uint32_t magic_of(int64_t d) { return (uint32_t)(0xffffffffull / (uint64_t)d); }

template <int KW, int PW, int NB, int OB, bool FAST, bool UNI, bool PATCH>
void launch_form(tpuhip_ctx *ctx, unsigned lds, const SplitArgs &a, const SplitPost *post) {
  const dim3 grid((a.n_tiles + 7) / 8 * 8), block(KW * PW * 64);
  auto go = [&](auto kernel, const auto &args) {
    if (lds > 65536 && !raise_lds_limit(ctx->device, (const void *)kernel, kLdsBytes)) return;
    if (ctx->prof_start)
      hipExtLaunchKernelGGL(kernel, grid, block, lds, ctx->stream, ctx->prof_start, ctx->prof_stop, 0, args);
    else
      hipLaunchKernelGGL(kernel, grid, block, lds, ctx->stream, args);
  };
  if (post) {
    go(conv_split_post_kernel<KW, PW, NB, OB, FAST, UNI, PATCH>, *post);
  } else {
    go(conv_split_kernel<KW, PW, NB, OB, FAST, UNI, PATCH>, a);
  }
}

template <int KW, int PW, int NB, int OB>
void launch_variant(tpuhip_ctx *ctx, const SplitPlan &pl, bool fast, bool uni, const SplitArgs &a, const SplitPost *post) {
  if (pl.th) {
    uni ? launch_form<KW, PW, NB, OB, true, true, true>(ctx, pl.lds, a, post) : launch_form<KW, PW, NB, OB, true, false, true>(ctx, pl.lds, a, post);
    return;
  }
  if (fast) uni ? launch_form<KW, PW, NB, OB, true, true, false>(ctx, pl.lds, a, post) : launch_form<KW, PW, NB, OB, true, false, false>(ctx, pl.lds, a, post);
  else uni ? launch_form<KW, PW, NB, OB, false, true, false>(ctx, pl.lds, a, post) : launch_form<KW, PW, NB, OB, false, false, false>(ctx, pl.lds, a, post);
}

}  // namespace

// The patch form: a window of more than one tap, a patch that fits; as many whole rows as the slots hold, or the part of a row
// that they hold, evened out over the image.  It saves what the taps of a block's pixels share and costs a trip through LDS and a
// barrier, so the line lies by the K that is fetched and the pixels of a wave.  Straight from memory / as a patch, from a graph:
//   16 pixels and 32: 64 -> 512 on 2 x 6 x 40 at stride 2 (9 slices) 2.40 / 3.02 us, 192 -> 96 on 35 x 19 (27) 2.88 / 3.70, 256 ->
//     256 on 14 x 14 (36) 3.44 / 3.38, 512 -> 512 on 7 x 7 (72) 4.52 / 3.95, 512 -> 1024 on 13 x 13 (72) 7.72 / 4.85;
//   64 and 128: 64 -> 64 on 56 x 56 (9) 3.02 / 3.84, 128 -> 256 on 52 x 52 (18) 8.19 / 5.85, 256 -> 512 on 26 x 26 (36) 7.50 / 5.37.
SplitPlan tpuhip::split_plan(const tpuhip_conv_desc &d, const SplitVariant &v, bool fast) {
  SplitPlan pl;
  const int slots = v.pw * v.nb * 16;
  const unsigned rest = (unsigned)(v.kw * v.pw * v.nb * v.ob) * 1024u + 256u;
  pl.lds = rest;
  const int slices = (d.kh * d.kw * ((d.ic + 15) / 16) + 3) / 4;
  if (!fast || d.kh * d.kw == 1 || slices <= (v.nb <= 2 ? 32 : 16)) return pl;
  const int pitch = ((d.ic + 15) / 16 | 1) * 16;
  auto width = [&](int tw) { return (int64_t)(tw - 1) * d.sw + (int64_t)(d.kw - 1) * d.dw + 1; };
  auto height = [&](int th) { return (int64_t)(th - 1) * d.sh + (int64_t)(d.kh - 1) * d.dh + 1; };
  auto bytes = [&](int th, int tw) { return height(th) * width(tw) * pitch + rest; };
  int th = std::max(1, std::min(d.oh, slots / std::min(d.ow, slots))), tw = std::min(d.ow, slots);
  while (th > 1 && bytes(th, tw) > kLdsBytes) --th;
  while (tw > 1 && bytes(th, tw) > kLdsBytes) --tw;
  if (bytes(th, tw) > kLdsBytes) return pl;
  const int rows = (d.oh + th - 1) / th, cols = (d.ow + tw - 1) / tw;
  pl.th = (d.oh + rows - 1) / rows;
  pl.tw = (d.ow + cols - 1) / cols;
  pl.ph = (int)height(pl.th);
  pl.pw = (int)width(pl.tw);
  pl.lds = (unsigned)bytes(pl.th, pl.tw);
  return pl;
}

int64_t tpuhip::split_tiles(const tpuhip_conv_desc &d, const SplitVariant &v, const SplitPlan &pl) {
  const int64_t pix = pl.th ? (int64_t)d.n * ceil_div64(d.oh, pl.th) * ceil_div64(d.ow, pl.tw)
                            : ceil_div64((int64_t)d.n * d.oh * d.ow, v.pw * v.nb * 16);
  return pix * ceil_div64(d.oc, 16 * v.ob);
}

bool tpuhip::split_args(const tpuhip_conv_desc &d, const SplitVariant &v, const SplitPlan &pl, SplitArgs *out) {
  SplitArgs a{};
  const int c16 = (d.ic + 15) / 16, slices = (d.kh * d.kw * c16 + 3) / 4;
  const int64_t n_oc = ceil_div64(d.oc, 16 * v.ob), tiles = split_tiles(d, v, pl), n_pix = tiles / n_oc;
  const int64_t npix = (int64_t)d.n * d.oh * d.ow, in_bytes = (int64_t)d.n * d.ih * d.iw * d.x_cs;
  for (int64_t u16 : {d.ih, d.iw, d.oh, d.ow, d.y_cs, d.oc, d.sh, d.sw, d.pt, d.pl, d.dh, d.dw, d.kw, 16 * slices + 15})
    if (u16 < 0 || u16 > 65535) return false;
  // the divisions by multiplying are exact where number * divisor stays below 2^32
  if (in_bytes >= 1ll << 31 || n_oc * v.ob * slices * 1024 >= 1ll << 31) return false;
  if ((tiles + 8) * std::max(n_pix, n_oc) >= 1ll << 32 || (npix + 256) * std::max(d.oh, d.ow) >= 1ll << 32) return false;
  a.x_bytes = (uint32_t)in_bytes;
  a.n_tiles = (uint32_t)tiles;
  // where the filter is the larger operand an XCD reads its own part of it only
  a.n_pix = n_oc * 16 * v.ob * (int64_t)slices * 64 > in_bytes ? (uint32_t)n_pix : 0;
  a.magic_tile = magic_of(a.n_pix ? n_pix : n_oc);
  if (pl.th) {
    const int64_t per_row = ceil_div64(d.ow, pl.tw), per_img = per_row * ceil_div64(d.oh, pl.th);
    if (per_img > 65535 || pl.th > 255 || pl.tw > 255 || pl.ph > 65535) return false;
    a.shape = (uint32_t)pl.th | (uint32_t)pl.tw << 8 | (uint32_t)pl.ph << 16;
    a.per_img = (uint16_t)per_img;
    a.per_row = (uint16_t)per_row;
    a.magic_img = magic_of(per_img);
    a.magic_row = magic_of(per_row);
    a.magic_pw = magic_of(pl.pw);
    a.by_tw = (uint16_t)(65535 / pl.tw);
  } else {
    a.shape = (uint32_t)npix;
    a.magic_img = magic_of(d.oh);
    a.magic_row = magic_of(d.ow);
  }
  a.magic_c16 = magic_of(c16);
  a.magic_kw = magic_of(d.kw);
  a.ih = (uint16_t)d.ih; a.iw = (uint16_t)d.iw; a.oh = (uint16_t)d.oh; a.ow = (uint16_t)d.ow;
  a.x_cs = (uint32_t)d.x_cs; a.y_cs = (uint16_t)d.y_cs; a.oc = (uint16_t)d.oc; a.c16 = (uint16_t)c16;
  a.sh = (uint16_t)d.sh; a.sw = (uint16_t)d.sw; a.pt = (uint16_t)d.pt; a.pl = (uint16_t)d.pl;
  a.dh = (uint16_t)d.dh; a.dw = (uint16_t)d.dw; a.kw = (uint16_t)d.kw;
  a.slices_pad_relu = (uint16_t)(slices * 16 + (4 * slices - d.kh * d.kw * c16) * 4 + (!d.do_relu ? 0 : d.relu_first ? 2 : 1));
  *out = a;
  return true;
}

void tpuhip::split_launch(tpuhip_ctx *ctx, const SplitVariant &v, const SplitPlan &pl, bool fast, bool uni, const SplitArgs &a,
                          const SplitPost *post) {
#define TPUHIP_FORM(KW, PW, NB, OB) \
  if (v.kw == KW && v.pw == PW && v.nb == NB && v.ob == OB) return launch_variant<KW, PW, NB, OB>(ctx, pl, fast, uni, a, post);
  TPUHIP_SPLIT_VARIANTS(TPUHIP_FORM)
#undef TPUHIP_FORM
}

// The blocks of a workgroup: those with which the busiest CU fetches the least, a workgroup fetching as many rows of operands as it
// has channels and rows.  Of nine shapes timed with all four it names the fastest in seven (100 x 2048 x 1000: 4.33, 4.21, 4.36,
// 6.29 us in the order below; 32 rows: 3.15, 4.05, 4.26, 4.93), 4 % from it in the others.  Beyond 256 rows, which only a K of more
// than 4096 brings, blocks of 32 channels alone: their rows are HBM's (4000 x 5000 x 16: 7.9 us with two workgroups of eight channels
// for every block of rows, 6.6).
// Waves: four where they hold all of K at once, up to four slices each; 4 x 2 blocks, which are more than four waves finish, become
// 2 x 2.  Eight: 256 x 64 x 4096 4.1 us, four 3.0; 256 x 1024 x 4096 7.9 and 7.1, 100 x 512 x 4096 3.6 and 3.5.
void tpuhip::fc_split(tpuhip_ctx *ctx, const FcArgs &a, bool fast) {
  const int kinds[][2] = {{1, 1}, {2, 1}, {2, 2}, {4, 2}};
  int best = 0;
  int64_t least = INT64_MAX;
  for (int k = a.rows > 256 ? 2 : 0; k < 4; ++k) {
    const int nb = kinds[k][0], ob = kinds[k][1];
    const int64_t tiles = ceil_div64(a.oc, 16 * ob) * ceil_div64(a.rows, 16 * nb);
    const int64_t cost = ceil_div64(tiles, ctx->num_cu) * (std::min(a.rows, 16 * nb) + 16 * ob);
    if (cost < least) {
      least = cost;
      best = k;
    }
  }
  const bool four = a.slices <= 4 * kDepth;
  if (four) best = std::min(best, 2);
  const int nb = kinds[best][0], ob = kinds[best][1];
  // Channel tiles in whole rounds of the XCDs, where that is an eighth more at most: those of one tile of channels meet its filter in
  // one L2 (2048 x 9216 x 4096: 316 us, 350 with an equal share of all tiles for each XCD).  Few tiles of channels would leave all
  // rows to as few XCDs (4000 x 5000 x 16 on one of the eight: 24 us).
  const int64_t across = (ob == 2 ? 1 : 2) * ceil_div64(a.oc, 32), rounds = ceil_div64(across, 8) * 8;
  const dim3 grid((unsigned)(rounds * 8 <= across * 9 ? rounds : across), (unsigned)ceil_div64(a.rows, 16 * nb)), block(four ? 256 : 512);
  auto go = [&](auto kernel) {
    if (ctx->prof_start || ctx->prof_stop)
      hipExtLaunchKernelGGL(kernel, grid, block, 0, ctx->stream, ctx->prof_start, ctx->prof_stop, 0, a);
    else
      hipLaunchKernelGGL(kernel, grid, block, 0, ctx->stream, a);
  };
#define TPUHIP_FC(KW, NB, OB) return fast ? go(fc_split_kernel<KW, NB, OB, true>) : go(fc_split_kernel<KW, NB, OB, false>)
  switch (four ? best + 4 : best) {
    case 0: TPUHIP_FC(8, 1, 1);
    case 1: TPUHIP_FC(8, 2, 1);
    case 2: TPUHIP_FC(8, 2, 2);
    case 3: TPUHIP_FC(8, 4, 2);
    case 4: TPUHIP_FC(4, 1, 1);
    case 5: TPUHIP_FC(4, 2, 1);
    default: TPUHIP_FC(4, 2, 2);
  }
#undef TPUHIP_FC
}
