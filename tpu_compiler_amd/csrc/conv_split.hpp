// Convs of few outputs: K split over the waves of a workgroup, blocks of 16 x 16 outputs (conv_split.hip).
#pragma once

#include "common.hpp"

namespace tpuhip {

// The arguments of a launch with nothing fused behind it: two cache lines for the kernel to wait for, and as many as a launch
// takes without costing the host more (112 bytes).
struct SplitArgs {
  const int8_t *x, *w;
  int8_t *y;
  const int32_t *bias;         // the planes of multiplier, right shift and 2^(right shift - 1) lie behind the biases
  uint32_t x_bytes;
  uint32_t n_tiles, n_pix;     // tiles; pixel tiles, or 0: the channel tiles of a pixel tile follow each other
  uint32_t shape;              // patch form: rows, columns << 8 of a tile, rows << 16 of its patch; gather form: the pixels there are
  // floor((2^32 - 1) / d) of what a number is divided by: x / d == umulhi(x + 1, magic)
  uint32_t magic_tile;         // n_pix, or the channel tiles
  uint32_t magic_img, magic_row;   // patch form: pixel tiles of an image, of a row of them; gather form: output rows, columns
  uint32_t magic_c16, magic_kw, magic_pw;   // pw: columns of the patch
  uint32_t x_cs;               // any that a layer may be given after its variant is chosen: 32 bits
  uint16_t per_img, per_row;   // patch form: what magic_img and magic_row divide by
  uint16_t by_tw;              // patch form: floor((2^16 - 1) / columns of a tile)
  uint16_t ih, iw, oh, ow, y_cs, oc, c16;
  uint16_t sh, sw, pt, pl, dh, dw, kw;
  uint16_t slices_pad_relu;    // slices of 64 bytes of K << 4 | groups of 16 bytes past its end << 2 | 1: ReLU behind the
                               // requantisation, 2: in front of it
};
static_assert(sizeof(SplitArgs) <= 112, "see above");

// and what is fused behind it
struct SplitPost {
  SplitArgs a;
  const int8_t *add_src;
  int8_t *add_dst, *lut_dst, *y2;
  int32_t add_m_src, add_m_conv, add_rshift, add_relu, add_pk, store_y, split_oc, y2_cs, lo2, has_lut;
  Table256 lut;
};

// a variant: waves along K and along the pixels, blocks of 16 pixels and of 16 channels per wave
struct SplitVariant {
  int kw, pw, nb, ob;
};
#define TPUHIP_SPLIT_VARIANTS(F) \
  F(4, 1, 1, 1) F(8, 1, 1, 1) F(8, 1, 2, 1) F(8, 1, 4, 1) F(8, 1, 2, 2) F(8, 1, 4, 2) F(4, 2, 4, 2)
// Rows x columns of outputs whose input lies in LDS as one patch of ph rows (th == 0: the operands come straight from memory).
struct SplitPlan {
  int th = 0, tw = 0, ph = 0, pw = 0;
  unsigned lds = 0;
};
SplitPlan split_plan(const tpuhip_conv_desc &d, const SplitVariant &v, bool fast);
int64_t split_tiles(const tpuhip_conv_desc &d, const SplitVariant &v, const SplitPlan &pl);
// What a launch of the layer takes but its pointers and what is fused behind it; false: a number is beyond the arguments' fields.
bool split_args(const tpuhip_conv_desc &d, const SplitVariant &v, const SplitPlan &pl, SplitArgs *out);
// post: NULL, nothing is fused
void split_launch(tpuhip_ctx *ctx, const SplitVariant &v, const SplitPlan &pl, bool fast, bool uni, const SplitArgs &a,
                  const SplitPost *post);

// FullyConnected from the filter as fragments of 32 channels x 32 bytes of K (the packing of mfma_reg_32x32)
struct FcArgs {
  const int8_t *x, *w;
  int8_t *y;
  const int32_t *bias;     // the planes as in SplitArgs
  int nparam;
  uint32_t x_bytes, w_bytes;
  int rows, oc, x_cs, y_cs, slices;   // slices of 64 bytes of K
  int relu_first, lo;
};
void fc_split(tpuhip_ctx *ctx, const FcArgs &a, bool fast);

}  // namespace tpuhip
