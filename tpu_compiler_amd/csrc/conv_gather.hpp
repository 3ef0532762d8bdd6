// Grouped convs and convs over an input with inserted zeros (transposed convs) on the matrix cores: the plan that
// conv.hip keeps with a packed conv, and its launch.
#pragma once

#include "common.hpp"

namespace tpuhip {

struct GatherPlan;

// Whether the gather kernel takes the layer (see the rule in conv_gather.hip), and its packed form on the device;
// *out stays NULL where it does not.  filter: OIHW int8 on the host (G x OC/G x IC/G x KH x KW).
int gather_prepack(tpuhip_ctx *ctx, const tpuhip_conv_desc &d, const int8_t *filter, GatherPlan **out);
// how a layer that is neither dense nor depthwise runs: tpuhip_conv2d_gather_form
int gather_form(const tpuhip_conv_desc &d, int num_cu, int *reach);
void gather_destroy(tpuhip_ctx *ctx, GatherPlan *plan);
// bias, and the planes of multiplier, rshift and 2^(rshift-1) of nparam entries each, indexed by output channel and padded
// beyond a multiple of 64 channels; fast: the layer's requantisation cannot overflow
int gather_run(tpuhip_ctx *ctx, const GatherPlan *plan, const void *x, void *y, const int32_t *bias, const int32_t *planes,
               int nparam, bool fast);

}  // namespace tpuhip
