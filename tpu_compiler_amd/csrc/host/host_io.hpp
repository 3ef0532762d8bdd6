// Tensors between a caller's host memory and the device: pageable buffers on one side, channels-last int8 on the
// other, a pinned staging buffer of the context in between.
//
// Only int8 crosses the bus, whatever type the caller holds, and no DMA is involved: the layout kernels read and write
// the pinned buffer themselves (a kernel moves it at the bus rate, 57 GB/s, and a copy engine in front of a kernel
// costs another 8 us).  The host pass (float <-> int8 with its check, or a plain copy) runs in pieces on a few threads,
// and the pieces overlap with the transfer of those before them.
#pragma once

#include <cstddef>
#include <cstdint>
#include <functional>

#include "common.hpp"

namespace tpuhip {

// n floats (at any alignment) -> int8; the return value tells whether one of them is no integer in [-128, 127] (is_unsigned: [0, 255],
// stored as the byte).  past_caches: with stores that leave the caches alone
bool floats_to_bytes(const void *src, int8_t *dst, size_t n, bool is_unsigned, bool past_caches = false);
// n int8 (is_unsigned: uint8) -> floats; past_caches: with stores that leave the caches alone
void bytes_to_floats(const int8_t *src, float *dst, size_t n, bool is_unsigned, bool past_caches = false);

// piece(0) .. piece(n - 1), on this thread and a few others; returns when all are done.  Pieces throw nothing.
void parallel_pieces(size_t n, const std::function<void(size_t)> &piece);

// What the host side holds: float-stored integers (converted and checked), int8 bytes, or floats that stay floats.
enum class HostKind { kFloatStored, kBytes, kFloats };

struct HostTensor {
  int n, c, h, w, cs;   // channels-last int8 on the device; for kFloats the device side is dense NCHW floats
  bool is_unsigned;
};

// host -> device, issued to the context's stream; the caller's buffer may be reused on return.  *bad: an element of a
// float-stored tensor is no integer of the byte range (nothing has been written to dst then).
int host_to_device(tpuhip_ctx *ctx, const HostTensor &t, HostKind kind, const void *src, void *dst, bool *bad);
// device -> host, several tensors in one go; waits for the work in front of it
struct HostRead {
  HostTensor t;
  HostKind kind;
  const void *src;
  void *dst;
};
int device_to_host(tpuhip_ctx *ctx, const HostRead *reads, size_t n);

// A result that is complete while its stream still has work in front of it: read_ahead() lays it out for the host there
// and then, finish_ahead() fetches it beside the rest of that work, settle_ahead() waits for that rest.
struct AheadRead {
  void *dense = nullptr, *pinned = nullptr;
  uint32_t *flag = nullptr, serial = 0;   // the flag, in pinned memory, shows the serial of what lies in `dense`
  size_t bytes = 0;
  bool refused = false;                   // there is no memory for it
  bool fetched = false;                   // `pinned` holds it, or a copy to there is in flight (not beyond settle_ahead())
  ~AheadRead();
};
int read_ahead(tpuhip_ctx *ctx, AheadRead &a, const HostTensor &t, const void *src, bool *done);   // !*done: there is no memory for it
// the host pass from a's bytes instead of r.src
int finish_ahead(tpuhip_ctx *ctx, AheadRead &a, const HostRead &r);
// waits for everything the context has issued; what else has been laid out early is fetched meanwhile
int settle_ahead(tpuhip_ctx *ctx);
// nobody will ask for it any more
void drop_ahead(tpuhip_ctx *ctx, AheadRead &a);

}  // namespace tpuhip
