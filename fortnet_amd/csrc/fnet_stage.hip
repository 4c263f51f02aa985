// Host I/O of a context through a ring of pinned memory.
//
// A call that changes a batch has a dozen small arrays to bring in, and a copy command for each
// costs 5-10 us (more from pageable memory) and, with its source on the host stack, a wait.  The
// arrays are written into the ring instead and one kernel copies all of them to their places, on
// the context's own stream, so nothing is waited for.  Results of small calls come back the same
// way: one kernel gathers them in the ring, one wait, plain memory copies from there.  Large arrays
// (kStageMax) keep their copy commands, whose bandwidth is better (1 MB up: 44 us against 50).
//
// The ring belongs to one context (one host thread, one stream): space is reused only after the
// stream has drained, which a context that waits for its results does anyway.
#include <cstring>

#include "fnet_internal.hpp"

namespace fnet {
namespace {

// Each block moves up to kSegBlock bytes of one segment, in 16-byte words where both ends are
// aligned to them, else in 4-byte ones (every array holds 4- or 8-byte values).
constexpr unsigned kSegBlock = 16384;

__global__ void __launch_bounds__(256) k_copy_segments(StageSegs a) {
  int k = 0;
  while (k + 1 < a.n && blockIdx.x >= a.first[k + 1]) ++k;
  const size_t at = (size_t)(blockIdx.x - a.first[k]) * kSegBlock;
  const size_t len = min((size_t)kSegBlock, a.bytes[k] - at);
  const char* src = (const char*)a.src[k] + at;
  char* dst = (char*)a.dst[k] + at;
  size_t done = 0;
  if ((((size_t)src | (size_t)dst) & 15) == 0) {
    for (size_t q = threadIdx.x; q < len / 16; q += 256) ((uint4*)dst)[q] = ((const uint4*)src)[q];
    done = len / 16 * 16;
  }
  for (size_t q = done / 4 + threadIdx.x; q < len / 4; q += 256)
    ((unsigned*)dst)[q] = ((const unsigned*)src)[q];
}

hipError_t launch_segments(StageSegs& segs, hipStream_t s) {
  if (segs.n == 0) return hipSuccess;
  unsigned blocks = 0;
  for (int k = 0; k < segs.n; ++k) {
    segs.first[k] = blocks;
    blocks += (unsigned)((segs.bytes[k] + kSegBlock - 1) / kSegBlock);
  }
  k_copy_segments<<<blocks, 256, 0, s>>>(segs);
  segs.n = 0;
  return hipGetLastError();
}

}  // namespace

hipError_t stage_flush(fnet_ctx* ctx) {
  FNET_HIP_TRY(launch_segments(ctx->segs, ctx->stream));
  if (ctx->stage_direct) {
    // a copy command read (or may still read) memory of the caller
    ctx->stage_direct = false;
    return hipStreamSynchronize(ctx->stream);
  }
  return hipSuccess;
}

// `bytes` of the ring, or null (too large, or no pinned memory)
static char* stage_take(fnet_ctx* ctx, size_t bytes) {
  if (bytes > kStageMax) return nullptr;
  if (!ctx->ring) {
    if (hipHostMalloc((void**)&ctx->ring, kStageRing, hipHostMallocDefault) != hipSuccess) {
      ctx->ring = nullptr;
      (void)hipGetLastError();
      return nullptr;
    }
    ctx->ring_at = 0;
  }
  const size_t need = (bytes + 63) & ~size_t(63);
  if (ctx->ring_at + need > kStageRing) {
    if (launch_segments(ctx->segs, ctx->stream) != hipSuccess ||
        hipStreamSynchronize(ctx->stream) != hipSuccess)
      return nullptr;
    ctx->ring_at = 0;
  }
  char* p = ctx->ring + ctx->ring_at;
  ctx->ring_at += need;
  return p;
}

static hipError_t stage_add(fnet_ctx* ctx, void* dst, const void* src, size_t bytes) {
  StageSegs& g = ctx->segs;
  if (g.n == kStageSegs) FNET_HIP_TRY(launch_segments(g, ctx->stream));
  g.dst[g.n] = dst;
  g.src[g.n] = src;
  g.bytes[g.n] = bytes;
  ++g.n;
  return hipSuccess;
}

hipError_t stage_in(fnet_ctx* ctx, void* dst, const void* src, size_t bytes) {
  if (bytes == 0) return hipSuccess;
  if (char* p = stage_take(ctx, bytes)) {
    std::memcpy(p, src, bytes);
    return stage_add(ctx, dst, p, bytes);
  }
  ctx->stage_direct = true;
  return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->stream);
}

hipError_t stage_out(fnet_ctx* ctx, const StageOut* out, int n) {
  size_t total = 0;
  for (int k = 0; k < n; ++k)
    if (out[k].host) total += (out[k].bytes + 63) & ~size_t(63);
  char* p = total <= kStageMax / 2 ? stage_take(ctx, total) : nullptr;
  if (!p) {
    for (int k = 0; k < n; ++k)
      if (out[k].host && out[k].bytes)
        FNET_HIP_TRY(hipMemcpyAsync(out[k].host, out[k].dev, out[k].bytes, hipMemcpyDeviceToHost,
                                    ctx->stream));
    return hipStreamSynchronize(ctx->stream);
  }
  char* q = p;
  for (int k = 0; k < n; ++k)
    if (out[k].host && out[k].bytes) {
      FNET_HIP_TRY(stage_add(ctx, q, out[k].dev, out[k].bytes));
      q += (out[k].bytes + 63) & ~size_t(63);
    }
  FNET_HIP_TRY(launch_segments(ctx->segs, ctx->stream));
  FNET_HIP_TRY(hipStreamSynchronize(ctx->stream));
  q = p;
  for (int k = 0; k < n; ++k)
    if (out[k].host && out[k].bytes) {
      std::memcpy(out[k].host, q, out[k].bytes);
      q += (out[k].bytes + 63) & ~size_t(63);
    }
  return hipSuccess;
}

}  // namespace fnet
