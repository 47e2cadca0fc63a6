// Copies between the runtime's page-locked arena and GPU memory by kernels on the
// calling thread's stream, for host tensors of up to a few MiB.
//
// Bound: PCIe, about 50 GB/s, and what surrounds it.  A copy engine's transfer is
// waited for across queues and costs 10 to 20 us however small it is; a kernel in
// the same stream costs a launch.  A result is sent in chunks, each followed by a
// word in host memory that says so, so that the calling thread copies chunk by
// chunk into the caller's array while the next ones arrive, and knows without
// asking the runtime when the last one has (a stream synchronisation costs 20 to
// 30 us).  Fused layer on host arrays, from Python: 128 x 768 x 3072 150 -> 91 us,
// 42 x 256 x 1024 72 -> 37, 149 x 512 x 320 71 -> 45, 7 x 256 x 256 36 -> 26.
#include "om_kernels.h"

namespace om {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(256) void k_copy_in(
    const v4i *__restrict__ src, v4i *__restrict__ dst, unsigned vectors) {
  const unsigned i = blockIdx.x * 256 + threadIdx.x;
  if (i < vectors)
    dst[i] = src[i];
}

// Blocks take the chunks in turn, few at a time, so that early chunks are
// complete early.  Stores at system scope (they do not stay in a cache of the
// GPU); the word is stored when the chunk's have been acknowledged.
__global__ __launch_bounds__(256) void k_copy_out(CopyOut a) {
  for (unsigned c = blockIdx.x; c < a.chunks; c += gridDim.x) {
    int s = 0;
#pragma unroll
    for (int i = 1; i < CopyOut::kTensors; ++i)
      if (i < a.tensors && c >= a.t[i].first_chunk)
        s = i;
    const char *src = a.t[0].src;
    char *dst = a.t[0].dst;
    unsigned bytes = a.t[0].bytes, first = 0;
#pragma unroll
    for (int i = 1; i < CopyOut::kTensors; ++i)
      if (i == s) {
        src = a.t[i].src;
        dst = a.t[i].dst;
        bytes = a.t[i].bytes;
        first = a.t[i].first_chunk;
      }
    const unsigned off = (c - first) * CopyOut::kChunk;
    const unsigned n =
        bytes - off < CopyOut::kChunk ? bytes - off : CopyOut::kChunk;
    // (both buffers hold whole vectors: their sizes are rounded up)
    const v4i *const sv = (const v4i *)(src + off);
    const __amdgpu_buffer_rsrc_t rsrc =
        __builtin_amdgcn_make_buffer_rsrc(dst + off, 0, CopyOut::kChunk, 0x00020000);
    constexpr int V = CopyOut::kChunk / 16 / 256;
    v4i v[V];
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const unsigned i = j * 256 + threadIdx.x;
      v[j] = i * 16 < n ? sv[i] : (v4i){0, 0, 0, 0};
    }
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const unsigned i = j * 256 + threadIdx.x;
      if (i * 16 < n)
        __builtin_amdgcn_raw_buffer_store_b128(v[j], rsrc, (int)(i * 16), 0, 17);
    }
    if (c == 0 && threadIdx.x < 2 && a.failed)
      __hip_atomic_store(&a.status[threadIdx.x], a.failed[threadIdx.x],
          __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0x0F70); // vmcnt(0): acknowledged
    __builtin_amdgcn_s_barrier();
    if (threadIdx.x == 0)
      __hip_atomic_store(&a.arrived[c], a.epoch, __ATOMIC_RELAXED,
          __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

} // namespace

hipError_t launch_copy_in(hipStream_t s, const void *src, void *dst, size_t bytes) {
  if (bytes > ((size_t)1 << 30) || ((((uintptr_t)src) | ((uintptr_t)dst)) & 15))
    return hipErrorInvalidValue;
  const unsigned vectors = (unsigned)((bytes + 15) / 16);
  if (vectors)
    k_copy_in<<<(vectors + 255) / 256, 256, 0, s>>>(
        (const v4i *)src, (v4i *)dst, vectors);
  return hipGetLastError();
}

hipError_t launch_copy_out(hipStream_t s, const CopyOut &a) {
  if (a.tensors < 1 || a.tensors > CopyOut::kTensors || a.chunks < 1)
    return hipErrorInvalidValue;
  k_copy_out<<<a.chunks < 24 ? a.chunks : 24u, 256, 0, s>>>(a);
  return hipGetLastError();
}

} // namespace om
