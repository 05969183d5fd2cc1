// Chunk permutation of the sequence axis for context parallelism (reference
// kvax/utils/permutation.py:9-116): a copy, bound by memory.  The order is a formula, so no index
// array is uploaded (an upload from pageable memory also makes the host wait for the stream).
// Measured, 16 chunks: 134 MB of keys 39 us = 6.9 TB/s read + written (an indexed library copy 107 us,
// its adjoint 230 us); 537 MB of queries 191 us = 5.6 TB/s.
#include "common.h"

namespace kvax {
namespace {

// The chunk of the source that chunk j of the result comes from; n even.
__device__ __forceinline__ int source_chunk(int j, int n, bool reverse) {
  if (!reverse) return j % 2 ? n - 1 - j / 2 : j / 2;
  return j < n / 2 ? 2 * j : 2 * (n - 1 - j) + 1;
}

// grid: (pieces of a chunk, chunks, batch); T is the widest element the chunk size and pointers allow
template <class T>
__global__ __launch_bounds__(256) void permute_chunks_kernel(const T* src, T* dst, int64_t per_chunk, int reverse) {
  const int n = gridDim.y, j = blockIdx.y;
  const T* from = src + ((int64_t)blockIdx.z * n + source_chunk(j, n, reverse)) * per_chunk;
  T* to = dst + ((int64_t)blockIdx.z * n + j) * per_chunk;
  // four independent elements per thread and round, so that enough loads are in flight
  const int64_t step = (int64_t)gridDim.x * 256;
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  for (; i + 3 * step < per_chunk; i += 4 * step) {
    const T a = from[i], b = from[i + step], c = from[i + 2 * step], d = from[i + 3 * step];
    to[i] = a, to[i + step] = b, to[i + 2 * step] = c, to[i + 3 * step] = d;
  }
  for (; i < per_chunk; i += step) to[i] = from[i];
}

template <class T>
int launch(const void* src, void* dst, int64_t batch, int n, int64_t chunk_bytes, int reverse, hipStream_t stream) {
  const int64_t per_chunk = chunk_bytes / (int64_t)sizeof(T);
  // about 16 work-groups per compute unit over the launch, each with at least one full round
  int64_t pieces = (per_chunk + 1023) / 1024;
  const int64_t want = (4096 + n * batch - 1) / (n * batch);
  pieces = pieces < want ? pieces : want;
  hipLaunchKernelGGL(permute_chunks_kernel<T>, dim3((unsigned)pieces, n, (unsigned)batch), dim3(256), 0, stream,
                     (const T*)src, (T*)dst, per_chunk, reverse);
  return check_launch("permute_chunks_kernel");
}

}  // namespace
}  // namespace kvax

using namespace kvax;

extern "C" int kvax_permute_chunks(const void* src, void* dst, int64_t batch, int num_chunks, int64_t chunk_bytes,
                                   int reverse, kvax_stream_t stream) {
  if (batch < 0 || batch > 65535 || num_chunks < 2 || num_chunks > 65534 || num_chunks % 2 || chunk_bytes < 0)
    return fail(KVAX_EINVAL, "cannot permute %lld x %d chunks of %lld bytes", (long long)batch, num_chunks,
                (long long)chunk_bytes);
  if (batch == 0 || chunk_bytes == 0) return KVAX_OK;
  if (!src || !dst) return fail(KVAX_EINVAL, "null tensor pointer");
  const uintptr_t all = (uintptr_t)src | (uintptr_t)dst | (uintptr_t)chunk_bytes;
  if (all % 4) return fail(KVAX_EINVAL, "chunks and pointers must be multiples of 4 bytes");
  return all % 16 ? launch<uint32_t>(src, dst, batch, num_chunks, chunk_bytes, reverse, (hipStream_t)stream)
                  : launch<uint4>(src, dst, batch, num_chunks, chunk_bytes, reverse, (hipStream_t)stream);
}
