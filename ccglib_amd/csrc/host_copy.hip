// Copies of page-locked host memory into device memory by the compute units: up to
// three buffers in one launch.
#include "common.h"

namespace ccglib_amd {
namespace {

typedef unsigned uint4_t __attribute__((ext_vector_type(4)));
typedef uint4_t uint4_any_t __attribute__((aligned(1)));

constexpr unsigned kLoads = 4;                       // 16-byte loads in flight a thread
constexpr unsigned kBlockBytes = 256 * 16 * kLoads;  // what a block copies

// Bound by the link: 256 threads with four loads each are 16 KiB under way, and a few such blocks
// cover its latency. Blocks below first[1] copy buffer 0, below first[2] buffer 1, the others
// buffer 2. The destinations are 16-byte aligned; a source may lie anywhere.
__global__ __launch_bounds__(256) void copy_from_host(const HostCopies c) {
  const unsigned n = blockIdx.x < c.first[1] ? 0u : blockIdx.x < c.first[2] ? 1u : 2u;
  const char *src = static_cast<const char *>(c.src[n]);
  char *dst = static_cast<char *>(c.dst[n]);
  const size_t bytes = c.bytes[n], base = (size_t)(blockIdx.x - c.first[n]) * kBlockBytes + threadIdx.x * 16;
  uint4_t v[kLoads];
#pragma unroll
  for (unsigned i = 0; i < kLoads; ++i) {
    const size_t at = base + i * 256 * 16;
    if (at + 16 <= bytes) v[i] = *reinterpret_cast<const uint4_any_t *>(src + at);
  }
#pragma unroll
  for (unsigned i = 0; i < kLoads; ++i) {
    const size_t at = base + i * 256 * 16;
    if (at + 16 <= bytes) {
      *reinterpret_cast<uint4_t *>(dst + at) = v[i];
    } else if (at < bytes) {
      for (size_t b = at; b < bytes; ++b) dst[b] = src[b];
    }
  }
}

}  // namespace

hipError_t launch_copy_from_host(HostCopies c, hipStream_t stream) {
  size_t blocks = 0;
  for (int i = 0; i < 3; ++i) {
    c.first[i] = (unsigned)blocks;
    blocks += ceil_div(c.bytes[i], (size_t)kBlockBytes);
  }
  if (blocks == 0) return hipSuccess;
  if (blocks > 0x7fffffffu) return hipErrorInvalidValue;
  hipLaunchKernelGGL(copy_from_host, dim3((unsigned)blocks), dim3(256), 0, stream, c);
  return hipGetLastError();
}

}  // namespace ccglib_amd
