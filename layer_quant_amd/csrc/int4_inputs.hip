// Small inputs of the attention calls: the largest cache position of a step, read by the host, and
// the additive bias of a 2-D keep-mask. Both are bound by their launch: they replace chains of torch
// kernels (a reduction and a copy; five elementwise kernels).
#include "lq_common.h"

namespace lq {

constexpr int MAX_THREADS = 1024;
constexpr int MAX_LOADS = 8;  // loads of a thread that are in flight together

// The largest of m and what load(0 .. n - 1) brings in (one or two positions each), MAX_LOADS per thread
// at a time; past the end the last one again, so that every batch is one round trip.
template <typename T, typename Load>
__device__ __forceinline__ int64_t thread_max(int64_t m, int64_t n, Load load) {
  for (int64_t i0 = threadIdx.x; i0 - threadIdx.x < n; i0 += (int64_t)MAX_LOADS * blockDim.x) {
    T v[MAX_LOADS];
#pragma unroll
    for (int u = 0; u < MAX_LOADS; ++u) v[u] = load(min(i0 + (int64_t)u * blockDim.x, n - 1));
#pragma unroll
    for (int u = 0; u < MAX_LOADS; ++u) {
      if constexpr (sizeof(T) == 16) {
        m = max(m, max((int64_t)v[u].x, (int64_t)v[u].y));
      } else {
        m = max(m, (int64_t)v[u]);
      }
    }
  }
  return m;
}

// One workgroup: each thread's loads (16 bytes where the positions are dense and aligned) go out eight
// at a time, then a shuffle reduction per wave and one over the waves. The result is stored with system
// scope to pinned host memory, so no copy follows. 16384 positions: 3.3 us, 65536 6.0, one 2.4 (8-byte
// loads under an unrolled loop, whose remainder went one at a time, 4.4 and 9.6 us; torch's reduction
// 7.2 us for 16384, then a copy). The call that packs 16384 tokens, which waits for it: 34.4 -> 22.8
// us, most of it from not waiting for the pack.
__global__ __launch_bounds__(MAX_THREADS) void max_position_kernel(const int64_t* pos,
                                                                   int64_t stride, int64_t n,
                                                                   int64_t* host_slot) {
  __shared__ int64_t part[MAX_THREADS / 64];
  const int tid = threadIdx.x;
  int64_t m = pos[(n - 1) * stride];  // the last of an odd count has no pair
  if (stride == 1 && ((uintptr_t)pos & 15) == 0) {
    m = thread_max<longlong2>(m, n >> 1, [&](int64_t i) { return ((const longlong2*)pos)[i]; });
  } else {
    m = thread_max<int64_t>(m, n, [&](int64_t i) { return pos[i * stride]; });
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = max(m, (int64_t)__shfl_xor((long long)m, o, 64));
  if ((tid & 63) == 0) part[tid >> 6] = m;
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) m = max(m, part[w]);
    __hip_atomic_store(host_slot, m, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

__device__ __forceinline__ bool nonzero(const void* base, int dtype, int64_t i) {
  switch (dtype) {
    case LQ_U8:
    case LQ_I8:
      return ((const uint8_t*)base)[i] != 0;
    case LQ_F16:
    case LQ_BF16:
      return (((const uint16_t*)base)[i] & 0x7fffu) != 0;
    case LQ_F32:
      return (((const uint32_t*)base)[i] & 0x7fffffffu) != 0;
    case LQ_I32:
      return ((const int32_t*)base)[i] != 0;
    default:
      return ((const int64_t*)base)[i] != 0;
  }
}

// One thread per key; rows in grid-stride over grid.y. Batch 8, 4001 keys of int64: 2.5 us, where
// the compare, fill, not, copy and masked fill of the torch expression took 14 us and their five
// launches (masked decode attention, batch 8, ctx 4001: 39.5 -> 21.7 us per call).
__global__ __launch_bounds__(256) void keep_mask_bias_kernel(View keep, View bias, int64_t B,
                                                             int64_t S) {
  const int64_t n = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (n >= S) return;
  for (int64_t b = blockIdx.y; b < B; b += gridDim.y) {
    const bool k = nonzero(keep.data, keep.dtype, b * keep.s[0] + n * keep.s[1]);
    ((float*)bias.data)[b * bias.s[0] + n * bias.s[3]] = k ? 0.0f : -INFINITY;
  }
}

}  // namespace lq

using namespace lq;

extern "C" int lq_max_position(const lq_tensor* positions, void* host_slot, void* stream) {
  int rc;
  if ((rc = check_tensor(positions, "positions", 1, false, LQ_I64)) != LQ_OK) return rc;
  if (host_slot == nullptr || ((uintptr_t)host_slot & 7) != 0) {
    return fail(LQ_ERR_INVALID_ARG, "host_slot must be an 8-byte aligned pinned host address");
  }
  const int64_t n = positions->shape[0];
  if (n < 1) return fail(LQ_ERR_INVALID_ARG, "positions is empty");
  const int threads = n <= 64 ? 64 : (n <= 4096 ? 256 : MAX_THREADS);
  hipLaunchKernelGGL(max_position_kernel, dim3(1), dim3(threads), 0, (hipStream_t)stream,
                     (const int64_t*)positions->data, positions->stride[0], n, (int64_t*)host_slot);
  return check_launch("lq_max_position");
}

extern "C" int lq_keep_mask_bias(const lq_tensor* keep, const lq_tensor* bias, void* stream) {
  int rc;
  if ((rc = check_tensor(keep, "keep", 2, false)) != LQ_OK) return rc;
  if ((rc = check_tensor(bias, "bias", 4, false, LQ_F32)) != LQ_OK) return rc;
  const int64_t B = keep->shape[0], S = keep->shape[1];
  if (bias->shape[0] != B || bias->shape[1] != 1 || bias->shape[2] != 1 || bias->shape[3] != S) {
    return fail(LQ_ERR_INVALID_ARG, "bias must be [%lld, 1, 1, %lld]", (long long)B, (long long)S);
  }
  if (B == 0 || S == 0) return LQ_OK;
  const int64_t blocks = (S + 255) / 256;
  if (blocks >= ((int64_t)1 << 24)) {
    return fail(LQ_ERR_UNSUPPORTED, "mask of %lld keys exceeds the launch limits", (long long)S);
  }
  const dim3 grid((unsigned)blocks, (unsigned)(B < 65535 ? B : 65535));
  hipLaunchKernelGGL(keep_mask_bias_kernel, grid, dim3(256), 0, (hipStream_t)stream,
                     make_view(keep), make_view(bias), B, S);
  return check_launch("lq_keep_mask_bias");
}
