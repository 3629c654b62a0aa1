// Calibration statistics that feed add_batch (G2PTQ / GuidedQuant).
//
// SaliencyCache.grad_hook (gptq_utils/g2ptq_utils.py:604-618): for the
// gradient of a linear's output (n tokens × hidden), the mean over each of G
// equal channel groups of grad², one (n, G) fp32 saliency per batch.
//   group_mean_square_kernel: one wave per (token, group); lanes stride the
//   group's columns (coalesced), a butterfly sums the squares, and the mean is
//   sum · fp32(1/gs), the product torch's mean reduction forms on the GPU.
//
// GradientCache.cache_gradient (:704-714): the per-token running mean of the
// weight gradient, cache ← cache·(k/(k+1)) + grad/(n·(k+1)).
//   running_mean_kernel: one elementwise HBM pass, in the reference's fp32
//   operation order; the division by the Python number n·(k+1) is, in torch
//   on the GPU, a multiplication by its fp32 reciprocal, and so it is here.
#include <algorithm>
#include <type_traits>

#include "common.hpp"

// Every product and sum is rounded on its own, as torch evaluates these
// expressions: no fused multiply-adds.  The __f*_rn helpers are plain
// operators in the HIP headers, so this translation unit is built with
// -ffp-contract=off (the pragma covers this file's own code).
#pragma clang fp contract(off)

namespace g2ptq {
namespace {

__device__ __forceinline__ float load_any(const void* p, int64_t i, int dtype) {
  if (dtype == 0) return __uint_as_float((uint32_t) static_cast<const uint16_t*>(p)[i] << 16);
  if (dtype == 1) return (float)static_cast<const _Float16*>(p)[i];
  return static_cast<const float*>(p)[i];
}

__global__ __launch_bounds__(256) void group_mean_square_kernel(const void* __restrict__ x,
                                                                int dtype, int64_t rows,
                                                                int64_t ldx, int64_t groups,
                                                                int64_t gs, float inv_gs,
                                                                float* __restrict__ out) {
  const int64_t pair = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (pair >= rows * groups) return;  // whole waves: no barrier below
  const int64_t t = pair / groups, g = pair - t * groups;
  const int64_t base = t * ldx + g * gs;
  float acc = 0.f;
  for (int64_t c = lane; c < gs; c += 64) {
    const float v = load_any(x, base + c, dtype);
    acc = __fadd_rn(acc, __fmul_rn(v, v));  // grad.float().pow(2), then the sum
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
  if (lane == 0) out[pair] = __fmul_rn(acc, inv_gs);
}

// Eight 16-bit (or 4 + 4 fp32) consecutive values from a 16-byte boundary.
template <typename T>
__device__ __forceinline__ void load8(const T* p, float (&v)[8]) {
  if constexpr (sizeof(T) == 2) {
    const uint4 u = *reinterpret_cast<const uint4*>(p);
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if constexpr (std::is_same_v<T, uint16_t>) {  // bf16
        v[2 * k] = __uint_as_float(w[k] << 16);
        v[2 * k + 1] = __uint_as_float(w[k] & 0xffff0000u);
      } else {
        v[2 * k] = (float)__builtin_bit_cast(_Float16, (unsigned short)(w[k] & 0xffffu));
        v[2 * k + 1] = (float)__builtin_bit_cast(_Float16, (unsigned short)(w[k] >> 16));
      }
    }
  } else {
    const float4 a = reinterpret_cast<const float4*>(p)[0], b = reinterpret_cast<const float4*>(p)[1];
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  }
}

// group_mean_square_kernel on 16-byte loads (rows and groups of a multiple of
// 8 values, 16-byte aligned): the 2-byte loads of the kernel above leave HBM
// at 1.7 TB/s.  One wave per (token, group), eight values per lane and step,
// four steps in flight, each of the eight positions summed apart and the
// eight sums added in a fixed order before the butterfly.  8192 × 4096 bf16 in
// 4 groups, MI355X: 40.0 -> 14.7 us (4.6 TB/s).
template <typename T>
__global__ __launch_bounds__(256) void group_mean_square_vec_kernel(const T* __restrict__ x,
                                                                    int64_t rows, int64_t ldx,
                                                                    int64_t groups, int64_t gs,
                                                                    float inv_gs,
                                                                    float* __restrict__ out) {
  const int64_t pair = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (pair >= rows * groups) return;  // whole waves: no barrier below
  const int64_t t = pair / groups, g = pair - t * groups;
  const T* row = x + t * ldx + g * gs;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int64_t c = (int64_t)lane * 8; c < gs; c += 512) {
    float v[8];
    load8(row + c, v);
#pragma unroll
    for (int k = 0; k < 8; ++k) acc[k] = __fadd_rn(acc[k], __fmul_rn(v[k], v[k]));
  }
  float s = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  if (lane == 0) out[pair] = __fmul_rn(s, inv_gs);
}

// running_mean_kernel on 16-byte loads and stores (4096 × 4096 bf16 gradients,
// two updates, MI355X: 30.9 -> 22.7 us each), the same operations per
// element.
template <typename T>
__global__ __launch_bounds__(256) void running_mean_vec_kernel(float4* __restrict__ cache,
                                                               const T* __restrict__ grad,
                                                               int64_t n8, float keep,
                                                               float inv_count, int first) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n8;
       i += (int64_t)gridDim.x * blockDim.x) {
    float v[8];
    load8(grad + 8 * i, v);
    float4 c[2] = {make_float4(0.f, 0.f, 0.f, 0.f), make_float4(0.f, 0.f, 0.f, 0.f)};
    if (!first) {
      c[0] = cache[2 * i];
      c[1] = cache[2 * i + 1];
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float* e = reinterpret_cast<float*>(&c[h]);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float d = __fmul_rn(v[4 * h + k], inv_count);
        e[k] = __fadd_rn(first ? 0.f : __fmul_rn(e[k], keep), d);
      }
      cache[2 * i + h] = c[h];
    }
  }
}

__global__ __launch_bounds__(256) void running_mean_kernel(float* __restrict__ cache,
                                                           const void* __restrict__ grad,
                                                           int dtype, int64_t n, float keep,
                                                           float inv_count, int first) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const float d = __fmul_rn(load_any(grad, i, dtype), inv_count);
    // first call: the cache is the Python int 0, so cache·keep + d is 0.0 + d
    const float c = first ? 0.f : __fmul_rn(cache[i], keep);
    cache[i] = __fadd_rn(c, d);
  }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

}  // namespace
}  // namespace g2ptq

using namespace g2ptq;

extern "C" int g2ptq_group_mean_square(void* stream, const void* x, int dtype, int64_t rows,
                                       int64_t cols, int64_t ldx, int64_t groups, float* out) {
  G2PTQ_CHECK(dtype >= 0 && dtype <= 2, "group_mean_square: dtype code %d", dtype);
  G2PTQ_CHECK(rows >= 0 && cols >= 0 && groups >= 1, "group_mean_square: bad sizes");
  G2PTQ_CHECK(cols % groups == 0, "group_mean_square: %lld columns do not split into %lld groups",
              (long long)cols, (long long)groups);
  if (rows == 0 || cols == 0) return G2PTQ_OK;
  G2PTQ_CHECK(x && out && ldx >= cols, "group_mean_square: bad operands");
  const int64_t gs = cols / groups;
  const int64_t waves = rows * groups;
  G2PTQ_CHECK(cdiv(waves, (int64_t)4) < (1ll << 31), "group_mean_square: too many rows");
  const dim3 grid((unsigned)cdiv(waves, (int64_t)4));
  hipStream_t st = as_stream(stream);
  const float inv_gs = 1.0f / (float)gs;
  // 16-byte loads where every group starts on a 16-byte boundary and holds
  // whole steps of eight values, from groups of 128 on: narrower ones leave
  // most of a wave's lanes without a step (8192 rows of 4096 bf16, one value
  // per lane and load against eight: groups of 32 148 and 181 µs, of 64 78 and
  // 93, of 128 51 and 48, of 256 38 and 25).
  if (gs >= 128 && gs % 8 == 0 && ldx % 8 == 0 && aligned16(x)) {
    if (dtype == 0)
      hipLaunchKernelGGL(group_mean_square_vec_kernel<uint16_t>, grid, dim3(256), 0, st,
                         static_cast<const uint16_t*>(x), rows, ldx, groups, gs, inv_gs, out);
    else if (dtype == 1)
      hipLaunchKernelGGL(group_mean_square_vec_kernel<_Float16>, grid, dim3(256), 0, st,
                         static_cast<const _Float16*>(x), rows, ldx, groups, gs, inv_gs, out);
    else
      hipLaunchKernelGGL(group_mean_square_vec_kernel<float>, grid, dim3(256), 0, st,
                         static_cast<const float*>(x), rows, ldx, groups, gs, inv_gs, out);
  } else {
    hipLaunchKernelGGL(group_mean_square_kernel, grid, dim3(256), 0, st, x, dtype, rows, ldx,
                       groups, gs, inv_gs, out);
  }
  G2PTQ_LAUNCHED();
  return G2PTQ_OK;
}

extern "C" int g2ptq_running_mean_update(void* stream, float* cache, const void* grad, int dtype,
                                         int64_t n, float keep, float inv_count, int first) {
  G2PTQ_CHECK(dtype >= 0 && dtype <= 2, "running_mean_update: dtype code %d", dtype);
  G2PTQ_CHECK(n >= 0, "running_mean_update: negative size");
  if (n == 0) return G2PTQ_OK;
  G2PTQ_CHECK(cache && grad, "running_mean_update: null pointer");
  hipStream_t st = as_stream(stream);
  if (n % 8 == 0 && aligned16(cache) && aligned16(grad)) {
    const unsigned vb = (unsigned)std::max<int64_t>(1, std::min<int64_t>(cdiv(n / 8, 256), 8192));
    float4* c4 = reinterpret_cast<float4*>(cache);
    if (dtype == 0)
      hipLaunchKernelGGL(running_mean_vec_kernel<uint16_t>, dim3(vb), dim3(256), 0, st, c4,
                         static_cast<const uint16_t*>(grad), n / 8, keep, inv_count, first);
    else if (dtype == 1)
      hipLaunchKernelGGL(running_mean_vec_kernel<_Float16>, dim3(vb), dim3(256), 0, st, c4,
                         static_cast<const _Float16*>(grad), n / 8, keep, inv_count, first);
    else
      hipLaunchKernelGGL(running_mean_vec_kernel<float>, dim3(vb), dim3(256), 0, st, c4,
                         static_cast<const float*>(grad), n / 8, keep, inv_count, first);
    G2PTQ_LAUNCHED();
    return G2PTQ_OK;
  }
  const unsigned blocks = (unsigned)std::max<int64_t>(1, std::min<int64_t>(cdiv(n, 256), 8192));
  hipLaunchKernelGGL(running_mean_kernel, dim3(blocks), dim3(256), 0, st, cache,
                     grad, dtype, n, keep, inv_count, first);
  G2PTQ_LAUNCHED();
  return G2PTQ_OK;
}
