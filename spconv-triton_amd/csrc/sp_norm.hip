// Eval-mode BatchNorm over feature rows, with or without a ReLU after it, in one
// pass: y = fma(weight * (x - mean), rsqrt(var + eps), bias) in fp32, rounded to
// the rows' type, then max(y, 0) (a NaN stays).  The steps and their order are
// those that torch's modules show (compared bit for bit in every type): weight *
// rsqrt taken first, as one scale a channel, flips last bits of 16-bit rows,
// which the layers after it carry on.
//
// Bound by memory: the rows are read and written once.  A thread holds one
// 16-byte piece of the channels for kNormRows rows, all loaded at once, the
// pieces of a row on neighbouring threads.  torch runs the same as up to five
// launches (two conversions of 16-bit statistics, the inverse deviations, the
// transform, the ReLU's own pass): 31 us a layer on the LiDAR encoder (67k to
// 196k rows of 16 to 128 fp16 channels), 9.6 us here (8 rows a thread: 10.8).
#include "sp_common.h"

namespace sp {

constexpr int kNormThreads = 256;
constexpr int kNormRows = 4;  // rows per thread

template <typename P>
__device__ __forceinline__ float norm_param(const void* p, int c, float none) {
  return p ? float(static_cast<const P*>(p)[c]) : none;
}

template <typename T>
__device__ __forceinline__ T norm_one(float x, float mean, float weight, float inv, float bias,
                                      bool relu) {
  float r = __builtin_fmaf(weight * (x - mean), inv, bias);
  // rounded to fp32 first: without this, the fp16 instances take the fused
  // multiply-add that rounds once, to fp16 (about 1 value in 16 000 differs)
  asm("" : "+v"(r));
  const T y = T(r);
  return relu && y < T(0) ? T(0) : y;
}

// V channels (16 bytes) a thread, `pieces` = C / V <= 256.  The workgroup works
// out the channels' parameters once, in LDS, while its rows are on their way:
// with each thread's own (a square root and a division for each of its 8
// channels) the launch took 13.2 us a layer on the LiDAR encoder.
template <typename T, typename P, int V>
__global__ __launch_bounds__(kNormThreads) void batchnorm_rows(
    const T* __restrict__ x, int64_t rows, int C, int pieces, const void* __restrict__ mean,
    const void* __restrict__ var, const void* __restrict__ weight, const void* __restrict__ bias,
    float eps, int relu, T* __restrict__ out) {
  using vec = __attribute__((ext_vector_type(V))) T;
  extern __shared__ float s_par[];  // mean, weight, 1 / deviation, bias: C each
  const int per = kNormThreads / pieces;  // rows side by side
  const int r0 = int(threadIdx.x) / pieces, c0 = (int(threadIdx.x) - r0 * pieces) * V;
  const int64_t base = int64_t(blockIdx.x) * (per * kNormRows) + r0;
  const bool idle = r0 >= per;
  vec v[kNormRows];
#pragma unroll
  for (int j = 0; j < kNormRows; ++j) {
    const int64_t r = base + int64_t(j) * per;
    if (!idle && r < rows) v[j] = *reinterpret_cast<const vec*>(x + r * C + c0);
  }
  for (int c = int(threadIdx.x); c < C; c += kNormThreads) {
    s_par[c] = norm_param<P>(mean, c, 0.f);
    s_par[C + c] = norm_param<P>(weight, c, 1.f);
    s_par[2 * C + c] = rsqrtf(norm_param<P>(var, c, 1.f) + eps);
    s_par[3 * C + c] = norm_param<P>(bias, c, 0.f);
  }
  __syncthreads();
  if (idle) return;
  float m[V], w[V], inv[V], b[V];
#pragma unroll
  for (int i = 0; i < V; ++i) {
    m[i] = s_par[c0 + i];
    w[i] = s_par[C + c0 + i];
    inv[i] = s_par[2 * C + c0 + i];
    b[i] = s_par[3 * C + c0 + i];
  }
#pragma unroll
  for (int j = 0; j < kNormRows; ++j) {
    const int64_t r = base + int64_t(j) * per;
    if (r >= rows) continue;
    vec y;
#pragma unroll
    for (int i = 0; i < V; ++i)
      y[i] = norm_one<T>(float(v[j][i]), m[i], w[i], inv[i], b[i], relu != 0);
    *reinterpret_cast<vec*>(out + r * C + c0) = y;
  }
}

// Any width: a thread per value.
template <typename T, typename P>
__global__ __launch_bounds__(kNormThreads) void batchnorm_values(
    const T* __restrict__ x, int64_t n, int C, const void* __restrict__ mean,
    const void* __restrict__ var, const void* __restrict__ weight, const void* __restrict__ bias,
    float eps, int relu, T* __restrict__ out) {
  const int64_t step = int64_t(gridDim.x) * kNormThreads;
  for (int64_t i = int64_t(blockIdx.x) * kNormThreads + threadIdx.x; i < n; i += step) {
    const int c = int(i % C);
    out[i] = norm_one<T>(float(x[i]), norm_param<P>(mean, c, 0.f), norm_param<P>(weight, c, 1.f),
                         rsqrtf(norm_param<P>(var, c, 1.f) + eps), norm_param<P>(bias, c, 0.f),
                         relu != 0);
  }
}

template <typename T, typename P>
static int run_batchnorm(const void* x, int64_t rows, int C, const void* mean, const void* var,
                         const void* weight, const void* bias, float eps, int relu, void* out,
                         hipStream_t s) {
  constexpr int V = 16 / int(sizeof(T));
  const T* xt = static_cast<const T*>(x);
  T* ot = static_cast<T*>(out);
  const bool aligned =
      ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out)) & 15) == 0;
  if (C % V == 0 && C / V <= kNormThreads && aligned) {
    const int pieces = C / V;
    const int64_t blocks = cdiv(rows, int64_t(kNormThreads / pieces) * kNormRows);
    SP_CHECK_ARG(blocks <= kMaxGridX, "batchnorm: too many rows");
    batchnorm_rows<T, P, V><<<unsigned(blocks), kNormThreads, 4 * C * sizeof(float), s>>>(
        xt, rows, C, pieces, mean, var, weight, bias, eps, relu, ot);
  } else {
    const int64_t blocks = cdiv(rows * C, kNormThreads);
    batchnorm_values<T, P><<<unsigned(blocks < 65536 ? blocks : 65536), kNormThreads, 0, s>>>(
        xt, rows * C, C, mean, var, weight, bias, eps, relu, ot);
  }
  SP_LAUNCHED();
  return SP_OK;
}

}  // namespace sp

using namespace sp;

extern "C" int sp_batchnorm_eval(const void* x, int32_t dtype, int64_t rows, int64_t C,
                                 const void* mean, const void* var, const void* weight,
                                 const void* bias, int32_t param_dtype, float eps, int32_t relu,
                                 void* out, void* stream) {
  SP_CHECK_ARG(rows >= 0 && C >= 1 && C < 65536, "batchnorm: bad sizes rows=%lld C=%lld",
               (long long)rows, (long long)C);
  SP_CHECK_ARG(dtype == SP_F16 || dtype == SP_BF16 || dtype == SP_F32,
               "batchnorm: dtype %d not supported (f16/bf16/f32)", dtype);
  SP_CHECK_ARG(param_dtype == dtype || param_dtype == SP_F32,
               "batchnorm: parameters must be of the rows' type or fp32");
  if (rows == 0) return SP_OK;
  SP_CHECK_ARG(x && mean && var && out, "batchnorm: null pointer");
  hipStream_t s = as_stream(stream);
  const bool f32 = param_dtype == SP_F32;
  switch (dtype) {
    case SP_F16:
      return f32 ? run_batchnorm<_Float16, float>(x, rows, int(C), mean, var, weight, bias, eps,
                                                  relu, out, s)
                 : run_batchnorm<_Float16, _Float16>(x, rows, int(C), mean, var, weight, bias,
                                                     eps, relu, out, s);
    case SP_BF16:
      return f32 ? run_batchnorm<__bf16, float>(x, rows, int(C), mean, var, weight, bias, eps,
                                                relu, out, s)
                 : run_batchnorm<__bf16, __bf16>(x, rows, int(C), mean, var, weight, bias, eps,
                                                 relu, out, s);
    default:
      return run_batchnorm<float, float>(x, rows, int(C), mean, var, weight, bias, eps, relu, out,
                                         s);
  }
}
