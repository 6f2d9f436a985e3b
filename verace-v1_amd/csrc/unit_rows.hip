// L2 normalisation of rows, forward and backward (F.normalize over the last dimension, as the SSSD
// sub-layer applies it to q, k and v in training, sssd_attention.py:116-119).
//
//   y = x / max(|x|, eps);   dx = (g - y (y . g)) / |x| for |x| >= eps, g / eps below.
//
// Bound by memory: one read of the inputs, one write of the result.  As torch ops the forward is a
// reduction, a clamp and a mixed-type division, the backward some ten kernels over [rows, D] in fp32:
// 170 us for each of q, k, v at [65536, 128] bf16 -> fp32 under autocast, 28 us here (12 + 17).
// A row of up to 1024 elements is held by G lanes, four elements each per step; rows of any length and
// alignment take element loads.
#include "vmi_common.h"
#include "vmi_dispatch.h"

namespace vmi {
namespace unit {

constexpr int NTH = 256;
constexpr int MAXV = 4;  // steps of 4 elements a lane holds at most

template <typename T>
__device__ __forceinline__ void load4(const T* row, int d0, int D, bool vec, float (&x)[4]) {
  if (vec) {
    struct alignas(4 * sizeof(T)) V4 { T e[4]; };
    const V4 v = *reinterpret_cast<const V4*>(row + d0);
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = io<T>::to_f32(v.e[j]);
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = d0 + j < D ? io<T>::load(row, d0 + j) : 0.f;
  }
}
template <typename T>
__device__ __forceinline__ void store4(T* row, int d0, int D, bool vec, const float (&x)[4]) {
  if (vec) {
    struct alignas(4 * sizeof(T)) V4 { T e[4]; };
    V4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) io<T>::store(v.e, j, x[j]);
    *reinterpret_cast<V4*>(row + d0) = v;
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (d0 + j < D) io<T>::store(row, d0 + j, x[j]);
  }
}
// over the G lanes (a power of two) that share a row
__device__ __forceinline__ float row_sum(float x, int G) {
  for (int off = G >> 1; off >= 1; off >>= 1) x += __shfl_xor(x, off);
  return x;
}

// BACKWARD: x the forward's input, g the gradient of its output, y receives dx.
template <typename X, typename Y, bool BACKWARD>
__global__ __launch_bounds__(NTH) void unit_rows_kernel(const X* __restrict__ x, const Y* __restrict__ g,
                                                        X* __restrict__ dx, Y* __restrict__ y,
                                                        int64_t rows, int D, int G, float eps, bool vec) {
  const int64_t r = (static_cast<int64_t>(blockIdx.x) * NTH + threadIdx.x) / G;
  const int lane = threadIdx.x % G;
  const bool on = r < rows;  // rows past the end take part in the shuffles with row 0's data
  const int64_t o = (on ? r : 0) * D;
  float xv[MAXV][4], gv[MAXV][4];
  float ss = 0.f, sg = 0.f;
#pragma unroll
  for (int v = 0; v < MAXV; ++v) {
    const int d0 = 4 * (lane + G * v);
    if (d0 >= D) break;
    load4(x + o, d0, D, vec, xv[v]);
    if constexpr (BACKWARD) load4(g + o, d0, D, vec, gv[v]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      ss = fmaf(xv[v][j], xv[v][j], ss);
      if constexpr (BACKWARD) sg = fmaf(xv[v][j], gv[v][j], sg);
    }
  }
  const float n = sqrtf(row_sum(ss, G));
  const float inv = 1.f / fmaxf(n, eps);  // NaN kept below: fmaxf(NaN, eps) is eps
  const float scale = n != n ? n : inv;
  if constexpr (BACKWARD) sg = row_sum(sg, G);
  if (!on) return;
  const float along = BACKWARD && n >= eps ? sg * inv * inv : 0.f;  // (y . g) / |x|
#pragma unroll
  for (int v = 0; v < MAXV; ++v) {
    const int d0 = 4 * (lane + G * v);
    if (d0 >= D) break;
    float t[4];
#pragma unroll
    for (int j = 0; j < 4; ++j)
      t[j] = BACKWARD ? (gv[v][j] - xv[v][j] * along) * scale : xv[v][j] * scale;
    if constexpr (BACKWARD) store4(dx + o, d0, D, vec, t);
    else store4(y + o, d0, D, vec, t);
  }
}

template <typename X, typename Y>
hipError_t launch(const void* x, const void* g, void* out, int64_t rows, int D, float eps, bool backward,
                  hipStream_t stream) {
  int G = 1;
  while (G < 64 && 4 * G < D) G *= 2;
  const uintptr_t bits = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(g) | reinterpret_cast<uintptr_t>(out);
  const bool vec = D % 4 == 0 && bits % 16 == 0;
  const int64_t per = NTH / G, blocks = (rows + per - 1) / per;
  if (backward)
    hipLaunchKernelGGL((unit_rows_kernel<X, Y, true>), dim3(static_cast<unsigned>(blocks)), dim3(NTH), 0,
                       stream, static_cast<const X*>(x), static_cast<const Y*>(g), static_cast<X*>(out),
                       nullptr, rows, D, G, eps, vec);
  else
    hipLaunchKernelGGL((unit_rows_kernel<X, Y, false>), dim3(static_cast<unsigned>(blocks)), dim3(NTH), 0,
                       stream, static_cast<const X*>(x), nullptr, nullptr, static_cast<Y*>(out), rows, D,
                       G, eps, vec);
  return hipGetLastError();
}

int run(const void* x, int x_dtype, const void* g, int y_dtype, void* out, int64_t rows, int64_t D,
        float eps, bool backward, void* stream) {
  if (rows < 0 || D < 1 || !(eps > 0.f)) return VMI_ERR_INVALID_ARG;
  if (rows > 0 && (x == nullptr || out == nullptr || (backward && g == nullptr))) return VMI_ERR_INVALID_ARG;
  if (D > 4 * 64 * MAXV || rows > INT32_MAX) return VMI_ERR_UNSUPPORTED;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int d = static_cast<int>(D);
  hipError_t e;
  if (rows == 0) return VMI_OK;
  if (x_dtype == VMI_F32 && y_dtype == VMI_F32) e = launch<float, float>(x, g, out, rows, d, eps, backward, s);
  else if (x_dtype == VMI_BF16 && y_dtype == VMI_F32) e = launch<bf16_t, float>(x, g, out, rows, d, eps, backward, s);
  else if (x_dtype == VMI_F16 && y_dtype == VMI_F32) e = launch<f16_t, float>(x, g, out, rows, d, eps, backward, s);
  else if (x_dtype == VMI_BF16 && y_dtype == VMI_BF16) e = launch<bf16_t, bf16_t>(x, g, out, rows, d, eps, backward, s);
  else return VMI_ERR_UNSUPPORTED;
  return hip_status(e);
}

}  // namespace unit
}  // namespace vmi

extern "C" int vmi_unit_rows(const void* x, int x_dtype, void* y, int y_dtype, int64_t rows, int64_t D,
                             float eps, void* stream) {
  return vmi::unit::run(x, x_dtype, nullptr, y_dtype, y, rows, D, eps, false, stream);
}

extern "C" int vmi_unit_rows_bwd(const void* x, int x_dtype, const void* dy, int y_dtype, void* dx,
                                 int64_t rows, int64_t D, float eps, void* stream) {
  return vmi::unit::run(x, x_dtype, dy, y_dtype, dx, rows, D, eps, true, stream);
}
