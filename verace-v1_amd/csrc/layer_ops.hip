// The element-wise steps between a layer's matrix products, fused: the M-CMoE activation and
// routing, the residual adds with the RMSNorms either side of them, and the halting update of the
// adaptive-depth loop.  As torch ops a layer runs some 75 such kernels per token batch; each moves
// little and costs a launch (4.1 us inside a replayed graph on MI355X), and at prefill sizes every
// one is a pass over [tokens, 2 hidden].
//
// All of them read each input once and write each output once (bound by launches at decode sizes
// and by memory at prefill sizes).  Sums are fp32; where the torch ops round an intermediate tensor
// that is itself an output or a residual stream (the sums h + x), so do these; other intermediates
// stay fp32.
#include <initializer_list>

#include "vmi_common.h"
#include "vmi_dispatch.h"

namespace vmi {
namespace layer {

// 16 bytes of T
template <typename T> struct Vec {
  static constexpr int N = 16 / sizeof(T);
  T e[N];
};
template <typename T> __device__ __forceinline__ Vec<T> ldv(const T* p) {
  return __builtin_bit_cast(Vec<T>, *reinterpret_cast<const uint4*>(p));
}
template <typename T> __device__ __forceinline__ void stv(T* p, const Vec<T>& v) {
  *reinterpret_cast<uint4*>(p) = __builtin_bit_cast(uint4, v);
}
template <typename T> __device__ __forceinline__ T round_to(float x) {
  T r;
  io<T>::store(&r, 0, x);
  return r;
}
template <typename T> __device__ __forceinline__ float rounded(float x) {
  return io<T>::to_f32(round_to<T>(x));
}

// tanh and sigmoid: the library's for an fp32 result; for a 16-bit one on v_exp_f32 and v_rcp_f32 (a
// few 2^-24 relative), tanh as 1 - 2 / (e^2x + 1) and below 0.1, where that cancels, the series to
// x^5 (next term 17/315 x^6 <= 6e-8 relative): 1e-6 relative at most, against 2^-11 of the result's
// rounding.  (tanhf, expf and three full divisions an element: the activation at [8192, 2048] bf16
// takes 34 us, so 24.)
template <typename T> __device__ __forceinline__ float sigmoid_for(float x) {
  if constexpr (sizeof(T) == 4) return 1.f / (1.f + expf(-x));
  return __builtin_amdgcn_rcpf(1.f + __expf(-x));
}
template <typename T> __device__ __forceinline__ float tanh_for(float x) {
  if constexpr (sizeof(T) == 4) return tanhf(x);
  const float x2 = x * x;
  const float small = x * (1.f + x2 * (-1.f / 3.f + x2 * (2.f / 15.f)));
  const float big = 1.f - 2.f * __builtin_amdgcn_rcpf(__expf(2.f * x) + 1.f);
  return fabsf(x) < 0.1f ? small : big;
}

// ------------------------------------------------------------------ SiTU-GLU
// out = [b1 tanh(g / b1) sigmoid(g)] [b2 tanh(u / b2)] (activations.py:8-31)
template <typename T>
__global__ __launch_bounds__(256) void situ_glu_kernel(const T* __restrict__ g, const T* __restrict__ u,
                                                       T* __restrict__ out, float b1, float b2,
                                                       int64_t nvec) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= nvec) return;
  constexpr int N = Vec<T>::N;
  const Vec<T> a = ldv(g + i * N), b = ldv(u + i * N);
  const float r1 = 1.f / b1, r2 = 1.f / b2;
  Vec<T> y;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const float x = io<T>::to_f32(a.e[j]), z = io<T>::to_f32(b.e[j]);
    float t1, t2;  // fp32: divided, as the tensor ops do
    if constexpr (sizeof(T) == 4) t1 = x / b1, t2 = z / b2;
    else t1 = x * r1, t2 = z * r2;
    y.e[j] = round_to<T>((b1 * tanh_for<T>(t1) * sigmoid_for<T>(x)) * (b2 * tanh_for<T>(t2)));
  }
  stv(out + i * N, y);
}

// ------------------------------------------------------------------ M-CMoE routing
// Lane = component (C <= 64): weights = softmax over the top-k logits (equal
// logits by lowest index, as torch.topk takes them), 0 elsewhere; coef[c][j] = vproj[c][j]
// sigmoid(sig[c][j]) weight[c].  Components off the top k are read and multiplied like the others: an
// infinite or NaN vproj or sig there gives NaN, as the tensor ops' product with a weight of 0 does.
// Four waves share a token's row, the first forms the weights.  (One wave per token with ds_bpermute
// ranks: 17 us for 64 tokens and 32 us for 8192 at C 64, r 32 bf16; all four waves ranking: 10 and 57;
// so 5 and 27.)
constexpr int GW = 4;  // waves per token
template <typename T>
__global__ __launch_bounds__(64 * GW) void mcmoe_coef_kernel(const T* __restrict__ logits,
                                                             const T* __restrict__ sig,
                                                             const T* __restrict__ vproj,
                                                             T* __restrict__ coef, int topk,
                                                             int C, int r) {
  __shared__ float ws[64];
  const int64_t t = blockIdx.x;
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x;
    const bool in = lane < C;
    const float l = in ? io<T>::load(logits, t * C + lane) : -__builtin_inff();
    // logits as unsigned integers in their order, NaN above everything (as topk takes it) and the
    // lanes past the components below; the rank counts those before this one
    const uint32_t b = __float_as_uint(l + 0.f);  // -0 counts as +0
    const uint32_t key = !in ? 0u : l != l ? ~0u : (b & 0x80000000u) ? ~b : b | 0x80000000u;
    int rank = 0;
#pragma unroll
    for (int c = 0; c < 64; ++c) {
      const uint32_t o = __builtin_amdgcn_readlane(key, c);
      rank += o > key || (o == key && c < lane);
    }
    const bool sel = in && rank < topk;
    float m = sel ? l : -__builtin_inff();
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    const float p = sel ? expf(l - m) : 0.f;  // NaN for a NaN logit or an infinite maximum
    float sum = p;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off);
    ws[lane] = p / sum;  // 0 off the top k; NaN throughout if the sum is not finite
  }
  __syncthreads();
  constexpr int N = Vec<T>::N;
  const int per = r / N, total = C * per;  // 16-byte pieces of a component / of the row
  for (int e = threadIdx.x; e < total; e += 64 * GW) {
    const float wc = ws[e / per];
    const int64_t o = t * C * r + static_cast<int64_t>(e) * N;
    const Vec<T> s = ldv(sig + o), v = ldv(vproj + o);
    Vec<T> y;
#pragma unroll
    for (int j = 0; j < N; ++j)
      y.e[j] = round_to<T>(io<T>::to_f32(v.e[j]) * sigmoid_for<T>(io<T>::to_f32(s.e[j])) * wc);
    stv(coef + o, y);
  }
}

// ------------------------------------------------------------------ RMSNorm, adds, RMSNorm
// x = w1 ? rmsnorm(a; w1) : a;  s = (x + c) + b (each term optional, rounded after each add as the
// tensor ops are);  s stored if `sum`;  out = w2 ? rmsnorm(s; w2).  One workgroup per row; a row's
// pieces stay in registers.
constexpr int NV = 8;       // 16-byte pieces a thread holds at most
constexpr int NTH = 128;
__device__ __forceinline__ float block_sum(float x, float* red) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = x;
  __syncthreads();
  const float y = red[0] + red[1];
  __syncthreads();
  return y;
}
template <typename T>
__global__ __launch_bounds__(NTH) void norm_add_kernel(const T* __restrict__ a, const T* __restrict__ w1,
                                                       float eps1, const T* __restrict__ c,
                                                       const T* __restrict__ b, T* __restrict__ sum,
                                                       const T* __restrict__ w2, float eps2,
                                                       T* __restrict__ out, int d) {
  __shared__ float red[NTH / 64];
  constexpr int N = Vec<T>::N;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * d;
  const int nvec = d / N;
  float x[NV][N];
  float ss = 0.f;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int i = threadIdx.x + NTH * v;
    if (i >= nvec) break;
    const Vec<T> q = ldv(a + row + i * N);
#pragma unroll
    for (int j = 0; j < N; ++j) {
      x[v][j] = io<T>::to_f32(q.e[j]);
      ss = fmaf(x[v][j], x[v][j], ss);
    }
  }
  float scale = 1.f;
  if (w1 != nullptr) scale = rsqrtf(block_sum(ss, red) / d + eps1);
  ss = 0.f;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int i = threadIdx.x + NTH * v;
    if (i >= nvec) break;
    if (w1 != nullptr) {
      const Vec<T> wv = ldv(w1 + i * N);
#pragma unroll
      for (int j = 0; j < N; ++j) x[v][j] = rounded<T>(x[v][j] * scale * io<T>::to_f32(wv.e[j]));
    }
    if (c != nullptr) {
      const Vec<T> q = ldv(c + row + i * N);
#pragma unroll
      for (int j = 0; j < N; ++j) x[v][j] = rounded<T>(x[v][j] + io<T>::to_f32(q.e[j]));
    }
    if (b != nullptr) {
      const Vec<T> q = ldv(b + row + i * N);
#pragma unroll
      for (int j = 0; j < N; ++j) x[v][j] = rounded<T>(x[v][j] + io<T>::to_f32(q.e[j]));
    }
    if (sum != nullptr) {
      Vec<T> y;
#pragma unroll
      for (int j = 0; j < N; ++j) y.e[j] = round_to<T>(x[v][j]);
      stv(sum + row + i * N, y);
    }
#pragma unroll
    for (int j = 0; j < N; ++j) ss = fmaf(x[v][j], x[v][j], ss);
  }
  if (w2 == nullptr) return;
  scale = rsqrtf(block_sum(ss, red) / d + eps2);
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int i = threadIdx.x + NTH * v;
    if (i >= nvec) break;
    const Vec<T> wv = ldv(w2 + i * N);
    Vec<T> y;
#pragma unroll
    for (int j = 0; j < N; ++j) y.e[j] = round_to<T>(x[v][j] * scale * io<T>::to_f32(wv.e[j]));
    stv(out + row + i * N, y);
  }
}

// ------------------------------------------------------------------ halting update
// One adaptive-depth step of every token (acd_engine.py:128-150), one workgroup per token, all
// quantities rounded to the stream's type after each operation as the tensor ops are:
//   h' = active ? out : h;  p = sigmoid(w . h' + b) (0 below the minimum depth);  acc' = acc + p;
//   halted = active and acc' >= threshold;  rem = 1 - acc, 0 where that is negative (NaN kept);
//   final += ((halted ? rem : p) active) h';  depth += active, then += rem halted;
//   active' = active and not halted
// (active and halted as 0 or 1: a NaN p or rem reaches the sums of every token, as in the tensor ops).
// mode: 0 as above, 1 below the minimum depth (p = 0), 2 the loop's end: final += (rem active) h,
// depth += rem active, and nothing else changes.
template <typename T>
__global__ __launch_bounds__(NTH) void halting_kernel(const T* out, const T* h, T* h_next,
                                                      const T* __restrict__ w, const T* __restrict__ bias,
                                                      T* __restrict__ acc, T* __restrict__ depth,
                                                      const uint8_t* active, uint8_t* still,
                                                      T* __restrict__ final_h, float threshold,
                                                      int mode, int d) {
  __shared__ float red[NTH / 64];
  constexpr int N = Vec<T>::N;
  const int64_t t = blockIdx.x, row = t * d;
  const int nvec = d / N;
  const bool on = active[t] != 0;
  const float a0 = io<T>::load(acc, t), dp = io<T>::load(depth, t);
  const T* src = on && mode != 2 ? out : h;
  Vec<T> x[NV];
  float dot = 0.f;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int i = threadIdx.x + NTH * v;
    if (i >= nvec) break;
    x[v] = ldv(src + row + i * N);
    if (mode != 0) continue;
    const Vec<T> wv = ldv(w + i * N);
#pragma unroll
    for (int j = 0; j < N; ++j) dot = fmaf(io<T>::to_f32(x[v].e[j]), io<T>::to_f32(wv.e[j]), dot);
  }
  dot = block_sum(dot, red);  // its barriers also put every read of acc, depth, active before the writes
  const float p = mode == 0 ? rounded<T>(sigmoid_for<float>(rounded<T>(dot + io<T>::load(bias, 0)))) : 0.f;
  const float a1 = rounded<T>(a0 + p);
  const bool halted = on && (mode == 2 || a1 >= threshold);
  const float left = rounded<T>(1.f - a0), rem = left < 0.f ? 0.f : left;
  const float wt = (halted ? rem : p) * (on ? 1.f : 0.f);
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    const int i = threadIdx.x + NTH * v;
    if (i >= nvec) break;
    Vec<T> f = ldv(final_h + row + i * N);
#pragma unroll
    for (int j = 0; j < N; ++j)
      f.e[j] = round_to<T>(io<T>::to_f32(f.e[j]) + rounded<T>(wt * io<T>::to_f32(x[v].e[j])));
    stv(final_h + row + i * N, f);
    if (mode != 2) stv(h_next + row + i * N, x[v]);
  }
  if (threadIdx.x == 0) {
    float dn = mode == 2 ? dp : rounded<T>(dp + (on ? 1.f : 0.f));
    dn = rounded<T>(dn + rem * (halted ? 1.f : 0.f));
    io<T>::store(depth, t, dn);
    if (mode == 2) return;
    io<T>::store(acc, t, a1);
    still[t] = on && !halted;
  }
}

template <typename F> int by_type(int dtype, F&& f) {
  if (dtype == VMI_F32) return f(float{});
  if (dtype == VMI_BF16) return f(bf16_t{});
  if (dtype == VMI_F16) return f(f16_t{});
  return VMI_ERR_INVALID_ARG;
}
bool aligned16(std::initializer_list<const void*> ps) {
  for (const void* p : ps)
    if (reinterpret_cast<uintptr_t>(p) % 16 != 0) return false;
  return true;
}
int elem_size(int dtype) { return dtype == VMI_F32 ? 4 : 2; }
// a row of d elements is whole 16-byte pieces and fits the registers of a workgroup
bool row_fits(int64_t d, int dtype) {
  const int n = 16 / elem_size(dtype);
  return d > 0 && d % n == 0 && d <= static_cast<int64_t>(NTH) * NV * n;
}

}  // namespace layer
}  // namespace vmi

using namespace vmi;
using namespace vmi::layer;

extern "C" int vmi_situ_glu(const void* gate, const void* up, int dtype, float beta1, float beta2,
                            void* out, int64_t n, void* stream) {
  if (n < 0 || (n > 0 && (gate == nullptr || up == nullptr || out == nullptr))) return VMI_ERR_INVALID_ARG;
  return by_type(dtype, [&](auto tag) -> int {
    using T = decltype(tag);
    constexpr int N = Vec<T>::N;
    if (n % N != 0 || !aligned16({gate, up, out})) return VMI_ERR_UNSUPPORTED;
    const int64_t nvec = n / N, blocks = (nvec + 255) / 256;
    if (blocks > INT32_MAX) return VMI_ERR_UNSUPPORTED;
    if (n == 0) return VMI_OK;
    hipLaunchKernelGGL(situ_glu_kernel<T>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0,
                       static_cast<hipStream_t>(stream), static_cast<const T*>(gate),
                       static_cast<const T*>(up), static_cast<T*>(out), beta1, beta2, nvec);
    return hip_status(hipGetLastError());
  });
}

extern "C" int vmi_mcmoe_coef(const void* logits, const void* sigma, const void* vproj, int dtype,
                              int64_t top_k, void* coef, int64_t n, int64_t components, int64_t rank,
                              void* stream) {
  if (n < 0 || components < 1 || rank < 1 || top_k < 1 || top_k > components) return VMI_ERR_INVALID_ARG;
  if (n > 0 && (logits == nullptr || sigma == nullptr || vproj == nullptr || coef == nullptr))
    return VMI_ERR_INVALID_ARG;
  return by_type(dtype, [&](auto tag) -> int {
    using T = decltype(tag);
    if (components > 64 || rank % Vec<T>::N != 0 || rank > 4096 || !aligned16({sigma, vproj, coef}))
      return VMI_ERR_UNSUPPORTED;
    if (n > INT32_MAX) return VMI_ERR_UNSUPPORTED;
    if (n == 0) return VMI_OK;
    hipLaunchKernelGGL(mcmoe_coef_kernel<T>, dim3(static_cast<unsigned>(n)), dim3(64 * GW), 0,
                       static_cast<hipStream_t>(stream), static_cast<const T*>(logits),
                       static_cast<const T*>(sigma), static_cast<const T*>(vproj),
                       static_cast<T*>(coef), static_cast<int>(top_k),
                       static_cast<int>(components), static_cast<int>(rank));
    return hip_status(hipGetLastError());
  });
}

extern "C" int vmi_norm_add(const void* a, const void* w1, float eps1, const void* c, const void* b,
                            void* sum, const void* w2, float eps2, void* out, int dtype, int64_t rows,
                            int64_t d, void* stream) {
  if (rows < 0 || d < 1 || (rows > 0 && a == nullptr) || (w2 != nullptr) != (out != nullptr) ||
      (sum == nullptr && out == nullptr))
    return VMI_ERR_INVALID_ARG;
  return by_type(dtype, [&](auto tag) -> int {
    using T = decltype(tag);
    if (!row_fits(d, dtype) || rows > INT32_MAX || !aligned16({a, w1, c, b, sum, w2, out}))
      return VMI_ERR_UNSUPPORTED;
    if (rows == 0) return VMI_OK;
    hipLaunchKernelGGL(norm_add_kernel<T>, dim3(static_cast<unsigned>(rows)), dim3(NTH), 0,
                       static_cast<hipStream_t>(stream), static_cast<const T*>(a),
                       static_cast<const T*>(w1), eps1, static_cast<const T*>(c),
                       static_cast<const T*>(b), static_cast<T*>(sum), static_cast<const T*>(w2), eps2,
                       static_cast<T*>(out), static_cast<int>(d));
    return hip_status(hipGetLastError());
  });
}

extern "C" int vmi_halting_update(const void* out, const void* h, void* h_next, const void* w,
                                  const void* bias, void* acc, void* depth, const uint8_t* active,
                                  uint8_t* still, void* final_h, float threshold, int mode, int dtype, int64_t rows, int64_t d, void* stream) {
  if (rows < 0 || d < 1 || mode < 0 || mode > 2) return VMI_ERR_INVALID_ARG;
  if (rows > 0 && (h == nullptr || acc == nullptr || depth == nullptr || active == nullptr || final_h == nullptr))
    return VMI_ERR_INVALID_ARG;
  if (rows > 0 && mode != 2 &&
      (out == nullptr || h_next == nullptr || w == nullptr || bias == nullptr || still == nullptr))
    return VMI_ERR_INVALID_ARG;
  return by_type(dtype, [&](auto tag) -> int {
    using T = decltype(tag);
    if (!row_fits(d, dtype) || rows > INT32_MAX || !aligned16({out, h, h_next, w, final_h})) return VMI_ERR_UNSUPPORTED;
    if (rows == 0) return VMI_OK;
    hipLaunchKernelGGL(halting_kernel<T>, dim3(static_cast<unsigned>(rows)), dim3(NTH), 0,
                       static_cast<hipStream_t>(stream), static_cast<const T*>(out), static_cast<const T*>(h),
                       static_cast<T*>(h_next), static_cast<const T*>(w), static_cast<const T*>(bias), static_cast<T*>(acc),
                       static_cast<T*>(depth), active, still, static_cast<T*>(final_h), threshold,
                       mode, static_cast<int>(d));
    return hip_status(hipGetLastError());
  });
}
