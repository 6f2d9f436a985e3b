// y = x W^T for a few rows: the projections around a decode step at a small batch (x [M, K], M <= 16,
// W [N, K] row-major, the reference's nn.Linear calls at seq_len 1, sssd_attention.py:114-126, :178).
//
// Bound by reading W (6.8 MB for the stacked SSSD projection at hidden 1024) and, at these sizes, by the
// launch.  A workgroup takes 16 rows of W and all of K, split over its 8 waves in pieces of 64 columns so
// that a wave's two loads cover whole 128-byte lines; a wave holds four pieces in flight.  W's rows are
// the A operand of the 16 x 16 matrix product and x's rows the B operand straight from memory (nothing is
// shared between waves, so nothing is staged); the 8 fp32 partials meet in LDS.  fp32 inputs take the
// exact fp32 product in the same arrangement.  [1, 1024] x [3328, 1024]^T bf16: 2.9 us (2.3 TB/s)
// against the library's 4.5, and 11 against 19.5 us of host time per call.
#include "vmi_common.h"
#include "vmi_dispatch.h"
#include "vmi_mfma.h"

namespace vmi {
namespace rowlin {

constexpr int NW = 8, NTH = 64 * NW;
constexpr int MR = 16;     // rows of W, and most rows of x, per workgroup
constexpr int PIECE = 64;  // columns a wave takes at a time
constexpr int FLY = 4;     // 16-byte loads of each operand in flight per lane

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// The k-slots of lane group g in one 16-byte load of each operand: 32 columns 16-bit, 16 columns fp32.
template <typename E>
__device__ __forceinline__ f32x4 product(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (sizeof(E) == 2) {
    typedef typename mfma_t<E>::v8 V8;
    return mfma_t<E>::mma16(__builtin_bit_cast(V8, a), __builtin_bit_cast(V8, b), c);
  } else {
    const f32x4 x = __builtin_bit_cast(f32x4, a), y = __builtin_bit_cast(f32x4, b);
#pragma unroll
    for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i], y[i], c, 0, 0, 0);
    return c;
  }
}

// K a multiple of the 16-byte piece, x, W and x_stride 16-byte aligned.
template <typename IO, typename E>
__global__ __launch_bounds__(NTH) void rows_linear_kernel(const E* __restrict__ x, int64_t x_stride,
                                                          const E* __restrict__ w, IO* __restrict__ y,
                                                          int M, int N, int64_t K) {
  constexpr int EL = 16 / sizeof(E);         // elements of a load
  constexpr int STEP = 4 * EL;               // columns of the four lane groups
  constexpr int SUB = PIECE / STEP;          // loads of a piece
  constexpr int NP = FLY / SUB;              // pieces in flight
  __shared__ float part[NW][MR][MR + 1];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * MR;
  // rows past the end repeat the last one; their results are not stored
  const E* wr = w + static_cast<int64_t>(min(n0 + l16, N - 1)) * K;
  const E* xr = x + static_cast<int64_t>(min(l16, M - 1)) * x_stride;
  f32x4 acc[2] = {};
  for (int64_t k0 = PIECE * wave; k0 < K; k0 += PIECE * NW * NP) {
    u32x4 a[FLY], b[FLY];
#pragma unroll
    for (int u = 0; u < FLY; ++u) {
      const int64_t k = k0 + PIECE * NW * (u / SUB) + STEP * (u % SUB) + EL * g;
      const int64_t kc = k < K ? k : 0;
      a[u] = *reinterpret_cast<const u32x4*>(wr + kc);
      b[u] = *reinterpret_cast<const u32x4*>(xr + kc);
    }
#pragma unroll
    for (int u = 0; u < FLY; ++u) {
      const int64_t k = k0 + PIECE * NW * (u / SUB) + STEP * (u % SUB) + EL * g;
      if (k >= K) a[u] = b[u] = u32x4{};
    }
#pragma unroll
    for (int u = 0; u < FLY; ++u) acc[u & 1] = product<E>(a[u], b[u], acc[u & 1]);
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) part[wave][4 * g + r][l16] = acc[0][r] + acc[1][r];
  __syncthreads();
  if (tid < MR * MR) {
    const int n = tid & 15, m = tid >> 4;
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < NW; ++i) s += part[i][n][m];
    if (m < M && n0 + n < N) io<IO>::store(y, static_cast<int64_t>(m) * N + n0 + n, s);
  }
}

}  // namespace rowlin
}  // namespace vmi

extern "C" int vmi_rows_linear(const void* x, int64_t x_stride, const void* w, int io_dtype, void* y,
                               int64_t M, int64_t N, int64_t K, void* stream) {
  using namespace vmi;
  using namespace vmi::rowlin;
  if (M < 0 || N < 0 || K < 0 || (M > 1 && x_stride < K)) return VMI_ERR_INVALID_ARG;
  if (io_dtype != VMI_F32 && io_dtype != VMI_BF16 && io_dtype != VMI_F16) return VMI_ERR_INVALID_ARG;
  const int64_t el = io_dtype == VMI_F32 ? 4 : 8;
  if (M > MR || K < 1 || K % el != 0 || (M > 1 && x_stride % el != 0) || N > INT32_MAX - MR)
    return VMI_ERR_UNSUPPORTED;
  if (M == 0 || N == 0) return VMI_OK;
  if (x == nullptr || w == nullptr || y == nullptr) return VMI_ERR_INVALID_ARG;
  if (((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w)) & 15) != 0) return VMI_ERR_UNSUPPORTED;
  const dim3 grid(static_cast<unsigned>((N + MR - 1) / MR)), block(NTH);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int m = static_cast<int>(M), n = static_cast<int>(N);
  if (io_dtype == VMI_BF16)
    hipLaunchKernelGGL((rows_linear_kernel<bf16_t, __bf16>), grid, block, 0, s, static_cast<const __bf16*>(x),
                       x_stride, static_cast<const __bf16*>(w), static_cast<bf16_t*>(y), m, n, K);
  else if (io_dtype == VMI_F16)
    hipLaunchKernelGGL((rows_linear_kernel<f16_t, _Float16>), grid, block, 0, s, static_cast<const _Float16*>(x),
                       x_stride, static_cast<const _Float16*>(w), static_cast<f16_t*>(y), m, n, K);
  else
    hipLaunchKernelGGL((rows_linear_kernel<float, float>), grid, block, 0, s, static_cast<const float*>(x),
                       x_stride, static_cast<const float*>(w), static_cast<float*>(y), m, n, K);
  return hip_status(hipGetLastError());
}
