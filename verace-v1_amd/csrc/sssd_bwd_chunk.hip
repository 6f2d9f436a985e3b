// Chunked (WY) backward of the SSSD scan: the per-token reverse recursion of sssd_bwd.hip
// regrouped by chunks of C = 16 tokens, so every state-dependent product is a small GEMM.
//
// Per chunk (U = [k_1 v_1 .. k_C v_C] D x 32, T~ = (I - L)^-1 blockdiag(M) 32 x 32, the
// forward's chunk factor I + U T~ U^T, states Psi_s -> Psi_e, adjoints Lam_s <- Lam_e):
//   Psi_s = Psi_e + U T~^T U^T Psi_e            (the factor is orthogonal)
//   W = U^T Psi_s,  Z = T~ W,  X = mask o (Z Q),  dX = mask o (U^T dO)
//   dZ = U^T Lam_e + dX Q^T,   dT~ = dZ W^T,     dW = T~^T dZ
//   dQ = Z^T dX + Psi_s^T dO,  dU = Lam_e Z^T + dO X^T + Psi_s dW^T
//   Lam_s = Lam_e + dO Q^T + U dW
// (mask[rho][t] = token(rho) <= t).  Then, per chunk and without the state, dT~ through
// T~ = A B (A = (I - L)^-1, B = blockdiag(M), L_ti = M_t G_ti for i < t):
//   dA = dT~ B^T, dB = A^T dT~, dL = A^T dA A^T (strictly lower blocks),
//   dM_t = dB_tt + sum_i dL_ti G_ti^T,  dG_ti = M_t^T dL_ti,
// M_t(delta_t, kk, vv, kv) as in vmi::cayley_coeffs, dU += U (dG + dG^T).
//
// Launches (S segments of the chunks, picked by plan()):
//   bwdc_prep_kernel    one wave per chunk: T~, A, G, M, dX -> workspace;
//   bwdc_pass_kernel<MAIN = false>  (S > 1) segments 1 .. S - 1 as maps of their end state:
//     Psi_start = X Psi_end, Lam_start = X Lam_end + B (both recursions share the factor);
//   bwdc_carry_kernel   (S > 1) the end state and adjoint of segments S - 2 .. 0;
//   bwdc_pass_kernel<MAIN = true>   every segment in reverse: dQ, and per chunk dT~ and dU;
//   bwdc_reduce_kernel  one workgroup per chunk: dT~ -> dM, dG -> dk, dv, ddelta.
//
// Split: a wave owns 16 columns of Psi and Lam as MFMA accumulators, a workgroup all D columns of
// one segment.  An accumulator tile (lane = column, registers = 4 rows per 16-lane group) is
// already an operand of every product that contracts over the state's rows or the rank, so those
// need no barrier; the three that contract over the columns (dU, dT~, X) read Lam_e, Psi_s, Z, dW,
// dZ and W back from LDS, once per chunk, and give complete sums.  (The earlier form gave a
// workgroup 16 columns of the whole sequence: seven barriers and a quarter of the work per
// barrier, and partial dU and dT~ of all column blocks through memory, 671 MB in fp32 at
// B4 T2048 H8 D128.)
//
// Measured at B4 T2048 H8 D128 (the earlier form in brackets): bf16 330 us (612): prep 33, maps 75,
// carry 34, main 132, reduce 56; fp32 615 us (1034): main 316 and maps 172, bound by the fp32 matrix
// rate (their 600 v_mfma_f32_16x16x4_f32 a wave and chunk are 16 of the 20 us); bf16 at D = 64: 155 us
// (448).  Relative error against fp64, fp32 inputs: 7e-7 .. 9e-7 (1.1e-6 .. 1.2e-6), bf16 2e-3 ..
// 3.8e-3 (4.2e-3: the partials were bf16).
#include <algorithm>
#include <type_traits>

#include "vmi_common.h"
#include "vmi_dispatch.h"
#include "vmi_lanes.h"
#include "vmi_mfma.h"

namespace vmi {
namespace bwdc {

constexpr int C = 16;   // tokens per chunk
constexpr int R = 32;   // rank rows of a chunk (k, v per token)
constexpr int NT = 256; // threads of the reduce kernel
// per-chunk record written by the prep kernel: T~, A = (I - L)^-1, G (R x R each), the M blocks,
// dX (R x C), then the bit mask of the chunk's tokens whose Cayley factor is not finite (the
// reference's non-finite guard, sssd_attention.py:45-71: such a token is the identity, its U rows
// count as zero and it gets no gradient) and 3 floats of padding (16-byte alignment)
constexpr int REC_A = R * R;
constexpr int REC_G = 2 * R * R;
constexpr int REC_M = 3 * R * R;
constexpr int REC_DX = REC_M + 4 * C;
constexpr int REC_BAD = REC_DX + R * C;
constexpr int REC = REC_BAD + 4;
// per-chunk result of the main pass: dT~ [R][R], then dU transposed, [R][D]
template <int D> struct PartC { static constexpr int size = R * R + D * R; };

typedef short s16x4 __attribute__((ext_vector_type(4)));

// two values as one word of bf16 (v_cvt_pk_bf16_f32: round to nearest even, the same bits as
// f32_to_bf16 for every non-NaN value, without its branch per element)
__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  const bf16x2_t v = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
  return __builtin_bit_cast(uint32_t, v);
}
__device__ __forceinline__ s16x4 pack4(f32x4 x) {
  return __builtin_bit_cast(s16x4, make_uint2(pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3])));
}
__device__ __forceinline__ f32x4 mma(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mma_bf16(s16x4 a, s16x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}
// Four k of a 16 x 16 product, lane group g holding k = 4 g + r in register r of both operands:
// exact fp32 products, or (LP) operands rounded to bf16; fp32 accumulation.
template <bool LP>
__device__ __forceinline__ f32x4 dot4(f32x4 a, f32x4 b, f32x4 c) {
  if constexpr (LP) return mma_bf16(pack4(a), pack4(b), c);
#pragma unroll
  for (int r = 0; r < 4; ++r) c = mma(a[r], b[r], c);
  return c;
}
__device__ __forceinline__ f32x4 lds4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
// Four rows' elements of one column (row pitch ld).
__device__ __forceinline__ f32x4 col4(const float* p, int ld) {
  return f32x4{p[0], p[ld], p[2 * ld], p[3 * ld]};
}

// N consecutive elements of a row as raw 32-bit words (one 8- or 16-byte load, two for 8
// fp32), and element j of them as a float.  The row must be aligned to its byte size.
template <typename T, int N> struct RowRaw {
  static constexpr int W = N * static_cast<int>(sizeof(T)) / 4;
  uint32_t w[W];
};
template <typename T, int N>
__device__ __forceinline__ RowRaw<T, N> load_raw(const T* p) {
  RowRaw<T, N> r;
  constexpr int W = RowRaw<T, N>::W;
  static_assert(W == 2 || W % 4 == 0, "8-byte or whole 16-byte pieces");
  if constexpr (W == 2) {
    const uint2 x = *reinterpret_cast<const uint2*>(p);
    r.w[0] = x.x; r.w[1] = x.y;
  } else {
#pragma unroll
    for (int i = 0; i < W / 4; ++i) {
      const uint4 x = reinterpret_cast<const uint4*>(p)[i];
      r.w[4 * i] = x.x; r.w[4 * i + 1] = x.y; r.w[4 * i + 2] = x.z; r.w[4 * i + 3] = x.w;
    }
  }
  return r;
}
// N consecutive raw elements (8 or 16 bytes) read with the nontemporal hint: streamed once.
template <typename T, int N>
__device__ __forceinline__ RowRaw<T, N> load_raw_nt(const T* p) {
  RowRaw<T, N> r;
  constexpr int W = RowRaw<T, N>::W;
  static_assert(W == 2 || W % 4 == 0, "8-byte or whole 16-byte pieces");
  if constexpr (W == 2) {
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    const u32x2 x = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(p));
    r.w[0] = x[0]; r.w[1] = x[1];
  } else {
#pragma unroll
    for (int i = 0; i < W / 4; ++i) {
      typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
      const u32x4 x = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p) + i);
      r.w[4 * i] = x[0]; r.w[4 * i + 1] = x[1]; r.w[4 * i + 2] = x[2]; r.w[4 * i + 3] = x[3];
    }
  }
  return r;
}
template <typename T, int N>
__device__ __forceinline__ void store_row(T* p, const float (&x)[N]) {
  RowRaw<T, N> r;
  constexpr int W = RowRaw<T, N>::W;
  if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int j = 0; j < N; ++j) r.w[j] = __float_as_uint(x[j]);
  } else {
#pragma unroll
    for (int j = 0; j < N; j += 2) {
      uint32_t lo, hi;
      if constexpr (std::is_same<T, bf16_t>::value) {
        const uint32_t w = pack_bf16x2(x[j], x[j + 1]);
        lo = w & 0xffffu;
        hi = w >> 16;
      } else {
        lo = __builtin_bit_cast(uint16_t, static_cast<f16_t>(x[j]));
        hi = __builtin_bit_cast(uint16_t, static_cast<f16_t>(x[j + 1]));
      }
      r.w[j >> 1] = lo | (hi << 16);
    }
  }
  if constexpr (W == 2) {
    *reinterpret_cast<uint2*>(p) = make_uint2(r.w[0], r.w[1]);
  } else {
#pragma unroll
    for (int i = 0; i < W / 4; ++i)
      reinterpret_cast<uint4*>(p)[i] = make_uint4(r.w[4 * i], r.w[4 * i + 1], r.w[4 * i + 2], r.w[4 * i + 3]);
  }
}
template <typename T, int N>
__device__ __forceinline__ float raw_elem(const RowRaw<T, N>& r, int j) {
  if constexpr (sizeof(T) == 4) {
    return __uint_as_float(r.w[j]);
  } else {
    const uint16_t hbits = static_cast<uint16_t>(r.w[j >> 1] >> (16 * (j & 1)));
    if constexpr (std::is_same<T, bf16_t>::value) return bf16_to_f32(hbits);
    else return static_cast<float>(__builtin_bit_cast(f16_t, hbits));
  }
}

// Workgroup barrier that orders LDS accesses only: it waits for this wave's LDS operations, not
// for its global loads and stores (which __syncthreads() also waits for).
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);  // vmcnt(63) expcnt(7) lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Four consecutive elements of a 16-bit or fp32 row, as they lie in memory (16-bit: x, y).
__device__ __forceinline__ uint4 load4_raw(const void* p, int64_t i, bool f32) {
  if (f32) return *reinterpret_cast<const uint4*>(static_cast<const float*>(p) + i);
  const uint2 w = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(p) + i);
  return make_uint4(w.x, w.y, 0u, 0u);
}
__device__ __forceinline__ f32x4 raw_f32(uint4 w, int dtype) {
  if (dtype == VMI_F32) return __builtin_bit_cast(f32x4, w);
  if (dtype == VMI_BF16)
    return f32x4{bf16_to_f32(w.x & 0xffffu), bf16_to_f32(w.x >> 16), bf16_to_f32(w.y & 0xffffu), bf16_to_f32(w.y >> 16)};
  const f16x4 h = __builtin_bit_cast(f16x4, make_uint2(w.x, w.y));
  return f32x4{static_cast<float>(h[0]), static_cast<float>(h[1]), static_cast<float>(h[2]), static_cast<float>(h[3])};
}
template <typename IO> constexpr int io_code() {
  return std::is_same<IO, float>::value ? VMI_F32 : std::is_same<IO, bf16_t>::value ? VMI_BF16 : VMI_F16;
}

// LDS row strides of the reduce kernel (64 banks of 4 B): with 37 every MFMA operand read is at
// most 2-way bank conflicted across the wave, in both orientations.
constexpr int L32 = 37;  // 32-wide matrices

// Cm (M x N, row stride ldc) = opA(A) opB(B), K the inner size, all in LDS, fp32.
// opA(m, k) = TA ? A[k lda + m] : A[m lda + k];  opB(k, n) = TB ? B[n ldb + k] : B[k ldb + n].
// 16 x 16 output tiles round robin over the NT / 64 waves.  Two accumulators over alternate k
// steps halve the dependent chain.
template <int M, int N, int K, bool TA, bool TB>
__device__ __forceinline__ void lgemm(const float* A, int lda, const float* B, int ldb, float* Cm,
                                      int ldc, int wave, int lane) {
  constexpr int TN = N / 16, NTILE = (M / 16) * TN;
  const int l16 = lane & 15, kq = lane >> 4;
  for (int tile = wave; tile < NTILE; tile += NT / 64) {
    const int tm = tile / TN, tn = tile % TN;
    const int am = 16 * tm + l16, bn = 16 * tn + l16;
    f32x4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int k0 = 0; k0 < K; k0 += 8) {
      const int k = k0 + kq, k1 = k + 4;
      acc0 = mma(TA ? A[k * lda + am] : A[am * lda + k], TB ? B[bn * ldb + k] : B[k * ldb + bn], acc0);
      acc1 = mma(TA ? A[k1 * lda + am] : A[am * lda + k1], TB ? B[bn * ldb + k1] : B[k1 * ldb + bn], acc1);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) Cm[(16 * tm + 4 * kq + r) * ldc + bn] = acc0[r] + acc1[r];
  }
}

// ---------------------------------------------------------------- T~, A, G, M, dX of every chunk
// One wave per chunk and no workgroup barrier.  The operands of G = U^T U and dX = mask o (U^T dO)
// come straight from global memory in the MFMA layout (lane l16 = rank row or token, group g:
// features 16 S + 4 g ..+ 3); G passes through LDS once, to be read by rows in the substitution.
constexpr int PW = 4;    // waves (chunks) per workgroup
constexpr int GP = 36;   // G row pitch in LDS (floats)

template <typename IO, int D>
__global__ __launch_bounds__(64 * PW) void bwdc_prep_kernel(
    const IO* __restrict__ k, const IO* __restrict__ v, const void* __restrict__ dout, int do_dtype,
    const void* __restrict__ delta, int delta_dtype, float* __restrict__ rec, int T, int H, int nch,
    int64_t total) {
  __shared__ __attribute__((aligned(16))) float Gs[PW][R * GP];
  __shared__ float4 Ms[PW][C];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int64_t id = static_cast<int64_t>(blockIdx.x) * PW + wave;
  if (id >= total) return;  // whole waves; no barrier below
  const int bh = static_cast<int>(id / nch), n = static_cast<int>(id - static_cast<int64_t>(bh) * nch);
  const int b = bh / H, h = bh - b * H;
  float* G = Gs[wave];
  float* out = rec + id * REC;
  // rank row rho = l16 of each 16-row half: token rho / 2, k for even rho and v for odd
  const IO* src = (l16 & 1) ? v : k;
  const int t0 = n * C + (l16 >> 1), t1 = t0 + C / 2, td = n * C + l16;
  const int64_t base = static_cast<int64_t>(b) * T * H + h;
  auto row = [&](int t) { return (base + static_cast<int64_t>(t < T ? t : 0) * H) * D; };
  float dl = 0.f;
  if (lane < C && td < T) dl = load_scalar(delta, delta_dtype, base + static_cast<int64_t>(td) * H);
  constexpr int SS = D / 16;
  constexpr int IOC = io_code<IO>();
  uint4 x0[SS], x1[SS], xd[SS];
#pragma unroll
  for (int S = 0; S < SS; ++S) {
    const int d = 16 * S + 4 * g;
    x0[S] = load4_raw(src, row(t0) + d, IOC == VMI_F32);
    x1[S] = load4_raw(src, row(t1) + d, IOC == VMI_F32);
  }
  if (do_dtype == VMI_F32) {  // uniform; every load issued before the first wait
#pragma unroll
    for (int S = 0; S < SS; ++S) xd[S] = load4_raw(dout, row(td) + 16 * S + 4 * g, true);
  } else {
#pragma unroll
    for (int S = 0; S < SS; ++S) xd[S] = load4_raw(dout, row(td) + 16 * S + 4 * g, false);
  }
  bool keep0 = t0 < T, keep1 = t1 < T;  // this lane's U rows count
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  auto gram = [&]() {
    f32x4 p[2][3] = {};
#pragma unroll
    for (int S = 0; S < SS; ++S) {
      const f32x4 a0 = keep0 ? raw_f32(x0[S], IOC) : zero, a1 = keep1 ? raw_f32(x1[S], IOC) : zero;
      p[S & 1][0] = dot4<false>(a0, a0, p[S & 1][0]);
      p[S & 1][1] = dot4<false>(a1, a0, p[S & 1][1]);
      p[S & 1][2] = dot4<false>(a1, a1, p[S & 1][2]);
    }
    const f32x4 g00 = p[0][0] + p[1][0], g10 = p[0][1] + p[1][1], g11 = p[0][2] + p[1][2];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      G[(4 * g + r) * GP + l16] = g00[r];
      G[(16 + 4 * g + r) * GP + l16] = g10[r];
      G[l16 * GP + 16 + 4 * g + r] = g10[r];
      G[(16 + 4 * g + r) * GP + 16 + l16] = g11[r];
    }
    __builtin_amdgcn_wave_barrier();
  };
  gram();
  bool ok = true;
  if (lane < C) {
    const int t = lane;
    const cayley2 m = cayley_guarded(dl, G[(2 * t) * GP + 2 * t], G[(2 * t + 1) * GP + 2 * t + 1],
                                     G[(2 * t + 1) * GP + 2 * t], ok);
    Ms[wave][t] = make_float4(m.m00, m.m01, m.m10, m.m11);
    *reinterpret_cast<float4*>(out + REC_M + 4 * t) = Ms[wave][t];
  }
  const int bad = static_cast<int>(__ballot(!ok));  // tokens are lanes 0 .. C - 1
  __builtin_amdgcn_wave_barrier();
  if (bad != 0) {  // uniform over the wave: their U rows count as zero
    keep0 = keep0 && !((bad >> (l16 >> 1)) & 1);
    keep1 = keep1 && !((bad >> (C / 2 + (l16 >> 1))) & 1);
    gram();
  }
  {  // dX = mask o (U^T dO)
    f32x4 p[2][2] = {};
#pragma unroll
    for (int S = 0; S < SS; ++S) {
      const f32x4 a0 = keep0 ? raw_f32(x0[S], IOC) : zero, a1 = keep1 ? raw_f32(x1[S], IOC) : zero;
      const f32x4 d = td < T ? raw_f32(xd[S], do_dtype) : zero;
      p[S & 1][0] = dot4<false>(a0, d, p[S & 1][0]);
      p[S & 1][1] = dot4<false>(a1, d, p[S & 1][1]);
    }
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int rho = 16 * half + 4 * g + r;
        out[REC_DX + rho * C + l16] = (rho >> 1) <= l16 ? p[0][half][r] + p[1][half][r] : 0.f;
      }
  }
  // A = I + L A by block rows: lane (a, c) = (lane >> 5, lane & 31) keeps column c of A in
  // registers and forms row 2t + a of sum_{i<t} G_ti A_i; the halves exchange their rows
  // (v_permlane32_swap) and M_t takes them to the two rows of A
  const int c = lane & 31, a = lane >> 5;
  float col[R];
#pragma unroll
  for (int t = 0; t < C; ++t) {
    const float* gr = G + (2 * t + a) * GP;
    float s0 = 0.f, s1 = 0.f;
#pragma unroll
    for (int m = 0; m < R; m += 4) {
      if (m + 4 > 2 * t) continue;
      const f32x4 g4 = lds4(gr + m);
      s0 = fmaf(g4[0], col[m], s0);
      s1 = fmaf(g4[1], col[m + 1], s1);
      s0 = fmaf(g4[2], col[m + 2], s0);
      s1 = fmaf(g4[3], col[m + 3], s1);
    }
    if ((2 * t) % 4 != 0) {
      const float2 g2 = *reinterpret_cast<const float2*>(gr + 2 * t - 2);
      s0 = fmaf(g2.x, col[2 * t - 2], s0);
      s1 = fmaf(g2.y, col[2 * t - 1], s1);
    }
    const float mine = s0 + s1;
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mine), __float_as_uint(mine),
                                                     false, false);
    // lanes 32-63 receive lanes 0-31 in the first result, lanes 0-31 lanes 32-63 in the second
    const float other = __uint_as_float(a ? sw[0] : sw[1]);
    const float rk = a ? other : mine, rv = a ? mine : other;
    const float4 m = Ms[wave][t];
    col[2 * t] = (2 * t == c ? 1.f : 0.f) + fmaf(m.x, rk, m.y * rv);
    col[2 * t + 1] = (2 * t + 1 == c ? 1.f : 0.f) + fmaf(m.z, rk, m.w * rv);
  }
  // T~ = A blockdiag(M): column c = 2s + cb takes A's columns 2s and 2s + 1 (this lane's and its
  // neighbour's) with M_s[.][cb]
  const float4 ms = Ms[wave][c >> 1];
  const float m_own = (c & 1) ? ms.w : ms.x, m_other = (c & 1) ? ms.y : ms.z;
  const uint32_t odd = a ? ~0u : 0u;  // (a bit select: `a ? x : y` became an indexed stack array)
#pragma unroll
  for (int r = 0; r < R; r += 2) {
    const float own = __uint_as_float((__float_as_uint(col[r + 1]) & odd) | (__float_as_uint(col[r]) & ~odd));
    const float nb = dpp_f32<0xB1>(own);  // quad_perm(1, 0, 3, 2): lane c ^ 1
    out[(r + a) * R + c] = fmaf(own, m_own, nb * m_other);
    out[REC_A + (r + a) * R + c] = own;
  }
#pragma unroll
  for (int i = 0; i < R * R / 256; ++i) {
    const int e = 4 * (lane + 64 * i);
    *reinterpret_cast<f32x4*>(out + REC_G + e) = lds4(G + (e / R) * GP + e % R);
  }
  if (lane == 0) out[REC_BAD] = __int_as_float(bad);
}

// ---------------------------------------------------------------- the segments, in reverse
struct Args {
  const void *q, *k, *v, *dout;
  int do_dtype;
  const float* rec;
  const float *psi_T, *dpsi_T;  // [BH][D][D]; dpsi_T may be null (zero)
  float *xmap, *bmap;           // MAIN = false: X, B of segment s >= 1 at [(s - 1) BH + bh]
  const float *epsi, *elam;     // MAIN: end states of segment s < S - 1 at [s BH + bh]
  void* dq;
  float* dpsi0;                 // may be null
  float* part;                  // MAIN: per chunk, PartC
  int T, H, BH, nch, seg_chunks, nseg;
};

// MAIN: psi, lam = the segment's end state and adjoint.  Else X from the identity and B from
// zero, which take the same steps.  Tile S, register r: row 16 S + 4 g + r of column colj.
template <int D, bool MAIN>
__device__ __forceinline__ void init_states(const Args& a, int bh, int seg, int colj, int g,
                                            f32x4 (&psi)[D / 16], f32x4 (&lam)[D / 16]) {
  constexpr int SS = D / 16;
  const int64_t DD = static_cast<int64_t>(D) * D;
  const float* ls = nullptr;
  if constexpr (MAIN) {
    const bool last = seg == a.nseg - 1;
    const int64_t o = (static_cast<int64_t>(seg) * a.BH + bh) * DD;
    const float* ps = last ? a.psi_T + bh * DD : a.epsi + o;
    ls = last ? (a.dpsi_T ? a.dpsi_T + bh * DD : nullptr) : a.elam + o;
#pragma unroll
    for (int S = 0; S < SS; ++S) psi[S] = col4(ps + (16 * S + 4 * g) * D + colj, D);
  } else {
#pragma unroll
    for (int S = 0; S < SS; ++S)
#pragma unroll
      for (int r = 0; r < 4; ++r) psi[S][r] = 16 * S + 4 * g + r == colj ? 1.f : 0.f;
  }
  if (ls != nullptr) {
#pragma unroll
    for (int S = 0; S < SS; ++S) lam[S] = col4(ls + (16 * S + 4 * g) * D + colj, D);
  } else {
#pragma unroll
    for (int S = 0; S < SS; ++S) lam[S] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
}

// dPsi_0 (MAIN, the first segment), or the segment's map X, B.
template <int D, bool MAIN>
__device__ __forceinline__ void store_states(const Args& a, int bh, int seg, int colj, int g,
                                             const f32x4 (&psi)[D / 16], const f32x4 (&lam)[D / 16]) {
  const int64_t DD = static_cast<int64_t>(D) * D;
  if (MAIN && (seg != 0 || a.dpsi0 == nullptr)) return;
  const int64_t o = MAIN ? bh * DD : (static_cast<int64_t>(seg - 1) * a.BH + bh) * DD;
#pragma unroll
  for (int S = 0; S < D / 16; ++S)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int64_t e = o + (16 * S + 4 * g + r) * D + colj;
      if constexpr (MAIN) {
        a.dpsi0[e] = lam[S][r];
      } else {
        a.xmap[e] = psi[S][r];
        a.bmap[e] = lam[S][r];
      }
    }
}

// The lane number as a value the compiler cannot see through: what is computed from it inside a
// loop stays there.  (The 30-odd LDS addresses of a pass, hoisted out of its chunk loop, spilled
// 53 registers at D = 128, and their reloads waited for the chunk's stores: 214 -> 131 us at B4 T2048
// H8; where nothing spills, hoisting them is 4 % faster.)
__device__ __forceinline__ int opaque(int lane) {
  asm volatile("" : "+v"(lane));
  return lane;
}

template <typename IO, int D, bool MAIN>
__global__ __launch_bounds__(4 * D) void bwdc_pass_kernel(Args a) {
  constexpr int NW = D / 16, NTC = 4 * D, SS = D / 16, LU = D + 4, KP = NW / 2;
  // bf16 / fp16 inputs: the per-chunk gradient products take bf16 operands (their 2e-2 bar);
  // the rebuild of Psi, W and the adjoint update, carried across chunks, stay fp32
  constexpr bool LP = !std::is_same<IO, float>::value;
  constexpr int IOC = io_code<IO>();
  constexpr int TP = 36, XPP = 20;
  // The chunk's inputs.  Pitches 4 mod 64 banks (or 4 times an odd number): 16-byte reads by 16
  // rows and 4-byte accesses of 4 x 16 blocks are conflict-free.
  __shared__ __attribute__((aligned(16))) float U[R * LU], Q[C * LU], dO[C * LU];  // token rows
  __shared__ __attribute__((aligned(16))) float Tt[R * TP], Gm[R * TP], dX[R * XPP];
  __shared__ __attribute__((aligned(16))) float XP[MAIN ? KP * R * XPP : 4];
  // What the products over the columns read.  bf16: column-major (one 8-byte write per lane and
  // tile, read by the transposing ds_read_b64_tr_b16), everything at once.  fp32: row-major, one
  // state and one 32-row matrix at a time.
  constexpr int PJ = D + 8, PZ = R + 4;
  __shared__ __attribute__((aligned(16))) uint16_t LSb[MAIN && LP ? D * PJ : 8], PSb[MAIN && LP ? D * PJ : 8];
  __shared__ __attribute__((aligned(16))) uint16_t Zb[MAIN && LP ? D * PZ : 8], dWb[MAIN && LP ? D * PZ : 8],
      dZb[MAIN && LP ? D * PZ : 8], Wb[MAIN && LP ? D * PZ : 8];
  __shared__ __attribute__((aligned(16))) float SB[MAIN && !LP ? D * LU : 4], ZB[MAIN && !LP ? R * LU : 4];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: scalar addresses and branches
  const int bh = blockIdx.x, seg = MAIN ? blockIdx.y : blockIdx.y + 1, b = bh / a.H, h = bh - b * a.H;
  const int T = a.T;
  const int c0 = seg * a.seg_chunks, c1 = min(a.nch, c0 + a.seg_chunks);

  // thread's share of a chunk's inputs: features fd .. fd + 3 of token ft's rows, RT elements of
  // T~ and of G, RX of dX
  constexpr int RT = R * R / NTC, RX = R * C / NTC;
  typedef float fRT __attribute__((ext_vector_type(RT)));
  const int ft = tid / (D / 4), fd = 4 * (tid % (D / 4));
  uint4 rk, rv, rq, rd;
  fRT rt, rg;
  float rx[RX];
  int rbad = 0;
  bool rok = false;
  auto tok = [&](int t) { return (static_cast<int64_t>(b) * T + t) * a.H + h; };
  auto fetch = [&](int c) {
    const int t = c * C + ft;
    rok = t < T;
    const int64_t o = tok(rok ? t : 0) * D + fd;
    rk = load4_raw(a.k, o, IOC == VMI_F32);
    rv = load4_raw(a.v, o, IOC == VMI_F32);
    rq = load4_raw(a.q, o, IOC == VMI_F32);
    rd = load4_raw(a.dout, o, a.do_dtype == VMI_F32);
    const float* rec = a.rec + (static_cast<int64_t>(bh) * a.nch + c) * REC;
    rt = *reinterpret_cast<const fRT*>(rec + RT * tid);
    rg = *reinterpret_cast<const fRT*>(rec + REC_G + RT * tid);
#pragma unroll
    for (int i = 0; i < RX; ++i) rx[i] = rec[REC_DX + RX * tid + i];
    rbad = __float_as_int(rec[opaque(REC_BAD)]);  // a vector load, like the others
  };
  // The wait for the next chunk's loads, placed before this chunk's stores: after them it would
  // also wait for the stores (some are under a branch, so their number is not known).
  auto landed = [&]() {
    asm volatile("" : "+v"(rk.x), "+v"(rv.x), "+v"(rq.x), "+v"(rd.x), "+v"(rt), "+v"(rg), "+v"(rx[RX - 1]), "+v"(rbad));
  };
  auto commit = [&]() {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    const bool uk = rok && !((rbad >> ft) & 1);
    *reinterpret_cast<f32x4*>(U + (2 * ft) * LU + fd) = uk ? raw_f32(rk, IOC) : zero;
    *reinterpret_cast<f32x4*>(U + (2 * ft + 1) * LU + fd) = uk ? raw_f32(rv, IOC) : zero;
    *reinterpret_cast<f32x4*>(Q + ft * LU + fd) = rok ? raw_f32(rq, IOC) : zero;
    *reinterpret_cast<f32x4*>(dO + ft * LU + fd) = rok ? raw_f32(rd, a.do_dtype) : zero;
    *reinterpret_cast<fRT*>(Tt + (RT * tid) / R * TP + (RT * tid) % R) = rt;
    *reinterpret_cast<fRT*>(Gm + (RT * tid) / R * TP + (RT * tid) % R) = rg;
#pragma unroll
    for (int i = 0; i < RX; ++i) dX[(RX * tid + i) / C * XPP + (RX * tid + i) % C] = rx[i];
  };

  if (c0 < c1) fetch(c1 - 1);
  f32x4 psi[SS], lam[SS];
  init_states<D, MAIN>(a, bh, seg, 16 * wave + (lane & 15), lane >> 4, psi, lam);
  if (c0 < c1) commit();
  lds_barrier();

  for (int c = c1 - 1; c >= c0; --c) {
    fetch(c > c0 ? c - 1 : c);  // past the end the last one again, never committed
    const int ln = MAIN && D == 128 ? opaque(lane) : lane, l16 = ln & 15, g = ln >> 4, colj = 16 * wave + l16;
    // S1 = U^T Psi_e, dZ = U^T Lam_e + dX Q^T.  In the loops over tiles a step's LDS operands are
    // read while the step before runs (the fences keep the compiler from sinking the reads back).
    f32x4 s1[2], dz[2];
    {
      f32x4 p[2][2] = {}, l[2][2] = {};
      f32x4 a0 = lds4(U + l16 * LU + 4 * g), a1 = lds4(U + (16 + l16) * LU + 4 * g), n0 = a0, n1 = a1;
#pragma unroll
      for (int S = 0; S < SS; ++S) {
        if (S + 1 < SS) {
          n0 = lds4(U + l16 * LU + 16 * (S + 1) + 4 * g);
          n1 = lds4(U + (16 + l16) * LU + 16 * (S + 1) + 4 * g);
        }
        __builtin_amdgcn_sched_barrier(0);
        p[S & 1][0] = dot4<false>(a0, psi[S], p[S & 1][0]);
        p[S & 1][1] = dot4<false>(a1, psi[S], p[S & 1][1]);
        l[S & 1][0] = dot4<LP>(a0, lam[S], l[S & 1][0]);
        l[S & 1][1] = dot4<LP>(a1, lam[S], l[S & 1][1]);
        __builtin_amdgcn_sched_barrier(0);
        a0 = n0;
        a1 = n1;
      }
      s1[0] = p[0][0] + p[1][0];
      s1[1] = p[0][1] + p[1][1];
      dz[0] = l[0][0] + l[1][0];
      dz[1] = l[0][1] + l[1][1];
    }
    const f32x4 qc = col4(Q + 4 * g * LU + colj, LU);  // Q^T's column: tokens 4 g + r
    dz[0] = dot4<LP>(lds4(dX + l16 * XPP + 4 * g), qc, dz[0]);
    dz[1] = dot4<LP>(lds4(dX + (16 + l16) * XPP + 4 * g), qc, dz[1]);
    // Wm = T~^T S1, dW = T~^T dZ; MAIN: W = U^T Psi_s = S1 + G Wm, Z = T~ W
    f32x4 wm[2] = {}, dw[2] = {}, w[2], z[2] = {};
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        const f32x4 tv = col4(Tt + (16 * kt + 4 * g) * TP + 16 * mt + l16, TP);
        wm[mt] = dot4<false>(tv, s1[kt], wm[mt]);
        dw[mt] = dot4<LP>(tv, dz[kt], dw[mt]);
      }
    if constexpr (MAIN) {
      w[0] = s1[0];
      w[1] = s1[1];
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
          w[mt] = dot4<false>(lds4(Gm + (16 * mt + l16) * TP + 16 * kt + 4 * g), wm[kt], w[mt]);
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
          z[mt] = dot4<LP>(lds4(Tt + (16 * mt + l16) * TP + 16 * kt + 4 * g), w[kt], z[mt]);
    }
    // per tile of 16 rows: Psi_s = Psi_e + U Wm, Lam_s = Lam_e + dO Q^T + U dW, and the second
    // term of dQ; Lam_e goes to LDS first
    f32x4 dq[2] = {};
    struct Rows { f32x4 u0, u1, dv, dr; };
    auto rows = [&](int S) {
      Rows x;
      x.u0 = col4(U + 4 * g * LU + 16 * S + l16, LU);
      x.u1 = col4(U + (16 + 4 * g) * LU + 16 * S + l16, LU);
      x.dv = col4(dO + 4 * g * LU + 16 * S + l16, LU);
      if constexpr (MAIN) x.dr = lds4(dO + l16 * LU + 16 * S + 4 * g);
      return x;
    };
    Rows cur = rows(0), nxt = cur;
#pragma unroll
    for (int S = 0; S < SS; ++S) {
      if (S + 1 < SS) nxt = rows(S + 1);
      __builtin_amdgcn_sched_barrier(0);
      const f32x4 u0 = cur.u0, u1 = cur.u1, dv = cur.dv;
      if constexpr (MAIN && LP) {
        *reinterpret_cast<s16x4*>(LSb + colj * PJ + 16 * S + 4 * g) = pack4(lam[S]);
      } else if constexpr (MAIN) {
#pragma unroll
        for (int r = 0; r < 4; ++r) SB[(16 * S + 4 * g + r) * LU + colj] = lam[S][r];
      }
      f32x4 d = {};
      d = dot4<false>(u0, wm[0], d);
      d = dot4<false>(u1, wm[1], d);
      psi[S] += d;
      f32x4 e = {};
      e = dot4<false>(dv, qc, e);
      e = dot4<false>(u0, dw[0], e);
      e = dot4<false>(u1, dw[1], e);
      lam[S] += e;
      if constexpr (MAIN) {
        if constexpr (LP) *reinterpret_cast<s16x4*>(PSb + colj * PJ + 16 * S + 4 * g) = pack4(psi[S]);
        dq[S & 1] = dot4<LP>(psi[S], cur.dr, dq[S & 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
      cur = nxt;
    }
    if constexpr (MAIN) {
      // dQ = Z^T dX + Psi_s^T dO: rows = this wave's columns 16 wave + 4 g + r, lane = token
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
        dq[kt] = dot4<LP>(z[kt], col4(dX + (16 * kt + 4 * g) * XPP + l16, XPP), dq[kt]);
      const f32x4 y = dq[0] + dq[1];
      landed();
      const int t = c * C + l16;
      if (t < T) {
        IO* dst = static_cast<IO*>(a.dq) + tok(t) * D + 16 * wave + 4 * g;
        const float yv[4] = {y[0], y[1], y[2], y[3]};
        store_row<IO, 4>(dst, yv);
      }
      f32x4 du[2] = {}, du2[2] = {}, dt = {};
      float* pp = a.part + (static_cast<int64_t>(bh) * a.nch + c) * PartC<D>::size;
      const f32x4 doc = col4(dO + 4 * g * LU + colj, LU);  // dO^T's column (row colj of dO)
      const int half = wave & 1, kp = wave >> 1;  // X: 16 rank rows, columns 32 kp .. + 31
      auto store_x = [&](f32x4 x) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int rho = 16 * half + 4 * g + r;
          XP[(kp * R + rho) * XPP + l16] = (rho >> 1) <= l16 ? x[r] : 0.f;
        }
      };
      auto store_dt = [&](f32x4 x) {  // tile (wave >> 1, wave & 1) of dT~
#pragma unroll
        for (int r = 0; r < 4; ++r) pp[(16 * (wave >> 1) + 4 * g + r) * R + 16 * (wave & 1) + l16] = x[r];
      };
      if constexpr (LP) {
#pragma unroll
        for (int mt = 0; mt < 2; ++mt) {
          *reinterpret_cast<s16x4*>(Zb + colj * PZ + 16 * mt + 4 * g) = pack4(z[mt]);
          *reinterpret_cast<s16x4*>(dWb + colj * PZ + 16 * mt + 4 * g) = pack4(dw[mt]);
          *reinterpret_cast<s16x4*>(dZb + colj * PZ + 16 * mt + 4 * g) = pack4(dz[mt]);
          *reinterpret_cast<s16x4*>(Wb + colj * PZ + 16 * mt + 4 * g) = pack4(w[mt]);
        }
        lds_barrier();
        // lane n of a 16-lane group receives rows k0 .. k0 + 3 (columns of the state) of column
        // n0 + n (a state or rank row) from lanes addressing row k0 + n / 4, columns n0 + 4 (n % 4)
        typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
        auto tr = [&](const uint16_t* m, int ld, int k0, int n0) {
          const uint16_t* p = m + (k0 + 4 * g + (l16 >> 2)) * ld + n0 + 4 * (l16 & 3);
          return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p));
        };
        struct Ops { s16x4 al, ap, z0, z1, w0, w1; };
        auto ops = [&](int kb) {
          return Ops{tr(LSb, PJ, 16 * kb, 16 * wave), tr(PSb, PJ, 16 * kb, 16 * wave),
                     tr(Zb, PZ, 16 * kb, 0), tr(Zb, PZ, 16 * kb, 16),
                     tr(dWb, PZ, 16 * kb, 0), tr(dWb, PZ, 16 * kb, 16)};
        };
        Ops oc = ops(0), on = oc;
#pragma unroll
        for (int kb = 0; kb < SS; ++kb) {
          if (kb + 1 < SS) on = ops(kb + 1);
          __builtin_amdgcn_sched_barrier(0);
          du[0] = mma_bf16(oc.al, oc.z0, du[0]);
          du[1] = mma_bf16(oc.al, oc.z1, du[1]);
          du2[0] = mma_bf16(oc.ap, oc.w0, du2[0]);
          du2[1] = mma_bf16(oc.ap, oc.w1, du2[1]);
          __builtin_amdgcn_sched_barrier(0);
          oc = on;
        }
        f32x4 x = {};
#pragma unroll
        for (int s = 0; s < 2; ++s)
          x = mma_bf16(tr(Zb, PZ, 32 * kp + 16 * s, 16 * half),
                       pack4(lds4(Q + l16 * LU + 32 * kp + 16 * s + 4 * g)), x);
        store_x(x);
        if (wave < 4) {
#pragma unroll
          for (int kb = 0; kb < SS; ++kb)
            dt = mma_bf16(tr(dZb, PZ, 16 * kb, 16 * (wave >> 1)), tr(Wb, PZ, 16 * kb, 16 * (wave & 1)), dt);
          store_dt(dt);
        }
      } else {
        auto rows32 = [&](float* m, const f32x4 (&x)[2]) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            m[(4 * g + r) * LU + colj] = x[0][r];
            m[(16 + 4 * g + r) * LU + colj] = x[1][r];
          }
        };
        auto outer = [&](f32x4 (&acc)[2]) {  // acc = rows 16 wave .. of SB times ZB^T
          f32x4 p[2][2] = {};
#pragma unroll
          for (int kb = 0; kb < SS; ++kb) {
            const f32x4 al = lds4(SB + colj * LU + 16 * kb + 4 * g);
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
              p[kb & 1][nt] = dot4<false>(al, lds4(ZB + (16 * nt + l16) * LU + 16 * kb + 4 * g), p[kb & 1][nt]);
          }
          acc[0] = p[0][0] + p[1][0];
          acc[1] = p[0][1] + p[1][1];
        };
        rows32(ZB, z);
        lds_barrier();
        outer(du);  // Lam_e Z^T
        f32x4 x = {};
#pragma unroll
        for (int s = 0; s < 2; ++s)
          x = dot4<false>(lds4(ZB + (16 * half + l16) * LU + 32 * kp + 16 * s + 4 * g),
                          lds4(Q + l16 * LU + 32 * kp + 16 * s + 4 * g), x);
        store_x(x);
        lds_barrier();
#pragma unroll
        for (int S = 0; S < SS; ++S)
#pragma unroll
          for (int r = 0; r < 4; ++r) SB[(16 * S + 4 * g + r) * LU + colj] = psi[S][r];
        rows32(ZB, dw);
        lds_barrier();
        outer(du2);  // Psi_s dW^T
        lds_barrier();
        rows32(SB, dz);
        rows32(SB + R * LU, w);
        lds_barrier();
        if (wave < 4) {
          f32x4 p = {};
#pragma unroll
          for (int kb = 0; kb < SS; ++kb) {
            const f32x4 al = lds4(SB + (16 * (wave >> 1) + l16) * LU + 16 * kb + 4 * g);
            const f32x4 bl = lds4(SB + (R + 16 * (wave & 1) + l16) * LU + 16 * kb + 4 * g);
            if (kb & 1) p = dot4<false>(al, bl, p);
            else dt = dot4<false>(al, bl, dt);
          }
          store_dt(dt + p);
        }
      }
      lds_barrier();  // X visible; the chunk's inputs and the stashes are free
      // dU += dO X^T, stored transposed: four consecutive features of rank row 16 nt + l16
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        f32x4 x = lds4(XP + (16 * nt + l16) * XPP + 4 * g);
#pragma unroll
        for (int i = 1; i < KP; ++i) x += lds4(XP + (i * R + 16 * nt + l16) * XPP + 4 * g);
        f32x4 e = {};
        e = dot4<LP>(doc, x, e);
        *reinterpret_cast<f32x4*>(pp + R * R + (16 * nt + l16) * D + 16 * wave + 4 * g) = (du[nt] + du2[nt]) + e;
      }
    } else {
      lds_barrier();
    }
    if (c > c0) commit();
    lds_barrier();
  }
  const int ln = MAIN && D == 128 ? opaque(lane) : lane;
  store_states<D, MAIN>(a, bh, seg, 16 * wave + (ln & 15), ln >> 4, psi, lam);
}

// The pass for bf16 inputs and a bf16 output gradient.  U, Q and dO are then bf16 numbers exactly,
// so the products that carry the states run on the bf16 matrix cores without losing anything: the
// fp32 operand (Psi, Wm, dW) is split in three bf16 parts, which hold all its 24 bits, and the three
// products with the exact bf16 operand are exact and accumulated in fp32 (v_mfma_f32_16x16x32_bf16:
// 3 x 16 cycles for 32 k against 8 x 32 on v_mfma_f32_16x16x4_f32); dO Q^T is one exact product.  The
// inputs stay bf16 in LDS: rows are read 8 bytes at a time, columns by ds_read_b64_tr_b16.
// No accumulator passes from a 16x16x32 to a 16x16x16 product.  The one build that had such a chain
// (dZ's two products, adjacent in one tile) gave a wrong dZ in that tile, as if the second had read the
// sum before the first had written it; why is not known, and the assembly of every kernel of the
// library has no other chain between products of different shapes.  So the sums of 16x16x32 products
// have a type of their own (Sum32), which a 16x16x16 product does not take: they leave it through a
// VALU addition or element by element.
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef short s16x8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ s16x8 cat(s16x4 a, s16x4 b) {
  return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}
struct Sum32 {
  f32x4 v;
  __device__ __forceinline__ float operator[](int r) const { return v[r]; }
};
__device__ __forceinline__ f32x4 operator+(Sum32 a, Sum32 b) { return a.v + b.v; }
__device__ __forceinline__ f32x4 operator+(Sum32 a, f32x4 b) { return a.v + b; }
__device__ __forceinline__ f32x4 operator+(f32x4 a, Sum32 b) { return a + b.v; }
__device__ __forceinline__ Sum32 mma32(s16x8 a, s16x8 b, Sum32 c) {
  return Sum32{__builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c.v, 0, 0, 0)};
}
__device__ __forceinline__ f32x4 unpack4(s16x4 x) {
  const uint2 w = __builtin_bit_cast(uint2, x);
  return f32x4{__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xffff0000u),
               __uint_as_float(w.y << 16), __uint_as_float(w.y & 0xffff0000u)};
}
// x0, x1 (k-slots 0-3 and 4-7 of a lane) as hi + mid + lo
struct Split8 { s16x8 h, m, l; };
__device__ __forceinline__ Split8 split3(f32x4 x0, f32x4 x1) {
  const s16x4 h0 = pack4(x0), h1 = pack4(x1);
  const f32x4 r0 = x0 - unpack4(h0), r1 = x1 - unpack4(h1);
  const s16x4 m0 = pack4(r0), m1 = pack4(r1);
  return Split8{cat(h0, h1), cat(m0, m1), cat(pack4(r0 - unpack4(m0)), pack4(r1 - unpack4(m1)))};
}
// 16-lane group g, lane n: rows k0 + 4 g .. + 3 of column n0 + n (lanes address row n / 4, columns
// 4 (n % 4) ..)
__device__ __forceinline__ s16x4 lds_tr(const uint16_t* m, int ld, int k0, int n0, int l16, int g) {
  const uint16_t* p = m + (k0 + 4 * g + (l16 >> 2)) * ld + n0 + 4 * (l16 & 3);
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p));
}
__device__ __forceinline__ s16x4 ldsb4(const uint16_t* p) { return *reinterpret_cast<const s16x4*>(p); }

template <int D, bool MAIN>
__global__ __launch_bounds__(4 * D) void bwdc_pass16_kernel(Args a) {
  constexpr int NW = D / 16, NTC = 4 * D, SS = D / 16, KP = NW / 2;
  constexpr int TP = 36, XPP = 20, PB = D + 8, PZ = R + 4;  // pitches (elements)
  __shared__ __attribute__((aligned(16))) uint16_t U[R * PB], Q[C * PB], dO[C * PB];  // token rows
  __shared__ __attribute__((aligned(16))) float Tt[R * TP], Gm[MAIN ? R * TP : 4], dX[R * XPP];
  __shared__ __attribute__((aligned(16))) float XP[MAIN ? KP * R * XPP : 4];
  // column-major copies for the products over the columns (one 8-byte write per lane and tile)
  __shared__ __attribute__((aligned(16))) uint16_t LSb[MAIN ? D * PB : 8], PSb[MAIN ? D * PB : 8];
  __shared__ __attribute__((aligned(16))) uint16_t Zb[MAIN ? D * PZ : 8], dWb[MAIN ? D * PZ : 8],
      dZb[MAIN ? D * PZ : 8], Wb[MAIN ? D * PZ : 8];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: scalar addresses and branches
  const int bh = blockIdx.x, seg = MAIN ? blockIdx.y : blockIdx.y + 1, b = bh / a.H, h = bh - b * a.H;
  const int T = a.T;
  const int c0 = seg * a.seg_chunks, c1 = min(a.nch, c0 + a.seg_chunks);
  constexpr int RT = R * R / NTC, RX = R * C / NTC;
  typedef float fRT __attribute__((ext_vector_type(RT)));
  const int ft = tid / (D / 4), fd = 4 * (tid % (D / 4));
  uint2 rk, rv, rq, rd;
  fRT rt, rg;
  float rx[RX];
  int rbad = 0;
  bool rok = false;
  auto tok = [&](int t) { return (static_cast<int64_t>(b) * T + t) * a.H + h; };
  auto row8 = [&](const void* p, int64_t o) {
    return *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(p) + o);
  };
  auto fetch = [&](int c) {
    const int t = c * C + ft;
    rok = t < T;
    const int64_t o = tok(rok ? t : 0) * D + fd;
    rk = row8(a.k, o);
    rv = row8(a.v, o);
    rq = row8(a.q, o);
    rd = row8(a.dout, o);
    const float* rec = a.rec + (static_cast<int64_t>(bh) * a.nch + c) * REC;
    rt = *reinterpret_cast<const fRT*>(rec + RT * tid);
    if (MAIN) rg = *reinterpret_cast<const fRT*>(rec + REC_G + RT * tid);
#pragma unroll
    for (int i = 0; i < RX; ++i) rx[i] = rec[REC_DX + RX * tid + i];
    rbad = __float_as_int(rec[opaque(REC_BAD)]);  // a vector load, like the others
  };
  // The wait for the next chunk's loads, placed before this chunk's stores: after them it would
  // also wait for the stores (some are under a branch, so their number is not known).
  auto landed = [&]() {
    asm volatile("" : "+v"(rk.x), "+v"(rv.x), "+v"(rq.x), "+v"(rd.x), "+v"(rt), "+v"(rg), "+v"(rx[RX - 1]), "+v"(rbad));
  };
  auto commit = [&]() {
    const uint2 zero = make_uint2(0u, 0u);
    const bool uk = rok && !((rbad >> ft) & 1);
    *reinterpret_cast<uint2*>(U + (2 * ft) * PB + fd) = uk ? rk : zero;
    *reinterpret_cast<uint2*>(U + (2 * ft + 1) * PB + fd) = uk ? rv : zero;
    *reinterpret_cast<uint2*>(Q + ft * PB + fd) = rok ? rq : zero;
    *reinterpret_cast<uint2*>(dO + ft * PB + fd) = rok ? rd : zero;
    *reinterpret_cast<fRT*>(Tt + (RT * tid) / R * TP + (RT * tid) % R) = rt;
    if (MAIN) *reinterpret_cast<fRT*>(Gm + (RT * tid) / R * TP + (RT * tid) % R) = rg;
#pragma unroll
    for (int i = 0; i < RX; ++i) dX[(RX * tid + i) / C * XPP + (RX * tid + i) % C] = rx[i];
  };

  if (c0 < c1) fetch(c1 - 1);
  f32x4 psi[SS], lam[SS];
  init_states<D, MAIN>(a, bh, seg, 16 * wave + (lane & 15), lane >> 4, psi, lam);
  if (c0 < c1) commit();
  lds_barrier();

  for (int c = c1 - 1; c >= c0; --c) {
    fetch(c > c0 ? c - 1 : c);  // past the end the last one again, never committed
    const int ln = MAIN && D == 128 ? opaque(lane) : lane, l16 = ln & 15, g = ln >> 4, colj = 16 * wave + l16;
    // S1 = U^T Psi_e (exact parts), dZ = U^T Lam_e + dX Q^T; two tiles (32 rows) a step
    f32x4 s1[2], dz[2];
    Sum32 ul[2] = {};
    {
      Sum32 ph[2] = {}, pl[2] = {};
      auto ua = [&](int half, int s) {
        const uint16_t* p = U + (16 * half + l16) * PB + 32 * s + 4 * g;
        return cat(ldsb4(p), ldsb4(p + 16));
      };
      s16x8 a0 = ua(0, 0), a1 = ua(1, 0), n0 = a0, n1 = a1;
#pragma unroll
      for (int s = 0; s < SS / 2; ++s) {
        if (s + 1 < SS / 2) {
          n0 = ua(0, s + 1);
          n1 = ua(1, s + 1);
        }
        const Split8 x = split3(psi[2 * s], psi[2 * s + 1]);
        const s16x8 y = cat(pack4(lam[2 * s]), pack4(lam[2 * s + 1]));
        __builtin_amdgcn_sched_barrier(0);
        pl[0] = mma32(a0, x.l, pl[0]);
        pl[1] = mma32(a1, x.l, pl[1]);
        ph[0] = mma32(a0, x.h, ph[0]);
        ph[1] = mma32(a1, x.h, ph[1]);
        ul[0] = mma32(a0, y, ul[0]);
        ul[1] = mma32(a1, y, ul[1]);
        pl[0] = mma32(a0, x.m, pl[0]);
        pl[1] = mma32(a1, x.m, pl[1]);
        __builtin_amdgcn_sched_barrier(0);
        a0 = n0;
        a1 = n1;
      }
      s1[0] = ph[0] + pl[0];
      s1[1] = ph[1] + pl[1];
    }
    const s16x4 qc = lds_tr(Q, PB, 0, 16 * wave, l16, g);  // tokens 4 g + r of column colj
    const f32x4 none = {0.f, 0.f, 0.f, 0.f};
    dz[0] = ul[0] + mma_bf16(pack4(lds4(dX + l16 * XPP + 4 * g)), qc, none);
    dz[1] = ul[1] + mma_bf16(pack4(lds4(dX + (16 + l16) * XPP + 4 * g)), qc, none);
    // Wm = T~^T S1, dW = T~^T dZ; MAIN: W = U^T Psi_s = S1 + G Wm, Z = T~ W
    f32x4 wm[2] = {}, dw[2] = {}, w[2], z[2] = {};
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        const f32x4 tv = col4(Tt + (16 * kt + 4 * g) * TP + 16 * mt + l16, TP);
        wm[mt] = dot4<false>(tv, s1[kt], wm[mt]);
        dw[mt] = dot4<true>(tv, dz[kt], dw[mt]);
      }
    if constexpr (MAIN) {
      w[0] = s1[0];
      w[1] = s1[1];
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
          w[mt] = dot4<false>(lds4(Gm + (16 * mt + l16) * TP + 16 * kt + 4 * g), wm[kt], w[mt]);
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
          z[mt] = dot4<true>(lds4(Tt + (16 * mt + l16) * TP + 16 * kt + 4 * g), w[kt], z[mt]);
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        *reinterpret_cast<s16x4*>(Zb + colj * PZ + 16 * mt + 4 * g) = pack4(z[mt]);
        *reinterpret_cast<s16x4*>(dWb + colj * PZ + 16 * mt + 4 * g) = pack4(dw[mt]);
        *reinterpret_cast<s16x4*>(dZb + colj * PZ + 16 * mt + 4 * g) = pack4(dz[mt]);
        *reinterpret_cast<s16x4*>(Wb + colj * PZ + 16 * mt + 4 * g) = pack4(w[mt]);
      }
    }
    // per tile of 16 rows: Psi_s = Psi_e + U Wm, Lam_s = Lam_e + dO Q^T + U dW, and the second
    // term of dQ; Lam_e goes to LDS first
    const Split8 xw = split3(wm[0], wm[1]), xd = split3(dw[0], dw[1]);
    f32x4 dq[2] = {};
    struct Rows { s16x8 u; s16x4 dv, dr; };
    auto rows = [&](int S) {
      Rows x;
      x.u = cat(lds_tr(U, PB, 0, 16 * S, l16, g), lds_tr(U, PB, 16, 16 * S, l16, g));
      x.dv = lds_tr(dO, PB, 0, 16 * S, l16, g);
      if constexpr (MAIN) x.dr = ldsb4(dO + l16 * PB + 16 * S + 4 * g);
      return x;
    };
    Rows cur = rows(0), nxt = cur;
#pragma unroll
    for (int S = 0; S < SS; ++S) {
      if (S + 1 < SS) nxt = rows(S + 1);
      if constexpr (MAIN) *reinterpret_cast<s16x4*>(LSb + colj * PB + 16 * S + 4 * g) = pack4(lam[S]);
      __builtin_amdgcn_sched_barrier(0);
      Sum32 d = {}, e = {};
      const f32x4 oq = mma_bf16(cur.dv, qc, none);
      d = mma32(cur.u, xw.l, d);
      e = mma32(cur.u, xd.l, e);
      d = mma32(cur.u, xw.m, d);
      e = mma32(cur.u, xd.m, e);
      d = mma32(cur.u, xw.h, d);
      e = mma32(cur.u, xd.h, e);
      psi[S] = psi[S] + d;
      lam[S] += e + oq;
      if constexpr (MAIN) {
        const s16x4 ps = pack4(psi[S]);
        *reinterpret_cast<s16x4*>(PSb + colj * PB + 16 * S + 4 * g) = ps;
        dq[S & 1] = mma_bf16(ps, cur.dr, dq[S & 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
      cur = nxt;
    }
    if constexpr (MAIN) {
      // dQ = Z^T dX + Psi_s^T dO: rows = this wave's columns 16 wave + 4 g + r, lane = token
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
        dq[kt] = dot4<true>(z[kt], col4(dX + (16 * kt + 4 * g) * XPP + l16, XPP), dq[kt]);
      const f32x4 y = dq[0] + dq[1];
      landed();
      const int t = c * C + l16;
      if (t < T) {
        const float yv[4] = {y[0], y[1], y[2], y[3]};
        store_row<bf16_t, 4>(static_cast<bf16_t*>(a.dq) + tok(t) * D + 16 * wave + 4 * g, yv);
      }
      float* pp = a.part + (static_cast<int64_t>(bh) * a.nch + c) * PartC<D>::size;
      const s16x4 doc = lds_tr(dO, PB, 0, 16 * wave, l16, g);  // dO^T's column colj
      const int half = wave & 1, kp = wave >> 1;               // X: 16 rank rows, columns 32 kp .. + 31
      lds_barrier();  // (1) the column copies visible
      Sum32 du[2] = {}, du2[2] = {}, dt = {}, x = {};
      struct Ops { s16x4 al, ap, z0, z1, w0, w1; };
      auto ops = [&](int kb) {
        return Ops{lds_tr(LSb, PB, 16 * kb, 16 * wave, l16, g), lds_tr(PSb, PB, 16 * kb, 16 * wave, l16, g),
                   lds_tr(Zb, PZ, 16 * kb, 0, l16, g), lds_tr(Zb, PZ, 16 * kb, 16, l16, g),
                   lds_tr(dWb, PZ, 16 * kb, 0, l16, g), lds_tr(dWb, PZ, 16 * kb, 16, l16, g)};
      };
      // dU = Lam_e Z^T + Psi_s dW^T, rows 16 wave .. + 15, two 16-column steps (32 k) at once
      Ops oa = ops(0), ob = ops(1), na = oa, nb = ob;
#pragma unroll
      for (int kb = 0; kb < SS; kb += 2) {
        if (kb + 2 < SS) {
          na = ops(kb + 2);
          nb = ops(kb + 3);
        }
        __builtin_amdgcn_sched_barrier(0);
        const s16x8 al = cat(oa.al, ob.al), ap = cat(oa.ap, ob.ap);
        du[0] = mma32(al, cat(oa.z0, ob.z0), du[0]);
        du[1] = mma32(al, cat(oa.z1, ob.z1), du[1]);
        du2[0] = mma32(ap, cat(oa.w0, ob.w0), du2[0]);
        du2[1] = mma32(ap, cat(oa.w1, ob.w1), du2[1]);
        __builtin_amdgcn_sched_barrier(0);
        oa = na;
        ob = nb;
      }
      {
        const uint16_t* qr = Q + l16 * PB + 32 * kp + 4 * g;
        x = mma32(cat(lds_tr(Zb, PZ, 32 * kp, 16 * half, l16, g), lds_tr(Zb, PZ, 32 * kp + 16, 16 * half, l16, g)),
                  cat(ldsb4(qr), ldsb4(qr + 16)), x);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int rho = 16 * half + 4 * g + r;
        XP[(kp * R + rho) * XPP + l16] = (rho >> 1) <= l16 ? x[r] : 0.f;
      }
      if (wave < 4) {  // tile (wave >> 1, wave & 1) of dT~ = dZ W^T
        const int m0 = 16 * (wave >> 1), n0 = 16 * (wave & 1);
#pragma unroll
        for (int kb = 0; kb < SS; kb += 2)
          dt = mma32(cat(lds_tr(dZb, PZ, 16 * kb, m0, l16, g), lds_tr(dZb, PZ, 16 * kb + 16, m0, l16, g)),
                     cat(lds_tr(Wb, PZ, 16 * kb, n0, l16, g), lds_tr(Wb, PZ, 16 * kb + 16, n0, l16, g)), dt);
#pragma unroll
        for (int r = 0; r < 4; ++r) pp[(m0 + 4 * g + r) * R + n0 + l16] = dt[r];
      }
      lds_barrier();  // (2) X visible; the chunk's inputs and the copies are free
      // dU += dO X^T, stored transposed: four consecutive features of rank row 16 nt + l16
#pragma unroll
      for (int nt = 0; nt < 2; ++nt) {
        f32x4 xs = lds4(XP + (16 * nt + l16) * XPP + 4 * g);
#pragma unroll
        for (int i = 1; i < KP; ++i) xs += lds4(XP + (i * R + 16 * nt + l16) * XPP + 4 * g);
        const f32x4 e = mma_bf16(doc, pack4(xs), none);
        *reinterpret_cast<f32x4*>(pp + R * R + (16 * nt + l16) * D + 16 * wave + 4 * g) = (du[nt] + du2[nt]) + e;
      }
    } else {
      lds_barrier();
    }
    if (c > c0) commit();
    lds_barrier();
  }
  const int ln = MAIN && D == 128 ? opaque(lane) : lane;
  store_states<D, MAIN>(a, bh, seg, 16 * wave + (ln & 15), ln >> 4, psi, lam);
}

// ---------------------------------------------------------------- end states of the segments
// 16 columns of Psi and Lam per workgroup, wave w the rows 16 w .. + 15: Y <- X_s Y (+ B_s) for
// s = S - 1 .. 1, the result being segment s - 1's end.  The map's rows come from global memory in
// the operand layout, two segments ahead (its 1 us of products does not cover the latency); the
// columns pass through LDS (transposed), one barrier per segment.  One load of a map serves both
// states (as two workgroups 38 us at B4 T2048 H8 D128, so 34).
template <int D>
__global__ __launch_bounds__(4 * D) void bwdc_carry_kernel(const float* __restrict__ psi_T,
                                                           const float* __restrict__ dpsi_T,
                                                           const float* __restrict__ xmap,
                                                           const float* __restrict__ bmap,
                                                           float* __restrict__ epsi,
                                                           float* __restrict__ elam, int BH, int nf) {
  constexpr int SS = D / 16, LU = D + 4;
  __shared__ __attribute__((aligned(16))) float Yp[2][16 * LU], Yl[2][16 * LU];  // [column][row]
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int bh = blockIdx.x, j0 = 16 * blockIdx.y;
  const int64_t DD = static_cast<int64_t>(D) * D;
  for (int e = tid; e < 16 * D; e += 4 * D) {
    const int64_t o = bh * DD + (e / 16) * D + j0 + e % 16;
    Yp[0][(e % 16) * LU + e / 16] = psi_T[o];
    Yl[0][(e % 16) * LU + e / 16] = dpsi_T ? dpsi_T[o] : 0.f;
  }
  struct Map { f32x4 x[SS], b; };
  auto fetch = [&](Map& m, int f) {
    const int64_t o = (static_cast<int64_t>(max(f, 0)) * BH + bh) * DD;
#pragma unroll
    for (int S = 0; S < SS; ++S)
      m.x[S] = *reinterpret_cast<const f32x4*>(xmap + o + (16 * wave + l16) * D + 16 * S + 4 * g);
    m.b = col4(bmap + o + (16 * wave + 4 * g) * D + j0 + l16, D);
  };
  auto step = [&](Map& m, int f, int cur) {
    f32x4 y[2][2] = {};
#pragma unroll
    for (int S = 0; S < SS; ++S) {
      y[S & 1][0] = dot4<false>(m.x[S], lds4(&Yp[cur][l16 * LU + 16 * S + 4 * g]), y[S & 1][0]);
      y[S & 1][1] = dot4<false>(m.x[S], lds4(&Yl[cur][l16 * LU + 16 * S + 4 * g]), y[S & 1][1]);
    }
    const f32x4 p = y[0][0] + y[1][0], l = (y[0][1] + y[1][1]) + m.b;
    fetch(m, f - 2);
    *reinterpret_cast<f32x4*>(&Yp[cur ^ 1][l16 * LU + 16 * wave + 4 * g]) = p;
    *reinterpret_cast<f32x4*>(&Yl[cur ^ 1][l16 * LU + 16 * wave + 4 * g]) = l;
    const int64_t o = (static_cast<int64_t>(f) * BH + bh) * DD + (16 * wave + 4 * g) * D + j0 + l16;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      epsi[o + i * D] = p[i];
      elam[o + i * D] = l[i];
    }
    lds_barrier();
  };
  Map a, b;
  fetch(a, nf - 1);
  fetch(b, nf - 2);
  lds_barrier();
  for (int f = nf - 1; f >= 0; f -= 2) {
    step(a, f, 0);
    if (f > 0) step(b, f - 1, 1);
  }
}

// ---------------------------------------------------------------- per chunk: dT~ -> dk, dv, ddelta
template <typename IO, int D>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void bwdc_reduce_kernel(
    const IO* __restrict__ k, const IO* __restrict__ v, const void* __restrict__ delta,
    int delta_dtype, const float* __restrict__ tt, const float* __restrict__ part,
    IO* __restrict__ dk, IO* __restrict__ dv, void* __restrict__ ddelta, int T, int H) {
  constexpr int PS = PartC<D>::size;
  static_assert(R * R % NT == 0 && D * C % NT == 0 && 4 * C <= NT, "record and tokens split evenly");
  constexpr int NR = R * R / NT, NK = D * C / NT;
  // 40 KB of LDS (four workgroups per CU): U (row stride 37), tmp and A (row stride 33), and a
  // pool whose buffers are dead by the last product, which writes its R x D result over them.
  // The dU rows stay in registers.  dT and G share a buffer (G is stored once dT is
  // consumed), and so do dG and L (the new dG, written once dG is consumed).
  constexpr int LA = 33;
  constexpr int POOL = 3 * R * R + R * LA + 4 * C + C;
  static_assert(POOL >= R * D, "the last product's output fits the pool");
  __shared__ float U[D * L32], tmp[R * LA], pool[POOL];
  float* const dT = pool;           // then G
  float* const dA = pool + R * R;
  float* const dG = pool + 2 * R * R;  // then L
  float* const A = pool + 3 * R * R;
  float* const Mb = A + R * LA;
  float* const dl = Mb + 4 * C;
  float* const G = dT;
  float* const L = dG;
  float* const dU = pool;           // the last product's output, R x D
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int n = blockIdx.x, bh = blockIdx.y, b = bh / H, hd = bh % H;
  const int nch = gridDim.x;
  auto tok = [&](int tg) { return (static_cast<int64_t>(b) * T + tg) * H + hd; };
  // every global load of the workgroup is issued before the first wait: the main pass's dT~ and
  // dU (read once, with the nontemporal hint), the chunk record (A, G, M) and the chunk's k, v,
  // delta.  Thread (ft = tid / 16, fi = NK (tid % 16)) loads elements fi .. fi + NK - 1 of rows
  // 2 ft and 2 ft + 1 of dU (the elements of dk, dv it stores at the end) and four consecutive
  // dT~ elements.
  static_assert(R * R == 4 * NT, "four dT~ elements per thread");
  const int ft = tid >> 4, fi = NK * (tid & 15);
  const float* pp = part + (static_cast<int64_t>(bh) * nch + n) * PS;
  const RowRaw<float, 4> xt = load_raw_nt<float, 4>(pp + 4 * tid);
  const RowRaw<float, NK> xk = load_raw_nt<float, NK>(pp + R * R + (2 * ft) * D + fi);
  const RowRaw<float, NK> xv = load_raw_nt<float, NK>(pp + R * R + (2 * ft + 1) * D + fi);
  float ra[NR], rg[NR], rm = 0.f, rd = 0.f;
  int bad;  // tokens of the chunk that are the identity (non-finite Cayley factor): no gradient
  {
    const float* rec = tt + (static_cast<int64_t>(bh) * nch + n) * REC;
    bad = __float_as_int(rec[REC_BAD]);
#pragma unroll
    for (int u = 0; u < NR; ++u) {
      ra[u] = rec[REC_A + tid + NT * u];
      rg[u] = rec[REC_G + tid + NT * u];
    }
    if (tid < 4 * C) rm = rec[REC_M + tid];
  }
  // the same (token, features) split of the chunk's k, v rows: one 8- or 16-byte load each
  const int64_t fo = tok(n * C + ft < T ? n * C + ft : 0) * D + fi;
  const RowRaw<IO, NK> rk = load_raw<IO, NK>(k + fo), rv = load_raw<IO, NK>(v + fo);
  if (tid < C) {
    const int tg = n * C + tid;
    rd = tg < T ? load_scalar(delta, delta_dtype, tok(tg)) : 0.f;
  }
#pragma unroll
  for (int u = 0; u < NR; ++u) {
    const int e = tid + NT * u;
    A[(e / R) * LA + e % R] = ra[u];
  }
  if (tid < 4 * C) Mb[tid] = rm;
  if (tid < C) dl[tid] = rd;
  {
    const bool ok = n * C + ft < T && !((bad >> ft) & 1);
#pragma unroll
    for (int j = 0; j < NK; ++j) {
      U[(fi + j) * L32 + 2 * ft] = ok ? raw_elem<IO, NK>(rk, j) : 0.f;
      U[(fi + j) * L32 + 2 * ft + 1] = ok ? raw_elem<IO, NK>(rv, j) : 0.f;
    }
  }
  *reinterpret_cast<float4*>(dT + 4 * tid) =
      make_float4(raw_elem<float, 4>(xt, 0), raw_elem<float, 4>(xt, 1), raw_elem<float, 4>(xt, 2), raw_elem<float, 4>(xt, 3));
  __syncthreads();
  // B = blockdiag(M); dA = dT~ B^T (block structure: dA[r][2s + a] = sum_b dT[r][2s + b] M_s[a][b])
  for (int e = tid; e < R * R; e += NT) {
    const int r = e / R, c = e % R, s = c >> 1, a = c & 1;
    dA[e] = dT[r * R + 2 * s] * Mb[4 * s + 2 * a] + dT[r * R + 2 * s + 1] * Mb[4 * s + 2 * a + 1];
  }
  __syncthreads();
  // tmp = A^T dA; dB = A^T dT~ (its diagonal blocks used) into dG
  lgemm<R, R, R, true, false>(A, LA, dA, R, tmp, LA, wave, lane);
  lgemm<R, R, R, true, false>(A, LA, dT, R, dG, R, wave, lane);
  __syncthreads();
  // dL = tmp A^T  (into dA); G over dT, which is consumed
  lgemm<R, R, R, false, true>(tmp, LA, A, LA, dA, R, wave, lane);
#pragma unroll
  for (int u = 0; u < NR; ++u) G[tid + NT * u] = rg[u];
  __syncthreads();
  // dM_t = dB_tt + sum_{i<t} dL_ti G_ti^T; then the M chain; dG_ti = M_t^T dL_ti (i < t)
  if (tid < 4 * C) {
    const int t = tid >> 2, a = (tid >> 1) & 1, c = tid & 1;
    float y = dG[(2 * t + a) * R + 2 * t + c];
    for (int i = 0; i < t; ++i)
#pragma unroll
      for (int m = 0; m < 2; ++m) y = fmaf(dA[(2 * t + a) * R + 2 * i + m], G[(2 * t + c) * R + 2 * i + m], y);
    tmp[tid] = y;  // dM_t[a][c]
  }
  __syncthreads();
  for (int e = tid; e < R * R; e += NT) {  // dG off-diagonal blocks (lower), zero elsewhere
    const int r = e / R, c = e % R, t = r >> 1, i = c >> 1, a = r & 1;
    float y = 0.f;
    if (i < t)  // (M_t^T dL_ti)[a][cb] = sum_m M_t[m][a] dL_ti[m][cb]
      y = Mb[4 * t + a] * dA[(2 * t) * R + c] + Mb[4 * t + 2 + a] * dA[(2 * t + 1) * R + c];
    L[e] = y;  // the new dG, over dG (consumed above)
  }
  __syncthreads();
  if (tid < C) {  // M chain (vmi::cayley_coeffs) -> ddelta and the diagonal Gram entries
    const int t = tid;
    const float kk = G[(2 * t) * R + 2 * t], vv = G[(2 * t + 1) * R + 2 * t + 1], kv = G[(2 * t) * R + 2 * t + 1];
    const float d00 = tmp[4 * t], d01 = tmp[4 * t + 1], d10 = tmp[4 * t + 2], d11 = tmp[4 * t + 3];
    const float hh = (bad >> t) & 1 ? 0.f : 0.5f * dl[t], P = hh * hh;  // identity token: no chain
    const float graw = kk * vv - kv * kv, g = fmaxf(graw, 0.f);
    const float c = 2.f / (1.f + P * g);
    const float N00 = -P * vv, N01 = P * kv - hh, N10 = P * kv + hh, N11 = -P * kk;
    const float S = d00 * N00 + d01 * N01 + d10 * N10 + d11 * N11;
    float dh = c * (d01 * (2.f * hh * kv - 1.f) + d10 * (2.f * hh * kv + 1.f) - 2.f * hh * (d00 * vv + d11 * kk));
    float dvv = -c * P * d00, dkk = -c * P * d11, dkv = c * P * (d01 + d10);
    dh += S * (-c * c * hh * g);
    const float dg = graw > 0.f ? S * (-0.5f * c * c * P) : 0.f;
    dkk += dg * vv;
    dvv += dg * kk;
    dkv += -2.f * dg * kv;
    L[(2 * t) * R + 2 * t] += dkk;
    L[(2 * t + 1) * R + 2 * t + 1] += dvv;
    L[(2 * t) * R + 2 * t + 1] += dkv;
    const int tg = n * C + t;
    if (tg < T) {
      const float dd = (bad >> t) & 1 ? 0.f : 0.5f * dh;
      const int64_t o = tok(tg);
      if (delta_dtype == VMI_F32) static_cast<float*>(ddelta)[o] = dd;
      else if (delta_dtype == VMI_BF16) static_cast<uint16_t*>(ddelta)[o] = f32_to_bf16(dd);
      else static_cast<f16_t*>(ddelta)[o] = static_cast<f16_t>(dd);
    }
  }
  __syncthreads();
  for (int e = tid; e < R * R; e += NT) {  // symmetrise: dG + dG^T
    const int r = e / R, c = e % R;
    tmp[r * LA + c] = L[r * R + c] + L[c * R + r];
  }
  __syncthreads();
  // dU^T = the main pass's + (dG + dG^T) U^T (both transposed, [R][D]); the
  // product goes over the pool, whose buffers are all consumed
  lgemm<R, D, R, false, true>(tmp, LA, U, L32, dU, D, wave, lane);
  __syncthreads();
  if (n * C + ft < T) {  // the same (token, features) split: one 8- or 16-byte store per row
    const bool z = (bad >> ft) & 1;
    float yk[NK], yv[NK];
#pragma unroll
    for (int j = 0; j < NK; ++j) {
      yk[j] = z ? 0.f : raw_elem<float, NK>(xk, j) + dU[(2 * ft) * D + fi + j];
      yv[j] = z ? 0.f : raw_elem<float, NK>(xv, j) + dU[(2 * ft + 1) * D + fi + j];
    }
    store_row<IO, NK>(dk + fo, yk);
    store_row<IO, NK>(dv + fo, yv);
  }
}

// ---------------------------------------------------------------- host side
struct Plan {
  int nch, nseg, seg_chunks;
  int64_t rec, part, xmap, bmap, epsi, elam, total;  // offsets in floats
};

Plan plan(int64_t B, int64_t T, int64_t H, int64_t D) {
  Plan p;
  const int64_t BH = B * H;
  p.nch = static_cast<int>((T + C - 1) / C);
  p.nseg = 1;
  p.seg_chunks = p.nch;
  // One segment more costs every chunk a map iteration beside its main one, a carry product and
  // two launches, and pays while the chip is not full: one workgroup per CU at D = 128 (162 KB of
  // LDS), two at 64.  Costs in main iterations.  At least four chunks a segment: below that the
  // segments' maps outweigh the per-chunk buffers.
  const double cm = 0.55, carry = 0.5, fixed = 2.0;
  const int64_t room = D == 128 ? 256 : 512;
  double best = p.nch;
  const int64_t smax = BH > 0 ? std::min<int64_t>({64, p.nch / 4, room / BH}) : 1;
  for (int s = 2; s <= smax; ++s) {
    const int len = std::max(4, (p.nch + s - 1) / s), n = (p.nch + len - 1) / len;
    const double cost = len * (1.0 + cm) + carry * (n - 1) + fixed;
    if (n > 1 && cost < best) {
      best = cost;
      p.nseg = n;
      p.seg_chunks = len;
    }
  }
  const int64_t chunks = BH * p.nch, maps = static_cast<int64_t>(p.nseg - 1) * BH * D * D;
  p.rec = 0;
  p.part = p.rec + chunks * REC;
  p.xmap = p.part + chunks * (R * R + D * R);
  p.bmap = p.xmap + maps;
  p.epsi = p.bmap + maps;
  p.elam = p.epsi + maps;
  p.total = p.elam + maps;
  return p;
}

template <typename IO, int D>
hipError_t launch_d(const void* q, const void* k, const void* v, const void* delta,
                    int delta_dtype, const float* psi_T, const void* dout, int do_dtype,
                    const float* dpsi_T, void* dq, void* dk, void* dv, void* ddelta, float* dpsi0,
                    int B, int T, int H, void* ws, hipStream_t stream) {
  const Plan pl = plan(B, T, H, D);
  const int BH = B * H;
  float* w = static_cast<float*>(ws);
  const int64_t chunks = static_cast<int64_t>(BH) * pl.nch;
  hipLaunchKernelGGL((bwdc_prep_kernel<IO, D>), dim3(static_cast<unsigned>((chunks + PW - 1) / PW)),
                     dim3(64 * PW), 0, stream, static_cast<const IO*>(k), static_cast<const IO*>(v),
                     dout, do_dtype, delta, delta_dtype, w + pl.rec, T, H, pl.nch, chunks);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  Args a;
  a.q = q; a.k = k; a.v = v; a.dout = dout;
  a.do_dtype = do_dtype;
  a.rec = w + pl.rec;
  a.psi_T = psi_T;
  a.dpsi_T = dpsi_T;
  a.xmap = w + pl.xmap;
  a.bmap = w + pl.bmap;
  a.epsi = w + pl.epsi;
  a.elam = w + pl.elam;
  a.dq = dq;
  a.dpsi0 = dpsi0;
  a.part = w + pl.part;
  a.T = T; a.H = H; a.BH = BH;
  a.nch = pl.nch;
  a.seg_chunks = pl.seg_chunks;
  a.nseg = pl.nseg;
  const bool exact16 = std::is_same<IO, bf16_t>::value && do_dtype == VMI_BF16;
  if (pl.nseg > 1) {
    if (exact16)
      hipLaunchKernelGGL((bwdc_pass16_kernel<D, false>), dim3(BH, pl.nseg - 1), dim3(4 * D), 0, stream, a);
    else
      hipLaunchKernelGGL((bwdc_pass_kernel<IO, D, false>), dim3(BH, pl.nseg - 1), dim3(4 * D), 0, stream, a);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL((bwdc_carry_kernel<D>), dim3(BH, D / 16), dim3(4 * D), 0, stream, psi_T,
                       dpsi_T, a.xmap, a.bmap, w + pl.epsi, w + pl.elam, BH, pl.nseg - 1);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if (exact16)
    hipLaunchKernelGGL((bwdc_pass16_kernel<D, true>), dim3(BH, pl.nseg), dim3(4 * D), 0, stream, a);
  else
    hipLaunchKernelGGL((bwdc_pass_kernel<IO, D, true>), dim3(BH, pl.nseg), dim3(4 * D), 0, stream, a);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  hipLaunchKernelGGL((bwdc_reduce_kernel<IO, D>), dim3(pl.nch, BH), dim3(NT), 0, stream,
                     static_cast<const IO*>(k), static_cast<const IO*>(v), delta, delta_dtype,
                     a.rec, a.part, static_cast<IO*>(dk), static_cast<IO*>(dv), ddelta, T, H);
  return hipGetLastError();
}

template <typename IO>
hipError_t launch_io(const void* q, const void* k, const void* v, const void* delta,
                     int delta_dtype, const float* psi_T, const void* dout, int dout_dtype,
                     const float* dpsi_T, void* dq, void* dk, void* dv, void* ddelta,
                     float* dpsi0, int B, int T, int H, int D, void* ws, hipStream_t stream) {
  if (D == 64)
    return launch_d<IO, 64>(q, k, v, delta, delta_dtype, psi_T, dout, dout_dtype, dpsi_T, dq, dk,
                            dv, ddelta, dpsi0, B, T, H, ws, stream);
  return launch_d<IO, 128>(q, k, v, delta, delta_dtype, psi_T, dout, dout_dtype, dpsi_T, dq, dk, dv,
                           ddelta, dpsi0, B, T, H, ws, stream);
}

}  // namespace bwdc

size_t sssd_bwd_chunk_workspace_bytes(int64_t B, int64_t T, int64_t H, int64_t D) {
  return static_cast<size_t>(bwdc::plan(B, T, H, D).total) * sizeof(float);
}

hipError_t launch_sssd_bwd_chunk(const void* q, const void* k, const void* v, const void* delta,
                                 int io_dtype, int delta_dtype, const float* psi_T,
                                 const void* dout, int dout_dtype, const float* dpsi_T, void* dq,
                                 void* dk, void* dv, void* ddelta, float* dpsi0, int B, int T,
                                 int H, int D, void* ws, hipStream_t stream) {
  if (io_dtype == VMI_F32)
    return bwdc::launch_io<float>(q, k, v, delta, delta_dtype, psi_T, dout, dout_dtype, dpsi_T, dq,
                                  dk, dv, ddelta, dpsi0, B, T, H, D, ws, stream);
  if (io_dtype == VMI_BF16)
    return bwdc::launch_io<bf16_t>(q, k, v, delta, delta_dtype, psi_T, dout, dout_dtype, dpsi_T,
                                   dq, dk, dv, ddelta, dpsi0, B, T, H, D, ws, stream);
  return bwdc::launch_io<f16_t>(q, k, v, delta, delta_dtype, psi_T, dout, dout_dtype, dpsi_T, dq,
                                dk, dv, ddelta, dpsi0, B, T, H, D, ws, stream);
}

}  // namespace vmi
