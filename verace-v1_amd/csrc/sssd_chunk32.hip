// Chunked SSSD scan in fp32 (any I/O dtype, head_dim <= 128): the scan of fp32 inputs and of the
// head sizes and lengths that the 16-bit chunk scan (sssd_chunk.hip) does not take.
//
// The same chunk algebra as there (C = 16 tokens, U = [k_1 v_1 .. k_16 v_16], rank 32):
//   G = U^T U,  T~_t = M_t (E_t + sum_{i<t} G_ti T~_i)   (forward substitution, 2 rows a step)
//   W = U^T Psi_s,  Z = T~ W,  Psi_e = Psi_s + U Z,  O = Psi_s Q + U (mask o (Z Q))
// with every product on v_mfma_f32_16x16x4f32 (exact fp32 products, fp32 accumulation) and
// nothing rounded below fp32.
//
// Launches (S segments of the chunks, picked by plan()):
//   c32_prep_kernel   one wave per chunk: T~ and the accuracy flag -> workspace;
//   c32_pass_kernel<READOUT = false>  (S > 1) transforms of segments 0 .. S - 2 from the identity;
//   c32_carry_kernel  (S > 1) start_s = P_{s-1} start_{s-1};
//   c32_pass_kernel<READOUT = true>   every segment from its start state, with outputs;
//   sssd_seq_kernel   the flagged sequences again, token by token (its other workgroups exit).
//
// What bounds it: the fp32 matrix rate (157 TFLOP/s).  A wave owns 16 state columns as MFMA
// accumulators; an accumulator tile (lane = column, registers = 4 rows per 16-lane group) is
// already the B operand of the products that contract over the rows (W) or the rank (U Z), so the
// state never moves for the recurrence.  Only the readout contracts over the columns: Psi_s and Z
// pass through LDS once per chunk.  Two waves per SIMD at D = 128.
//
// Measured (fp32; pass C at D = 128 issues its products at about 65 % of the matrix rate):
//   B4 T2048 H8 D128: 272 us (pass C 130, pass A 88, carry 23, prep 20) against 13420 us for the
//   token-sequential kernel, which keeps one workgroup per (b, h) for all T tokens and pays a
//   barrier, two LDS round trips and a shuffle reduction per token (6.6 us);
//   B2 T128 H4 D64: 35 us against 401 us; bf16 B4 T2048 H8 D64: 111 us against 6640 us.
// Relative error against fp64 (output, state): 2.5e-7, 3.2e-7 at B4 T2048 H8 D128 (token by token
// 8.0e-7, 1.1e-6): the state is rounded once a chunk, not once a token.
#include <algorithm>

#include "vmi_common.h"
#include "vmi_dispatch.h"
#include "vmi_mfma.h"

namespace vmi {
namespace c32 {

constexpr int C = 16;     // tokens per chunk
constexpr int R = 32;     // rank rows of a chunk
constexpr int TTP = 36;   // T~ row pitch (floats): 16-byte rows, conflict-free 16-byte reads
constexpr int LX = 20;    // X row pitch: the four 16-lane groups of a write in distinct banks
constexpr int MAX_SEG = 64;
constexpr float kMaxSkew2 = 0.003f;  // largest ((delta / 2) |k| |v|)^2 of a token (c32_prep_kernel)

// Four consecutive elements of a row as they lie in memory.
template <typename IO> struct Raw4 { uint2 w; };
template <> struct Raw4<float> { float4 w; };

__device__ __forceinline__ float4 to_f4(const Raw4<float>& r) { return r.w; }
__device__ __forceinline__ float4 to_f4(const Raw4<bf16_t>& r) {
  return make_float4(bf16_to_f32(r.w.x & 0xffffu), bf16_to_f32(r.w.x >> 16),
                     bf16_to_f32(r.w.y & 0xffffu), bf16_to_f32(r.w.y >> 16));
}
__device__ __forceinline__ float4 to_f4(const Raw4<f16_t>& r) {
  const f16x4 h = __builtin_bit_cast(f16x4, r.w);
  return make_float4(static_cast<float>(h[0]), static_cast<float>(h[1]), static_cast<float>(h[2]),
                     static_cast<float>(h[3]));
}

// Elements d0 .. d0 + 3 of a row of D one by one, zeros past its end: for rows that are not
// aligned to four elements (else the four are one load).
template <typename IO>
__device__ __forceinline__ Raw4<IO> load4(const IO* row, int d0, int D) {
  Raw4<IO> r;
  auto word = [&](int j) {
    if constexpr (sizeof(IO) == 4) return d0 + j < D ? row[d0 + j] : 0.f;
    else return d0 + j < D ? static_cast<uint32_t>(__builtin_bit_cast(uint16_t, row[d0 + j])) : 0u;
  };
  if constexpr (sizeof(IO) == 4) r.w = make_float4(word(0), word(1), word(2), word(3));
  else r.w = make_uint2(word(0) | word(1) << 16, word(2) | word(3) << 16);
  return r;
}

__device__ __forceinline__ f32x4 mma(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float elem(const float4& x, int i) {
  return i == 0 ? x.x : i == 1 ? x.y : i == 2 ? x.z : x.w;
}
__device__ __forceinline__ float4 lds4(const float* p) { return *reinterpret_cast<const float4*>(p); }

// Sums over the state's rows or columns run in NCH accumulators added as a tree, which keeps the
// rounding error of a 128-term sum below that of the token-sequential kernel's tree of lanes.
template <int N, int M>
__device__ __forceinline__ f32x4 tree(const f32x4 (&p)[N][M], int m) {
  if constexpr (N == 4) return (p[0][m] + p[1][m]) + (p[2][m] + p[3][m]);
  else return p[0][m] + p[1][m];
}

// Orders LDS accesses only: the loads of the next chunk and the stores of the last one stay in
// flight across it.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xC07F);  // vmcnt(63) expcnt(7) lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// ------------------------------------------------------------------ T~ of every chunk
// One wave per chunk and no workgroup barrier.  The Gram matrix's operands come straight from
// global memory in the MFMA layout (lane l16 = rank row, group g: features 16 S + 4 g ..+ 3), so U
// needs no LDS; G passes through it once, to be read by rows in the substitution.
constexpr int PW = 4;  // waves (chunks) per workgroup

template <typename IO, int DP>
__global__ __launch_bounds__(64 * PW) void c32_prep_kernel(
    const IO* __restrict__ k, const IO* __restrict__ v, const void* __restrict__ delta,
    int delta_dtype, float* __restrict__ tt, uint32_t* __restrict__ flags, int T, int H, int D,
    int nch, int64_t total, bool vec) {
  __shared__ __attribute__((aligned(16))) float Gs[PW][R * TTP];
  __shared__ float4 Ms[PW][C];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
  const int64_t id = static_cast<int64_t>(blockIdx.x) * PW + wave;
  if (id >= total) return;  // whole waves; no barrier below
  const int bh = static_cast<int>(id / nch), n = static_cast<int>(id - static_cast<int64_t>(bh) * nch);
  const int b = bh / H, h = bh - b * H;
  float* G = Gs[wave];
  // rank row rho = l16 of each 16-row half: token rho / 2, k for even rho and v for odd
  const IO* src = (l16 & 1) ? v : k;
  const int t0 = n * C + (l16 >> 1), t1 = t0 + C / 2;
  const int64_t base = static_cast<int64_t>(b) * T * H + h;
  const IO* r0 = src + (base + static_cast<int64_t>(t0 < T ? t0 : 0) * H) * D;
  const IO* r1 = src + (base + static_cast<int64_t>(t1 < T ? t1 : 0) * H) * D;
  float dl = 0.f;
  if (lane < C && n * C + lane < T)
    dl = load_scalar(delta, delta_dtype, base + static_cast<int64_t>(n * C + lane) * H);
  constexpr int SS = DP / 16;
  Raw4<IO> x0[SS], x1[SS];
  if (vec) {  // every load issued (clamped) before the first wait
#pragma unroll
    for (int S = 0; S < SS; ++S) {
      const int d = 16 * S + 4 * g < D ? 16 * S + 4 * g : 0;
      x0[S].w = *reinterpret_cast<const decltype(x0[S].w)*>(r0 + d);
      x1[S].w = *reinterpret_cast<const decltype(x0[S].w)*>(r1 + d);
    }
  } else {
#pragma unroll
    for (int S = 0; S < SS; ++S) {
      x0[S] = load4(r0, 16 * S + 4 * g, D);
      x1[S] = load4(r1, 16 * S + 4 * g, D);
    }
  }
  f32x4 gp[2][3] = {};
#pragma unroll
  for (int S = 0; S < SS; ++S) {
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
    const bool in = 16 * S + 4 * g < D;
    const float4 a0 = in && t0 < T ? to_f4(x0[S]) : zero, a1 = in && t1 < T ? to_f4(x1[S]) : zero;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      gp[S & 1][0] = mma(elem(a0, r), elem(a0, r), gp[S & 1][0]);
      gp[S & 1][1] = mma(elem(a1, r), elem(a0, r), gp[S & 1][1]);
      gp[S & 1][2] = mma(elem(a1, r), elem(a1, r), gp[S & 1][2]);
    }
  }
  const f32x4 g00 = tree(gp, 0), g10 = tree(gp, 1), g11 = tree(gp, 2);
  // rows and columns below / left of the diagonal blocks are all the substitution reads
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    G[(4 * g + r) * TTP + l16] = g00[r];
    G[(16 + 4 * g + r) * TTP + l16] = g10[r];
    G[(16 + 4 * g + r) * TTP + 16 + l16] = g11[r];
  }
  __builtin_amdgcn_wave_barrier();
  bool out = false;
  if (lane < C) {
    const int t = lane;
    const float kk = G[(2 * t) * TTP + 2 * t], vv = G[(2 * t + 1) * TTP + 2 * t + 1];
    const float kv = G[(2 * t + 1) * TTP + 2 * t];
    bool ok;
    const cayley2 m = cayley_guarded(dl, kk, vv, kv, ok);
    Ms[wave][t] = make_float4(m.m00, m.m01, m.m10, m.m11);
    // Rounding of T~.  Its terms have the size of s = (delta / 2) |k| |v| (the rotation's m is
    // s sin(angle(k, v)), much smaller where k and v are nearly parallel) and cancel over the chunk's
    // substitution.  In fp32 against fp64 (adversarial tokens: few distinct near-parallel pairs
    // repeated), the state's error over the token-sequential scan's is at most 1.5 at s^2 <= 0.003,
    // 2.3 at 0.005, 4 at 0.01, 20 at 0.06, and without a bound on s the state is lost (0.4 relative
    // at |k| = |v| = 30, angle 0.003, m = 0.135).  Unit k, v and delta <= 0.1 give s^2 <= 0.0025.
    const float s = 0.5f * dl;
    out = !ok || (s * kk) * (s * vv) > kMaxSkew2;
  }
  const uint64_t any = __ballot(out);
  __builtin_amdgcn_wave_barrier();
  // lane (a, c) = (lane >> 5, lane & 31) keeps column c of T~ in registers and forms row 2t + a of
  // E_t + sum_{i<t} G_ti T~_i; the halves exchange their rows (v_permlane32_swap) and each takes
  // M_t's row a of the pair
  const int c = lane & 31, a = lane >> 5;
  float col[R];
#pragma unroll
  for (int t = 0; t < C; ++t) {
    const float* gr = G + (2 * t + a) * TTP;
    float s0 = (2 * t + a) == c ? 1.f : 0.f, s1 = 0.f;
#pragma unroll
    for (int m = 0; m < R; m += 4) {
      if (m + 4 > 2 * t) continue;
      const float4 g4 = lds4(gr + m);
      s0 = fmaf(g4.x, col[m], s0);
      s1 = fmaf(g4.y, col[m + 1], s1);
      s0 = fmaf(g4.z, col[m + 2], s0);
      s1 = fmaf(g4.w, col[m + 3], s1);
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
    col[2 * t] = fmaf(m.x, rk, m.y * rv);
    col[2 * t + 1] = fmaf(m.z, rk, m.w * rv);
  }
  float* dst = tt + id * (R * R) + c;
  const uint32_t odd = a ? ~0u : 0u;  // (a bit select: `a ? x : y` became an indexed stack array)
#pragma unroll
  for (int r = 0; r < R; r += 2)
    dst[(r + a) * R] = __uint_as_float((__float_as_uint(col[r + 1]) & odd) | (__float_as_uint(col[r]) & ~odd));
  if (lane == 0) flags[id] = any != 0;
}

// ------------------------------------------------------------------ the segments
struct Args {
  const void *q, *k, *v;
  const float* tt;          // T~ of chunk (bh, n) at tt + (bh nch + n) R R
  const uint32_t* flags;    // accuracy flag of chunk (bh, n)
  const float* psi_in;      // [BH][D][D] or null (identity)
  const float* starts;      // start of segment s >= 1: [(s-1) BH + bh][DP][DP]
  float* factors;           // pass A: transform of segment s: [s BH + bh][DP][DP]
  float* psi_out;           // [BH][D][D]
  void* out;                // [B][T][H][D] or null
  uint32_t* seg_flags;      // pass C: 1 if a chunk of segment (bh, s) is flagged: [bh S + s]
  int T, H, D, BH, nch, seg_chunks, nseg;
  bool vec;
};

template <typename IO, int DP, bool READOUT>
__global__ __launch_bounds__(4 * DP) void c32_pass_kernel(Args a) {
  constexpr int NW = DP / 16, NT = 4 * DP, SS = DP / 16, LU = DP + 4, KP = NW / 2;
  constexpr int NCH = SS >= 4 ? 4 : 2;
  // chunk inputs, double buffered.  All row pitches are 4 mod 64 (or 4 times an odd number), so
  // both the 16-byte reads by 16 rows and the 4-byte reads and writes of 4 x 16 blocks are
  // conflict-free.
  __shared__ __attribute__((aligned(16))) float UT[2][R * LU];     // U^T: row rho = 2t + {k, v}
  __shared__ __attribute__((aligned(16))) float TT[2][R * TTP];
  __shared__ __attribute__((aligned(16))) float QT[2][READOUT ? C * LU : 4];
  __shared__ __attribute__((aligned(16))) float PS[READOUT ? DP * LU : 4];  // Psi_s
  __shared__ __attribute__((aligned(16))) float ZS[READOUT ? R * LU : 4];   // Z
  __shared__ float XP[READOUT ? KP * R * LX : 4];  // mask o (Z Q) over 32 columns each
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int bh = blockIdx.x, seg = blockIdx.y, b = bh / a.H, h = bh - b * a.H;
  const int D = a.D, T = a.T;
  const int c0 = seg * a.seg_chunks, c1 = min(a.nch, c0 + a.seg_chunks);
  const bool readout = READOUT && a.out != nullptr;
  const int64_t DD = static_cast<int64_t>(D) * D;
  const IO* kp = static_cast<const IO*>(a.k);
  const IO* vp = static_cast<const IO*>(a.v);
  const IO* qp = static_cast<const IO*>(a.q);

  // thread's share of a chunk's inputs: features fd .. fd + 3 of token ft, and RT consecutive
  // elements of T~
  constexpr int RT = R * R / NT;
  const int ft = tid / (DP / 4), fd = 4 * (tid % (DP / 4));
  Raw4<IO> rk, rv, rq = {};
  float4 rt[RT / 4 > 0 ? RT / 4 : 1];
  bool rok = false;  // the registers hold a token of the sequence and features below D
  auto fetch = [&](int c) {
    const int t = c * C + ft;
    rok = t < T && fd < D;
    const int64_t o = ((static_cast<int64_t>(b) * T + (rok ? t : 0)) * a.H + h) * D;
    const int d = rok ? fd : 0;
    if (a.vec) {  // clamped loads, no branch per row
      rk.w = *reinterpret_cast<const decltype(rk.w)*>(kp + o + d);
      rv.w = *reinterpret_cast<const decltype(rk.w)*>(vp + o + d);
      if (readout) rq.w = *reinterpret_cast<const decltype(rk.w)*>(qp + o + d);
    } else {
      rk = load4(kp + o, d, D);
      rv = load4(vp + o, d, D);
      if (readout) rq = load4(qp + o, d, D);
    }
    const float* rec = a.tt + (static_cast<int64_t>(bh) * a.nch + c) * (R * R) + RT * tid;
    if constexpr (RT == 2) {
      const float2 x = *reinterpret_cast<const float2*>(rec);
      rt[0] = make_float4(x.x, x.y, 0.f, 0.f);
    } else {
#pragma unroll
      for (int i = 0; i < RT / 4; ++i) rt[i] = reinterpret_cast<const float4*>(rec)[i];
    }
  };
  auto commit = [&](int p) {
    const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
    *reinterpret_cast<float4*>(&UT[p][(2 * ft) * LU + fd]) = rok ? to_f4(rk) : zero;
    *reinterpret_cast<float4*>(&UT[p][(2 * ft + 1) * LU + fd]) = rok ? to_f4(rv) : zero;
    if (READOUT) *reinterpret_cast<float4*>(&QT[p][ft * LU + fd]) = rok ? to_f4(rq) : zero;
    float* d = &TT[p][(RT * tid) / R * TTP + (RT * tid) % R];
    if constexpr (RT == 2) {
      *reinterpret_cast<float2*>(d) = make_float2(rt[0].x, rt[0].y);
    } else {
#pragma unroll
      for (int i = 0; i < RT / 4; ++i) reinterpret_cast<float4*>(d)[i] = rt[i];
    }
  };

  if (c0 < c1) fetch(c0);
  uint32_t flagged = 0;
  for (int c = c0 + tid; c < c1; c += NT) flagged |= a.flags[static_cast<int64_t>(bh) * a.nch + c];
  // state: tile S, register r = row 16 S + 4 g + r of column 16 wave + l16
  f32x4 psi[SS];
  {
    const int col = 16 * wave + l16;
    const float* src = nullptr;
    int ld = D;
    if (READOUT) {
      if (seg > 0) {
        src = a.starts + (static_cast<int64_t>(seg - 1) * a.BH + bh) * DP * DP;
        ld = DP;
      } else if (a.psi_in != nullptr) {
        src = a.psi_in + bh * DD;
      }
    }
    if (src == nullptr) {
#pragma unroll
      for (int S = 0; S < SS; ++S)
#pragma unroll
        for (int r = 0; r < 4; ++r) psi[S][r] = 16 * S + 4 * g + r == col ? 1.f : 0.f;
    } else {  // every load issued (clamped), then the padding cleared
#pragma unroll
      for (int S = 0; S < SS; ++S)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          psi[S][r] = src[static_cast<int64_t>(min(16 * S + 4 * g + r, ld - 1)) * ld + min(col, ld - 1)];
#pragma unroll
      for (int S = 0; S < SS; ++S)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (16 * S + 4 * g + r >= ld || col >= ld) psi[S][r] = 0.f;
    }
  }
  if (c0 < c1) commit(0);
  {  // Inputs visible.  With a flagged chunk the sequence runs again token by token, which writes all
     // of it, so this segment ends here: a call whose sequences are all flagged pays the preparation.
    const int any = __syncthreads_or(flagged != 0);
    if (READOUT && tid == 0) a.seg_flags[static_cast<int64_t>(bh) * a.nseg + seg] = any != 0;
    if (any) return;
  }
  for (int c = c0; c < c1; ++c) {
    const int p = (c - c0) & 1;
    const float *U = UT[p], *Tt = TT[p], *Q = QT[p];
    fetch(c + 1 < c1 ? c + 1 : c);  // the last one again past the end: never committed
    // W = U^T Psi: lane l16 = rank row; step r of tile S takes row 16 S + 4 g + r.  In this and
    // the products below a step's operands are read from LDS while the step before runs (the
    // fences keep the compiler from sinking the reads back to their use).
    f32x4 wp[NCH][2] = {}, w[2], z[2] = {};
    float4 a0 = lds4(U + l16 * LU + 4 * g), a1 = lds4(U + (16 + l16) * LU + 4 * g);
    float4 t0 = lds4(Tt + l16 * TTP + 4 * g), t1 = lds4(Tt + (16 + l16) * TTP + 4 * g);
    float4 t2 = lds4(Tt + l16 * TTP + 16 + 4 * g), t3 = lds4(Tt + (16 + l16) * TTP + 16 + 4 * g);
#pragma unroll
    for (int S = 0; S < SS; ++S) {
      float4 n0 = a0, n1 = a1;
      if (S + 1 < SS) {
        n0 = lds4(U + l16 * LU + 16 * (S + 1) + 4 * g);
        n1 = lds4(U + (16 + l16) * LU + 16 * (S + 1) + 4 * g);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        wp[S % NCH][0] = mma(elem(a0, r), psi[S][r], wp[S % NCH][0]);
        wp[S % NCH][1] = mma(elem(a1, r), psi[S][r], wp[S % NCH][1]);
      }
      __builtin_amdgcn_sched_barrier(0);
      a0 = n0;
      a1 = n1;
    }
    w[0] = tree(wp, 0);
    w[1] = tree(wp, 1);
    // Z = T~ W
    float u[8], un[8];
    auto row_tile = [&](float (&x)[8], int S) {  // U rows 16 S + l16, rank 16 kt + 4 g + r
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = U[(16 * (e >> 2) + 4 * g + (e & 3)) * LU + 16 * S + l16];
    };
    row_tile(u, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      z[0] = mma(elem(t0, r), w[0][r], z[0]);
      z[1] = mma(elem(t1, r), w[0][r], z[1]);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      z[0] = mma(elem(t2, r), w[1][r], z[0]);
      z[1] = mma(elem(t3, r), w[1][r], z[1]);
    }
    if (READOUT) {
      const int col = 16 * wave + l16;
#pragma unroll
      for (int S = 0; S < SS; ++S)
#pragma unroll
        for (int r = 0; r < 4; ++r) PS[(16 * S + 4 * g + r) * LU + col] = psi[S][r];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        ZS[(4 * g + r) * LU + col] = z[0][r];
        ZS[(16 + 4 * g + r) * LU + col] = z[1][r];
      }
      lds_barrier();  // (1) Psi_s and Z of every column visible
    }
    // Psi += U Z, the product first: one rounding at the state's magnitude per chunk
#pragma unroll
    for (int S = 0; S < SS; ++S) {
      if (S + 1 < SS) row_tile(un, S + 1);
      __builtin_amdgcn_sched_barrier(0);
      f32x4 d = {};
#pragma unroll
      for (int e = 0; e < 8; ++e) d = mma(u[e], z[e >> 2][e & 3], d);
      psi[S] += d;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int e = 0; e < 8; ++e) u[e] = un[e];
    }
    f32x4 o = {};
    if (READOUT) {
      // X over columns 32 kp .. + 31, 16 rank rows of it (wave = 2 kp + half)
      const int half = wave & 1, part = wave >> 1;
      f32x4 x = {};
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const float4 az = lds4(ZS + (16 * half + l16) * LU + 32 * part + 16 * s + 4 * g);
        const float4 bq = lds4(Q + l16 * LU + 32 * part + 16 * s + 4 * g);
#pragma unroll
        for (int r = 0; r < 4; ++r) x = mma(elem(az, r), elem(bq, r), x);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int rho = 16 * half + 4 * g + r;
        XP[(part * R + rho) * LX + l16] = (rho >> 1) <= l16 ? x[r] : 0.f;
      }
      // rows 16 wave .. + 15 of O = Psi_s Q
      f32x4 op[NCH][1] = {};
#pragma unroll
      for (int S = 0; S < SS; ++S) {
        const float4 ap = lds4(PS + (16 * wave + l16) * LU + 16 * S + 4 * g);
        const float4 bq = lds4(Q + l16 * LU + 16 * S + 4 * g);
#pragma unroll
        for (int r = 0; r < 4; ++r) op[S % NCH][0] = mma(elem(ap, r), elem(bq, r), op[S % NCH][0]);
      }
      o = tree(op, 0);
    }
    if (c + 1 < c1) commit(p ^ 1);
    lds_barrier();  // (2) X visible, the stashes free again, the next chunk's inputs visible
    if (READOUT) {
      f32x4 d = {};
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int rho = 16 * kt + 4 * g + r;
          float x = XP[rho * LX + l16];
#pragma unroll
          for (int i = 1; i < KP; ++i) x += XP[(i * R + rho) * LX + l16];
          d = mma(U[rho * LU + 16 * wave + l16], x, d);
        }
      o += d;
      const int t = c * C + l16, d0 = 16 * wave + 4 * g;
      if (readout && t < T && d0 < D) {
        IO* dst = static_cast<IO*>(a.out) + ((static_cast<int64_t>(b) * T + t) * a.H + h) * D + d0;
        if (a.vec) {
          if constexpr (sizeof(IO) == 4) {
            *reinterpret_cast<float4*>(dst) = make_float4(o[0], o[1], o[2], o[3]);
          } else {
            IO e[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) io<IO>::store(e, r, o[r]);
            uint2 wv;
            __builtin_memcpy(&wv, e, 8);
            *reinterpret_cast<uint2*>(dst) = wv;
          }
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (d0 + r < D) io<IO>::store(dst, r, o[r]);
        }
      }
    }
  }
  // end state
  if (READOUT && seg != a.nseg - 1) return;
  {
    const int col = 16 * wave + l16;
    float* dst = READOUT ? a.psi_out + bh * DD
                         : a.factors + (static_cast<int64_t>(seg) * a.BH + bh) * DP * DP;
    const int ld = READOUT ? D : DP;
#pragma unroll
    for (int S = 0; S < SS; ++S)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * S + 4 * g + r;
        if (row < ld && col < ld) dst[static_cast<int64_t>(row) * ld + col] = psi[S][r];
      }
  }
}

// ------------------------------------------------------------------ segment start states
// 16 columns of start_s = P_{s-1} start_{s-1} per workgroup, wave w the rows 16 w .. + 15: the
// factor's rows come from global memory in the operand layout two factors ahead, the columns pass through LDS
// (transposed, so a lane's four rows are one 16-byte access); one barrier per factor.
template <int DP>
__global__ __launch_bounds__(4 * DP) void c32_carry_kernel(const float* __restrict__ psi_in,
                                                           const float* __restrict__ factors,
                                                           float* __restrict__ starts, int BH,
                                                           int nf, int D) {
  constexpr int SS = DP / 16, LU = DP + 4;
  __shared__ __attribute__((aligned(16))) float X[2][16 * LU];  // [column][row]
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int bh = blockIdx.x, j0 = 16 * blockIdx.y;
  for (int e = tid; e < 16 * DP; e += 4 * DP) {
    const int row = e / 16, j = e % 16, col = j0 + j;
    float x = row == col ? 1.f : 0.f;
    if (psi_in != nullptr) {
      x = psi_in[static_cast<int64_t>(bh) * D * D + static_cast<int64_t>(min(row, D - 1)) * D + min(col, D - 1)];
      x = row < D && col < D ? x : 0.f;
    }
    X[0][j * LU + row] = x;
  }
  float4 pa[SS], pb[SS];
  auto fetch = [&](float4 (&p)[SS], int f) {
    const float* src = factors + ((static_cast<int64_t>(min(f, nf - 1)) * BH + bh) * DP + 16 * wave + l16) * DP + 4 * g;
#pragma unroll
    for (int S = 0; S < SS; ++S) p[S] = *reinterpret_cast<const float4*>(src + 16 * S);
  };
  auto step = [&](float4 (&p)[SS], int f, int cur) {
    const float* x = X[cur];
    f32x4 y0 = {}, y1 = {};
#pragma unroll
    for (int S = 0; S < SS; ++S) {
      const float4 b4 = lds4(x + l16 * LU + 16 * S + 4 * g);
#pragma unroll
      for (int r = 0; r < 4; r += 2) {
        y0 = mma(elem(p[S], r), elem(b4, r), y0);
        y1 = mma(elem(p[S], r + 1), elem(b4, r + 1), y1);
      }
    }
    fetch(p, f + 2);
    const f32x4 y = y0 + y1;
    *reinterpret_cast<float4*>(&X[cur ^ 1][l16 * LU + 16 * wave + 4 * g]) =
        make_float4(y[0], y[1], y[2], y[3]);
    float* dst = starts + (static_cast<int64_t>(f) * BH + bh) * DP * DP + j0 + l16;
#pragma unroll
    for (int r = 0; r < 4; ++r) dst[static_cast<int64_t>(16 * wave + 4 * g + r) * DP] = y[r];
    lds_barrier();
  };
  fetch(pa, 0);
  fetch(pb, 1);
  lds_barrier();
  for (int f = 0; f < nf; f += 2) {
    step(pa, f, 0);
    if (f + 1 < nf) step(pb, f + 1, 1);
  }
}

// ------------------------------------------------------------------ host side
struct Plan {
  int nch, nseg, seg_chunks, dp;
  size_t tt, flags, segf, fac, st, total;  // byte offsets in the workspace
};

Plan plan(int64_t B, int64_t T, int64_t H, int64_t D) {
  Plan p;
  const int64_t BH = B * H;
  p.dp = D <= 32 ? 32 : D <= 64 ? 64 : 128;
  p.nch = static_cast<int>((T + C - 1) / C);
  p.nseg = 1;
  p.seg_chunks = p.nch;
  // Segments: one more costs every chunk a pass A iteration beside its pass C one, a carry product
  // and two launches, and pays while the chip is not full: one workgroup per CU at D = 128 (155 KB
  // of LDS), two below.  Costs in pass C iterations (measured at D = 128: pass C 8.1 us a chunk,
  // pass A 5.5, a carry product 3, launches and start-up about 12; at D = 64: 3.0, 1.8, 1.1, 11).
  const double ca = 0.65, carry = 0.37, fixed = p.dp == 128 ? 1.5 : 4.0;
  const int64_t room = p.dp == 128 ? 256 : 512;
  double best = p.nch;
  const int64_t smax = std::min<int64_t>({MAX_SEG, p.nch, BH > 0 ? std::max<int64_t>(1, room / BH) : 1});
  for (int s = 2; s <= smax; ++s) {
    const int len = (p.nch + s - 1) / s, n = (p.nch + len - 1) / len;
    const double cost = len * (1.0 + ca) + carry * (n - 1) + fixed;
    if (cost < best) {
      best = cost;
      p.nseg = n;
      p.seg_chunks = len;
    }
  }
  auto up = [](size_t x) { return (x + 255) / 256 * 256; };
  size_t o = 0;
  const size_t chunks = static_cast<size_t>(BH) * p.nch, st = static_cast<size_t>(p.dp) * p.dp * 4;
  p.tt = o;
  o = up(o + chunks * R * R * 4);
  p.flags = o;
  o = up(o + chunks * 4);
  p.segf = o;
  o = up(o + static_cast<size_t>(BH) * p.nseg * 4);
  p.fac = o;
  o = up(o + static_cast<size_t>(p.nseg - 1) * BH * st);
  p.st = o;
  o = up(o + static_cast<size_t>(p.nseg - 1) * BH * st);
  p.total = o;
  return p;
}

template <typename IO, int DP>
hipError_t launch(const Plan& pl, const void* q, const void* k, const void* v, const void* delta,
                  int delta_dtype, const float* psi_in, void* out, float* psi_out, int B, int T,
                  int H, int D, char* ws, hipStream_t stream) {
  const int BH = B * H;
  const int64_t chunks = static_cast<int64_t>(BH) * pl.nch;
  float* tt = reinterpret_cast<float*>(ws + pl.tt);
  uint32_t* flags = reinterpret_cast<uint32_t*>(ws + pl.flags);
  const uintptr_t bits = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) |
                         reinterpret_cast<uintptr_t>(v) | reinterpret_cast<uintptr_t>(out);
  const bool vec = D % 4 == 0 && bits % (4 * sizeof(IO)) == 0;
  hipLaunchKernelGGL((c32_prep_kernel<IO, DP>), dim3(static_cast<unsigned>((chunks + PW - 1) / PW)),
                     dim3(64 * PW), 0, stream, static_cast<const IO*>(k), static_cast<const IO*>(v),
                     delta, delta_dtype, tt, flags, T, H, D, pl.nch, chunks, vec);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  Args a;
  a.q = q; a.k = k; a.v = v;
  a.tt = tt;
  a.flags = flags;
  a.psi_in = psi_in;
  a.starts = reinterpret_cast<float*>(ws + pl.st);
  a.factors = reinterpret_cast<float*>(ws + pl.fac);
  a.psi_out = psi_out;
  a.out = out;
  a.seg_flags = reinterpret_cast<uint32_t*>(ws + pl.segf);
  a.T = T; a.H = H; a.D = D; a.BH = BH;
  a.nch = pl.nch;
  a.seg_chunks = pl.seg_chunks;
  a.nseg = pl.nseg;
  a.vec = vec;
  if (pl.nseg > 1) {
    hipLaunchKernelGGL((c32_pass_kernel<IO, DP, false>), dim3(BH, pl.nseg - 1), dim3(4 * DP), 0,
                       stream, a);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL((c32_carry_kernel<DP>), dim3(BH, DP / 16), dim3(4 * DP), 0, stream, psi_in,
                       a.factors, reinterpret_cast<float*>(ws + pl.st), BH, pl.nseg - 1, D);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  hipLaunchKernelGGL((c32_pass_kernel<IO, DP, true>), dim3(BH, pl.nseg), dim3(4 * DP), 0, stream, a);
  return hipGetLastError();
}

template <typename IO>
hipError_t launch_io(const Plan& pl, const void* q, const void* k, const void* v, const void* delta,
                     int delta_dtype, const float* psi_in, void* out, float* psi_out, int B, int T,
                     int H, int D, char* ws, hipStream_t stream) {
  if (pl.dp == 32)
    return launch<IO, 32>(pl, q, k, v, delta, delta_dtype, psi_in, out, psi_out, B, T, H, D, ws, stream);
  if (pl.dp == 64)
    return launch<IO, 64>(pl, q, k, v, delta, delta_dtype, psi_in, out, psi_out, B, T, H, D, ws, stream);
  return launch<IO, 128>(pl, q, k, v, delta, delta_dtype, psi_in, out, psi_out, B, T, H, D, ws, stream);
}

}  // namespace c32

// Up to 16 tokens are one chunk: four launches whose time is that of filling the chip, where the
// token-sequential scan takes one launch and 2.3 / 3 / 6 us a token at head_dim 32 / 64 / 128.  Both in us
// (fp32, chunk / sequential):
//   D 128: T 5 BH 4 20 / 35, BH 4096 205 / 359: the chunk from 5 tokens on at any number of heads;
//   D 64:  T 5 BH 512 19 / 22, BH 2048 46 / 38; T 9 BH 2048 46 / 57 (D 33 bf16, rows unaligned, 53 / 56);
//   D 32:  the chunk's time grows with the heads already below a full chip: T 6 BH 32 15 / 17, BH 128
//          20 / 17; T 8 BH 128 20 / 22, BH 256 26 / 22; T 10 BH 256 26 / 27, BH 4096 55 / 57.  16-bit
//          rows take 1.5 more (T 9 BH 192 25.5 / 24.7, T 5 BH 16 15.0 / 14.1), and rows that are not
//          whole 4-element pieces more again (D 7 T 7 BH 64 21 / 19; bf16 T 17 BH 4096 96 / 86).
int64_t chunk32_min_tokens(int64_t BH, int64_t D, int io_dtype) {
  if (D > 64) return 5;
  if (D > 32) return BH <= 512 ? 5 : 9;
  const bool f32 = io_dtype == VMI_F32, pieces = D % 4 == 0;
  if (BH <= 16 && f32 && pieces) return 5;
  if (BH > 128 && !pieces) return 20;
  return std::min<int64_t>(10, 6 + (BH + 31) / 64) + (f32 ? 0 : 1) + (pieces ? 0 : 2);
}

bool use_chunk32(int64_t BH, int64_t T, int64_t D, int io_dtype) {
  // a launch holds fewer than 2^32 threads: 64 per chunk in the preparation, 4 per padded feature and
  // sequence in the passes (one segment then; the sequential kernel's are no more)
  constexpr int64_t kThreads = int64_t(1) << 32;
  const int64_t dp = D <= 32 ? 32 : D <= 64 ? 64 : 128;
  return D <= 128 && T >= chunk32_min_tokens(BH, D, io_dtype) && 4 * dp * BH < kThreads &&
         (T + c32::C - 1) / c32::C * BH < kThreads / 64 - c32::PW;
}

size_t chunk32_workspace_bytes(int64_t B, int64_t T, int64_t H, int64_t D, int io_dtype) {
  if (B <= 0 || H <= 0 || !use_chunk32(B * H, T, D, io_dtype)) return 0;
  return c32::plan(B, T, H, D).total;
}

hipError_t launch_sssd_chunk32(const void* q, const void* k, const void* v, const void* delta,
                               int io_dtype, int delta_dtype, const float* psi_in, void* out,
                               float* psi_out, int B, int T, int H, int D, void* workspace,
                               hipStream_t stream) {
  const c32::Plan pl = c32::plan(B, T, H, D);
  char* ws = static_cast<char*>(workspace);
  hipError_t e;
  if (io_dtype == VMI_F32)
    e = c32::launch_io<float>(pl, q, k, v, delta, delta_dtype, psi_in, out, psi_out, B, T, H, D, ws, stream);
  else if (io_dtype == VMI_BF16)
    e = c32::launch_io<bf16_t>(pl, q, k, v, delta, delta_dtype, psi_in, out, psi_out, B, T, H, D, ws, stream);
  else
    e = c32::launch_io<f16_t>(pl, q, k, v, delta, delta_dtype, psi_in, out, psi_out, B, T, H, D, ws, stream);
  if (e != hipSuccess) return e;
  const FlaggedSegments map{reinterpret_cast<const uint32_t*>(ws + pl.segf), pl.nseg};
  return launch_sssd_seq(q, k, v, delta, io_dtype, delta_dtype, psi_in, out, psi_out, B, T, H, D,
                         stream, map);
}

}  // namespace vmi
