// Shared helpers of the LUCID-Path kernels (head dim K = V = 64 or 128, small chunk 64,
// large chunk PR = 16 small chunks = 1024 positions).
//
// fp32 inputs (template flag F32): the caller's tensors are fp32, and every bf16 MFMA
// operand buffer of the workspace holds two bf16 planes, hi = bf16(x) and lo = bf16(x - hi),
// the lo plane at a fixed element offset from the hi plane (PathFwdWs / PathBwdWs lo_*).
// Each product then takes hi.hi + hi.lo + lo.hi (~fp32 accuracy, mm3 below).
#pragma once
#include <type_traits>
#include "lucid_common.h"

namespace lucid {

constexpr int PC = 64;  // small chunk (positions)
constexpr int PR = 16;  // small chunks per large chunk (S = 1024 positions)

// element type of the caller's tensors
template <bool F32>
using pin_t = std::conditional_t<F32, float, bf16>;

// acc + a b over the NP planes of each operand: a[0] b[0] (NP = 1), or the 3-term split
// a[0] b[0] + a[0] b[1] + a[1] b[0] (NP = 2)
template <int NP>
__device__ __forceinline__ f32x16 mm3(const bf16x8* a, const bf16x8* b, f32x16 acc) {
  acc = mfma32(a[0], b[0], acc);
  if constexpr (NP == 2) {
    acc = mfma32(a[0], b[1], acc);
    acc = mfma32(a[1], b[0], acc);
  }
  return acc;
}

// x as bf16 into hi[i], and (NP = 2) its residual into hi[i + lo]
template <int NP>
__device__ __forceinline__ void put_split(bf16* hi, int64_t lo, int64_t i, float x) {
  const bf16 h = (bf16)x;
  hi[i] = h;
  if constexpr (NP == 2) hi[i + lo] = (bf16)(x - (float)h);
}

// acc[i][j] += sum_k opA(A)[r0+i][k] * opB(B)[k][c0+j] for 64x64 fp32 LDS matrices
// (row stride 68); thread t owns the 4x4 block r0 = 4*(t/16), c0 = 4*(t%16).
// Four k-steps per iteration: every operand is read as 16-byte vectors (along k for
// the row-indexed operands, along the block for the others), 8 reads per 64 FMAs.
template <bool TA, bool TB>
__device__ __forceinline__ void lds_gemm64(const float (*A)[68], const float (*B)[68], float acc[4][4]) {
  const int tid = threadIdx.x;
  const int r0 = (tid >> 4) * 4, c0 = (tid & 15) * 4;
#pragma unroll 2
  for (int k = 0; k < 64; k += 4) {
    float a[4][4], b[4][4];  // a[kk][i] = opA[r0+i][k+kk], b[kk][j] = opB[k+kk][c0+j]
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (TA) {
        const f32x4 t4 = *reinterpret_cast<const f32x4*>(&A[k + q][r0]);
#pragma unroll
        for (int i = 0; i < 4; ++i) a[q][i] = t4[i];
      } else {
        const f32x4 t4 = *reinterpret_cast<const f32x4*>(&A[r0 + q][k]);
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) a[kk][q] = t4[kk];
      }
      if (TB) {
        const f32x4 t4 = *reinterpret_cast<const f32x4*>(&B[c0 + q][k]);
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) b[kk][q] = t4[kk];
      } else {
        const f32x4 t4 = *reinterpret_cast<const f32x4*>(&B[k + q][c0]);
#pragma unroll
        for (int j = 0; j < 4; ++j) b[q][j] = t4[j];
      }
    }
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[kk][i], b[kk][j], acc[i][j]);
  }
}

__device__ __forceinline__ void zero44(float acc[4][4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;
}

// One merge of two inverted S x S diagonal blocks A = [a, a+S), B = [a+S, a+2S) of a unit
// lower matrix (I + N): X_BA = -X_B (N_BA X_A), computed in place in the N_BA block in two
// products (Y = N_BA X_A, then -X_B Y) with a barrier after each read and each write; thread
// qd owns 4 consecutive columns of one row of a pair.
template <int S>
struct MergeQuad {
  bool act;
  int i, j0, ao, bo;
  __device__ __forceinline__ explicit MergeQuad(int qd) {
    constexpr int QPP = S * S / 4;  // column quads per pair
    act = qd < (64 / (2 * S)) * QPP;
    const int p = qd / QPP, rem = qd - p * QPP;
    i = rem / (S / 4);
    j0 = 4 * (rem - i * (S / 4));
    ao = 2 * p * S;
    bo = ao + S;
  }
  // Y = N_BA X_A (X = false) or X_B Y (X = true)
  template <bool X>
  __device__ __forceinline__ f32x4 product(const float (*M)[68]) const {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (act) {
#pragma unroll
      for (int kk = 0; kk < S; ++kk) {
        const float a = M[bo + i][(X ? bo : ao) + kk];
        const f32x4 x = *reinterpret_cast<const f32x4*>(&M[(X ? bo : ao) + kk][ao + j0]);
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[e] = fmaf(a, x[e], acc[e]);
      }
    }
    return acc;
  }
  __device__ __forceinline__ void put(float (*M)[68], const f32x4& x) const {
    if (act) *reinterpret_cast<f32x4*>(&M[bo + i][ao + j0]) = x;
  }
};

template <int S>
__device__ __forceinline__ void merge_lower_blocks(float (*M)[68]) {
  const MergeQuad<S> m(threadIdx.x);
  const f32x4 y = m.template product<false>(M);
  __syncthreads();
  m.put(M, y);
  __syncthreads();
  const f32x4 x = m.template product<true>(M);
  __syncthreads();
  m.put(M, -x);
  __syncthreads();
}

// The four 16x16 diagonal blocks of (I + M)^-1 in place (wave w < 4: block w) by forward
// substitution: lane c < 16 solves column c, x_r = delta_rc - sum_{k<r} M_rk x_k.
__device__ __forceinline__ void invert_lower16(float (*M)[68], int w, int c) {
  if (c < 16) {
    const int o = 16 * w;
    float x[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float a0 = (r == c) ? 1.f : 0.f, a1 = 0.f;
#pragma unroll
      for (int kk = 0; kk < (r & ~3); kk += 4) {
        const f32x4 m4 = *reinterpret_cast<const f32x4*>(&M[o + r][o + kk]);
        a0 = fmaf(-m4[0], x[kk], a0);
        a1 = fmaf(-m4[1], x[kk + 1], a1);
        a0 = fmaf(-m4[2], x[kk + 2], a0);
        a1 = fmaf(-m4[3], x[kk + 3], a1);
      }
#pragma unroll
      for (int kk = (r & ~3); kk < r; ++kk) a0 = fmaf(-M[o + r][o + kk], x[kk], a0);
      x[r] = a0 + a1;
    }
    // only this wave reads its diagonal block, so it may write it back right away
#pragma unroll
    for (int r = 0; r < 16; ++r) M[o + r][o + c] = x[r];
  }
}

// Step st = 0 .. 8 of invert_unit_lower64 for the four waves w4 (thread ht of their 256), a
// barrier of the whole block after each: lets other waves of the block work between them.
struct InvertSteps {
  MergeQuad<16> m16;
  MergeQuad<32> m32;
  f32x4 x;
  __device__ __forceinline__ explicit InvertSteps(int ht) : m16(ht), m32(ht) {}
  template <int ST>
  __device__ __forceinline__ void step(float (*M)[68], int w4) {
    if constexpr (ST == 0) invert_lower16(M, w4, threadIdx.x & 63);
    if constexpr (ST == 1) x = m16.product<false>(M);
    if constexpr (ST == 2) m16.put(M, x);
    if constexpr (ST == 3) x = m16.product<true>(M);
    if constexpr (ST == 4) m16.put(M, -x);
    if constexpr (ST == 5) x = m32.product<false>(M);
    if constexpr (ST == 6) m32.put(M, x);
    if constexpr (ST == 7) x = m32.product<true>(M);
    if constexpr (ST == 8) m32.put(M, -x);
  }
};

// (I + M)^-1 in place for a strictly lower 64x64 fp32 LDS matrix M (its diagonal and
// strictly upper part must hold zeros; the result has a unit diagonal and zeros above).
// Called by all 256 threads of the block; the caller syncs before, the function syncs
// before returning.  Wave w inverts the 16x16 diagonal block w; the blocks are then merged
// 16 -> 32 -> 64 through X_BA = -X_B N_BA X_A.  A 64-deep solve in one wave has four times
// the dependent work and leaves three waves idle.
__device__ __forceinline__ void invert_unit_lower64(float (*M)[68]) {
  invert_lower16(M, threadIdx.x >> 6, threadIdx.x & 63);
  __syncthreads();
  merge_lower_blocks<16>(M);
  merge_lower_blocks<32>(M);
}

// Load a 64x64 block of fp32 rows (row stride st elements) into an fp32 LDS matrix.
__device__ __forceinline__ void load_rows64_f32(float (*dst)[68], const float* __restrict__ src, int64_t st) {
  const int tid = threadIdx.x;
  const int r = tid >> 2, c = (tid & 3) * 16;
#pragma unroll
  for (int q4 = 0; q4 < 4; ++q4)
    *reinterpret_cast<f32x4*>(&dst[r][c + 4 * q4]) = *reinterpret_cast<const f32x4*>(src + (int64_t)r * st + c + 4 * q4);
}
// The same from bf16 hi / lo planes (lo = element offset of the lo plane; 0: none).
__device__ __forceinline__ void load_rows64_split(float (*dst)[68], const bf16* __restrict__ src, int64_t st,
                                                  int64_t lo) {
  const int tid = threadIdx.x;
  const int r = tid >> 2, c = (tid & 3) * 16;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const bf16x8 x = ld8(src + (int64_t)r * st + c + 8 * h);
    bf16x8 y{};
    if (lo) y = ld8(src + lo + (int64_t)r * st + c + 8 * h);
#pragma unroll
    for (int e = 0; e < 8; ++e) dst[r][c + 8 * h + e] = (float)x[e] + (lo ? (float)y[e] : 0.f);
  }
}
// Load a 64x64 block of bf16 rows (row stride st elements) into an fp32 LDS matrix.
__device__ __forceinline__ void load_rows64_f32(float (*dst)[68], const bf16* __restrict__ src, int64_t st) {
  const int tid = threadIdx.x;
  const int r = tid >> 2, c = (tid & 3) * 16;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const bf16x8 x = ld8(src + (int64_t)r * st + c + 8 * h);
#pragma unroll
    for (int e = 0; e < 8; ++e) dst[r][c + 8 * h + e] = (float)x[e];
  }
}

// Load a 64x64 fp32 row-major matrix (contiguous) into LDS, optionally transposed.
template <bool TRANS>
__device__ __forceinline__ void load_mat64(float (*dst)[68], const float* __restrict__ src) {
  for (int idx = threadIdx.x; idx < 4096; idx += 256) {
    const int r = idx >> 6, c = idx & 63;
    if (TRANS)
      dst[c][r] = src[idx];
    else
      dst[r][c] = src[idx];
  }
}

// x <- x M for x [64 rows][64] in LDS (fp32) and M^T in LDS (MT[n][k] = M[k][n]),
// computed as D^T = M^T x^T with a 3-term bf16 split (~fp32 accuracy).  Each of the
// four waves produces one 32x32 tile; returns it in D layout (m = column n of the
// product, lane <-> row) through `o`; the caller syncs before writing it back.
__device__ __forceinline__ f32x16 mat_xM_tile(const float (*X)[68], const float (*MT)[68], int dt, int rt) {
  const int lane = threadIdx.x & 63, g = lane >> 5, l32 = lane & 31;
  f32x16 o = zero16();
#pragma unroll
  for (int st = 0; st < 4; ++st) {
    bf16x8 ah, al, bh8, bl;
    split8(&MT[dt * 32 + l32][16 * st + 8 * g], ah, al);
    split8(&X[rt * 32 + l32][16 * st + 8 * g], bh8, bl);
    o = mfma32(ah, bh8, o);
    o = mfma32(ah, bl, o);
    o = mfma32(al, bh8, o);
  }
  return o;
}

// ---------------------------------------------------------------------------
// 64x64 fp32 LDS matrix products on the matrix cores.  Wave w owns the 32x32 output
// tile (tm = w >> 1, tn = w & 1) in MFMA D layout: element e of lane l is
// C[32 tm + drow(e, l / 32)][32 tn + l % 32] (dl_row / dl_col below).
// acc += opA(A) opB(B) with a 3-term bf16 split (hi.hi + hi.lo + lo.hi, ~fp32
// accuracy); operands are read along k as 16-byte vectors where the layout allows
// (A not transposed, B transposed) and gathered otherwise.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int dl_row(int e) {
  return 32 * ((int)threadIdx.x >> 7) + drow(e, ((int)threadIdx.x >> 5) & 1);
}
__device__ __forceinline__ int dl_col() { return 32 * (((int)threadIdx.x >> 6) & 1) + ((int)threadIdx.x & 31); }

__device__ __forceinline__ void split_vals(const float v[8], bf16x8& hi, bf16x8& lo) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const bf16 h = (bf16)v[e];
    hi[e] = h;
    lo[e] = (bf16)(v[e] - (float)h);
  }
}

template <bool TA, bool TB>
__device__ __forceinline__ f32x16 mgemm64(const float (*A)[68], const float (*B)[68], f32x16 acc) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, g = lane >> 5, l32 = lane & 31;
  const int m = 32 * (w >> 1) + l32, n = 32 * (w & 1) + l32;
#pragma unroll
  for (int st = 0; st < 4; ++st) {
    const int k0 = 16 * st + 8 * g;
    float a[8], b[8];
    if (TA) {
#pragma unroll
      for (int i = 0; i < 8; ++i) a[i] = A[k0 + i][m];
    } else {
      const f32x4 x = *reinterpret_cast<const f32x4*>(&A[m][k0]);
      const f32x4 y = *reinterpret_cast<const f32x4*>(&A[m][k0 + 4]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a[i] = x[i];
        a[4 + i] = y[i];
      }
    }
    if (TB) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(&B[n][k0]);
      const f32x4 y = *reinterpret_cast<const f32x4*>(&B[n][k0 + 4]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        b[i] = x[i];
        b[4 + i] = y[i];
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) b[i] = B[k0 + i][n];
    }
    bf16x8 ah, al, bh, bl;
    split_vals(a, ah, al);
    split_vals(b, bh, bl);
    acc = mfma32(ah, bh, acc);
    acc = mfma32(ah, bl, acc);
    acc = mfma32(al, bh, acc);
  }
  return acc;
}

// D-layout tile helpers for mgemm64 results: S[row][col] <- x (masked), x <- S[row][col]
#define DL_FOR_E _Pragma("unroll") for (int e = 0; e < 16; ++e)
__device__ __forceinline__ void dl_store(float (*S)[68], const f32x16& x, int mode) {
  // mode 0: all, 1: col <= row (tril), 2: col < row (strictly lower)
  const int cl = dl_col();
  DL_FOR_E {
    const int r = dl_row(e);
    const bool keep = mode == 0 || (mode == 1 ? cl <= r : cl < r);
    S[r][cl] = keep ? x[e] : 0.f;
  }
}
// 64 x 64 block of an fp32 row-major matrix (row stride ld) into an LDS block, and back
__device__ __forceinline__ void load_blk(float (*dst)[68], const float* __restrict__ src, int ld) {
  for (int idx = threadIdx.x; idx < 1024; idx += 256) {
    const int r = idx >> 4, c4 = (idx & 15) * 4;
    *reinterpret_cast<f32x4*>(&dst[r][c4]) = *reinterpret_cast<const f32x4*>(src + (int64_t)r * ld + c4);
  }
}
__device__ __forceinline__ void store_blk(float* __restrict__ dst, int ld, const float (*src)[68]) {
  for (int idx = threadIdx.x; idx < 1024; idx += 256) {
    const int r = idx >> 4, c4 = (idx & 15) * 4;
    *reinterpret_cast<f32x4*>(dst + (int64_t)r * ld + c4) = *reinterpret_cast<const f32x4*>(&src[r][c4]);
  }
}
// D-layout tile (this wave's 32 x 32 of a 64 x 64 block) to a row-major fp32 / bf16 matrix
__device__ __forceinline__ void dl_put(float* __restrict__ dst, int ld, const f32x16& x) {
  const int cl = dl_col();
  DL_FOR_E dst[(int64_t)dl_row(e) * ld + cl] = x[e];
}

// 64x64 fp32 row-major matrix: thread t holds rows (t + 256 i) / 16, 4 columns each
__device__ __forceinline__ void mat_fetch(f32x4 v[4], const float* __restrict__ src) {
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const f32x4*>(src + 4 * (threadIdx.x + 256 * i));
}
__device__ __forceinline__ void mat_put(float (*S)[68], const f32x4 v[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int f = 4 * (threadIdx.x + 256 * i);
    *reinterpret_cast<f32x4*>(&S[f >> 6][f & 63]) = v[i];
  }
}
__device__ __forceinline__ f32x16 dl_neg(f32x16 x) {
  DL_FOR_E x[e] = -x[e];
  return x;
}

// ---------------------------------------------------------------------------
// 64x64 matrices held in LDS as bf16 planes, split once when they are written: plane 0 the
// rounded value, plane 1 (NP = 2) the rest, so a product reads operands that mgemm64 would
// gather and split anew at every use (same 3-term products, same rounding).  Rows of 128
// bytes, 16-byte chunks swizzled (chunk c of row r at c ^ (r & 7)); columns come through
// transposing reads.  NP = 1: a matrix of bf16 values, whose second term is zero and left out.
// Tiles are transposed to mgemm64's: of wave w4's 32x32 tile (rows 32 (w4 >> 1), columns
// 32 (w4 & 1)), lane l holds row l % 32, columns drow(e, l / 32).
// ---------------------------------------------------------------------------
template <int NP>
struct PlaneMat {
  bf16 p[NP][64 * 64];
};

// opA(A) opB(B) + acc for wave w4 of four
template <bool TA, bool TB, int NA, int NB>
__device__ __forceinline__ f32x16 pgemm64(const PlaneMat<NA>& A, const PlaneMat<NB>& B, int w4, f32x16 acc) {
  const int lane = threadIdx.x & 63, g = lane >> 5, l32 = lane & 31;
  const int m0 = 32 * (w4 >> 1), n0 = 32 * (w4 & 1);
  // rows r0 + l32 of X, depth 16 st + slot; PERM: depth 16 st + jmap(slot), the transposing reads' order
  auto rows = [&](const bf16* X, int r0, int st, auto perm) {
    if constexpr (!decltype(perm)::value) return ld8(swz<8>(X, r0 + l32, 2 * st + g));
    const bf16x4 a = *reinterpret_cast<const bf16x4*>(swz<8>(X, r0 + l32, 2 * st) + 4 * g);
    const bf16x4 b = *reinterpret_cast<const bf16x4*>(swz<8>(X, r0 + l32, 2 * st + 1) + 4 * g);
    return bf16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  };
#pragma unroll
  for (int st = 0; st < 4; ++st) {
    bf16x8 a[NA], b[NB];
#pragma unroll
    for (int pl = 0; pl < NA; ++pl) {
      if constexpr (TA) a[pl] = lds_tr_a<8>(A.p[pl], 16 * st, m0);
      else a[pl] = rows(A.p[pl], m0, st, std::bool_constant<!TB>{});
    }
#pragma unroll
    for (int pl = 0; pl < NB; ++pl) {
      if constexpr (!TB) b[pl] = lds_tr_a<8>(B.p[pl], 16 * st, n0);
      else b[pl] = rows(B.p[pl], n0, st, std::bool_constant<TA>{});
    }
    acc = mfma32(b[0], a[0], acc);
    if constexpr (NA == 2) acc = mfma32(b[0], a[1], acc);
    if constexpr (NB == 2) acc = mfma32(b[1], a[0], acc);
  }
  return acc;
}

// row and first column of quad q (four columns, elements 4 q .. 4 q + 3) of this lane's tile
__device__ __forceinline__ int pl_row(int w4) { return 32 * (w4 >> 1) + ((int)threadIdx.x & 31); }
__device__ __forceinline__ int pl_col(int w4, int q) {
  return 32 * (w4 & 1) + 8 * q + 4 * (((int)threadIdx.x >> 5) & 1);
}
// M[tile] <- x; mode 0: all, 1: col <= row (tril), 2: col < row (strictly lower)
__device__ __forceinline__ f32x4 pl_quad(const f32x16& x, int w4, int q, int mode) {
  const int r = pl_row(w4), c0 = pl_col(w4, q);
  f32x4 f;
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const bool keep = mode == 0 || (mode == 1 ? c0 + u <= r : c0 + u < r);
    f[u] = keep ? x[4 * q + u] : 0.f;
  }
  return f;
}
__device__ __forceinline__ void pl_store(PlaneMat<2>& M, const f32x16& x, int w4, int mode) {
  const int r = pl_row(w4);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int c0 = pl_col(w4, q);
    const f32x4 f = pl_quad(x, w4, q, mode);
    bf16x4 h, l;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      h[u] = (bf16)f[u];
      l[u] = (bf16)(f[u] - (float)h[u]);
    }
    const int off = swz_off<8>(r, c0 >> 3) + (c0 & 7);
    *reinterpret_cast<bf16x4*>(M.p[0] + off) = h;
    *reinterpret_cast<bf16x4*>(M.p[1] + off) = l;
  }
}
// 16-byte chunk c of row r from eight fp32 values
template <int NP>
__device__ __forceinline__ void pl_put8(PlaneMat<NP>& M, int r, int c, const f32x4& x, const f32x4& y) {
  const float v[8] = {x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
  bf16x8 h, l;
  split_vals(v, h, l);
  *reinterpret_cast<bf16x8*>(M.p[0] + swz_off<8>(r, c)) = h;
  if constexpr (NP == 2) *reinterpret_cast<bf16x8*>(M.p[1] + swz_off<8>(r, c)) = l;
}
// this lane's tile of row-major fp32 64x64 rows (row stride st; 64 for a matrix), and back
__device__ __forceinline__ f32x16 pl_load(const float* __restrict__ src, int w4, int64_t st = 64) {
  f32x16 x;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const f32x4 f = *reinterpret_cast<const f32x4*>(src + pl_row(w4) * st + pl_col(w4, q));
#pragma unroll
    for (int u = 0; u < 4; ++u) x[4 * q + u] = f[u];
  }
  return x;
}
__device__ __forceinline__ void pl_save(float* __restrict__ dst, const f32x16& x, int w4) {
#pragma unroll
  for (int q = 0; q < 4; ++q) *reinterpret_cast<f32x4*>(dst + pl_row(w4) * 64 + pl_col(w4, q)) = pl_quad(x, w4, q, 0);
}

// this lane's tile of rows of the caller's tensor in fp32 (row stride st), whose bf16 planes
// are in M: from the plane where that is the whole value, else from memory
template <bool F32>
__device__ __forceinline__ f32x16 pl_rows(const PlaneMat<F32 ? 2 : 1>& M, const pin_t<F32>* __restrict__ src,
                                          int64_t st, int w4) {
  if constexpr (F32) return pl_load(src, w4, st);
  f32x16 x;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int c0 = pl_col(w4, q);
    const bf16x4 v = *reinterpret_cast<const bf16x4*>(M.p[0] + swz_off<8>(pl_row(w4), c0 >> 3) + (c0 & 7));
#pragma unroll
    for (int u = 0; u < 4; ++u) x[4 * q + u] = (float)v[u];
  }
  return x;
}
// eight values of the caller's row (chunk c of row r) into the planes; x: the values in fp32
template <bool F32>
__device__ __forceinline__ void pl_rows_in(PlaneMat<F32 ? 2 : 1>& M, const pin_t<F32>* __restrict__ src, int r, int c,
                                           f32x4 x[2]) {
  if constexpr (F32) {
    x[0] = *reinterpret_cast<const f32x4*>(src);
    x[1] = *reinterpret_cast<const f32x4*>(src + 4);
    pl_put8(M, r, c, x[0], x[1]);
  } else {
    const bf16x8 v = ld8(src);
    *reinterpret_cast<bf16x8*>(M.p[0] + swz_off<8>(r, c)) = v;
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e >> 2][e & 3] = (float)v[e];
  }
}
// this lane's tile to row-major bf16 rows (row stride 64) and, NP = 2, the rest at dst + lo
template <int NP>
__device__ __forceinline__ void pl_save_split(bf16* __restrict__ dst, int64_t lo, const f32x16& x, int w4) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    bf16x4 h, l;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      h[u] = (bf16)x[4 * q + u];
      l[u] = (bf16)(x[4 * q + u] - (float)h[u]);
    }
    bf16* d = dst + pl_row(w4) * 64 + pl_col(w4, q);
    *reinterpret_cast<bf16x4*>(d) = h;
    if constexpr (NP == 2) *reinterpret_cast<bf16x4*>(d + lo) = l;
  }
}

}  // namespace lucid
