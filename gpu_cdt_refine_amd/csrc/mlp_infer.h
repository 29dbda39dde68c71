// The priority network's layout, BF16 helpers and inference steps, shared by
// the inference kernel (gcdt_mlp.hip) and the small-pass refinement kernel
// (gcdt_refine.hip).  Weight layout: see gcdt_mlp.hip.
#pragma once

#include <hip/hip_runtime.h>

namespace gcdt {

constexpr int MLP_IN = 16, MLP_H = 64;
constexpr int OFF_W1 = 0, OFF_B1 = OFF_W1 + MLP_IN * MLP_H, OFF_W2 = OFF_B1 + MLP_H,
              OFF_B2 = OFF_W2 + MLP_H * MLP_H, OFF_W3 = OFF_B2 + MLP_H,
              OFF_B3 = OFF_W3 + MLP_H, MLP_NPARAM = OFF_B3 + 1;

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ short f2bf(float f) {  // round to nearest even
  unsigned u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return (short)(u >> 16);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (short)(u >> 16);
}
__device__ __forceinline__ float bf2f(short h) {
  return __uint_as_float(((unsigned)(unsigned short)h) << 16);
}

__device__ __forceinline__ floatx4 mfma(bf16x4 a, bf16x4 b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// gfx950's double-K BF16 MFMA (v_mfma_f32_16x16x32_bf16), used for the 64-wide
// hidden layer by inference and by the gradient kernel: two instructions per 16x16 output
// block instead of four.  Operand layout (checked by k_mfma_probe32 against a
// host product): A[16][32]: lane l holds row l%16, k = 8*(l/16) + 0..7;
// B[32][16]: lane l holds col l%16, k = 8*(l/16) + 0..7; D as for 16x16x16.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short shortx8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ floatx4 mfma32(shortx8 a, shortx8 b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// LDS written by some lanes of a wave and read by others: release, the
// wave's convergence point, acquire (wavefront scope).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int W2T_STRIDE = MLP_H + 8;  // transposed W2 rows, padded against bank conflicts
constexpr int H1_STRIDE = MLP_H + 8;

// Weights of a block, converted to BF16 once.
struct MlpWeights {
  __align__(16) short w2t[MLP_H * W2T_STRIDE];  // [c][k]
  short w1[MLP_IN * MLP_H];                     // [k][c]
  float b1[MLP_H], b2[MLP_H], w3[MLP_H], b3;
};

// Staged by NT threads (t of them), every load in flight at once; the caller
// synchronises.
template <int NT>
__device__ __forceinline__ void mlp_stage(const float *P, MlpWeights &w, int t) {
  constexpr int N1 = MLP_IN * MLP_H / NT, N2 = MLP_H * MLP_H / NT;
  float v1[N1], v2[N2], vb1 = 0.f, vb2 = 0.f, vw3 = 0.f;
#pragma unroll
  for (int q = 0; q < N1; q++) v1[q] = P[OFF_W1 + q * NT + t];
#pragma unroll
  for (int q = 0; q < N2; q++) v2[q] = P[OFF_W2 + q * NT + t];
  if (t < MLP_H) {
    vb1 = P[OFF_B1 + t];
    vb2 = P[OFF_B2 + t];
    vw3 = P[OFF_W3 + t];
  }
  if (t == 0) w.b3 = P[OFF_B3];
#pragma unroll
  for (int q = 0; q < N1; q++) w.w1[q * NT + t] = f2bf(v1[q]);
#pragma unroll
  for (int q = 0; q < N2; q++) {
    const int k = (q * NT + t) / MLP_H, c = t % MLP_H;
    w.w2t[c * W2T_STRIDE + k] = f2bf(v2[q]);
  }
  if (t < MLP_H) {
    w.b1[t] = vb1;
    w.b2[t] = vb2;
    w.w3[t] = bf2f(f2bf(vw3));
  }
}

// One wave: outputs y of rows row0 .. row0 + 15 (those below n); H: the
// wave's 16 x H1_STRIDE activations, rewritten by the wave's next call after a
// wave_sync().
__device__ __forceinline__ void mlp_rows16(const float *X, int n, int row0, const MlpWeights &w,
                                           short *H, float *y) {
  const int l = threadIdx.x & 63, r = l % 16, kb = l / 16;
  // layer 1 (K = 16): A = X[row0 + r][4kb..4kb+3]
  bf16x4 a;
  const int row = row0 + r;
  for (int j = 0; j < 4; j++)
    a[j] = row < n ? f2bf(X[(size_t)row * MLP_IN + 4 * kb + j]) : (short)0;
  for (int cb = 0; cb < 4; cb++) {
    bf16x4 b;
    for (int j = 0; j < 4; j++) b[j] = w.w1[(4 * kb + j) * MLP_H + cb * 16 + r];
    floatx4 z = {0.f, 0.f, 0.f, 0.f};
    z = mfma(a, b, z);
    const float bias = w.b1[cb * 16 + r];
    // D layout: column cb*16 + r, rows 4kb + j
    for (int j = 0; j < 4; j++) H[(4 * kb + j) * H1_STRIDE + cb * 16 + r] = f2bf(fmaxf(z[j] + bias, 0.f));
  }
  wave_sync();  // H written by the wave's lanes, read by others
  // layer 2 (K = 64 = 2 x 32): A row r, k = kk*32 + 8kb + 0..7 (contiguous in H)
  floatx4 h2[4];
  for (int cb = 0; cb < 4; cb++) {
    floatx4 z = {0.f, 0.f, 0.f, 0.f};
    for (int kk = 0; kk < 2; kk++) {
      const shortx8 a2 = *reinterpret_cast<const shortx8 *>(&H[r * H1_STRIDE + kk * 32 + 8 * kb]);
      const shortx8 b2v =
          *reinterpret_cast<const shortx8 *>(&w.w2t[(cb * 16 + r) * W2T_STRIDE + kk * 32 + 8 * kb]);
      z = mfma32(a2, b2v, z);
    }
    const float bias = w.b2[cb * 16 + r];
    for (int j = 0; j < 4; j++) z[j] = fmaxf(z[j] + bias, 0.f);
    h2[cb] = z;
  }
  // layer 3: y[row] = sum_c H2[row][c] W3[c] + b3 over the 16 lanes of a group
  for (int j = 0; j < 4; j++) {
    float s = 0.f;
    for (int cb = 0; cb < 4; cb++) s += h2[cb][j] * w.w3[cb * 16 + r];
    for (int off = 8; off > 0; off >>= 1) s += __shfl_xor(s, off, 16);
    const int ro = row0 + 4 * kb + j;
    if (r == 0 && ro < n) y[ro] = s + w.b3;
  }
}

}  // namespace gcdt
