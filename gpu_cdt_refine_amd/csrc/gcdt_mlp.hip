// Learned insertion priority: a 3-layer MLP (16 -> 64 -> 64 -> 1, ReLU) with
// BF16 weights and activations feeding v_mfma_f32_16x16x16_bf16 (FP32
// accumulate), trained on the GPU by the forward/backward kernels below.
//
// Inputs are per-candidate features the cavity kernel records (minimum angle,
// circumradius / shortest-edge ratio, cavity and ring size, distance to the
// nearest cavity subsegment, pass index); the target is the candidate's
// conflict degree from the claim logs (how many other candidates claim the
// triangles of its cavity and ring).  The prediction orders candidates inside
// a priority bucket; every insertion is still decided by exact predicates.
//
// Weight layout (FP32 master copy, GCDT_MLP_NPARAM floats):
//   W1[16][64] | b1[64] | W2[64][64] | b2[64] | W3[64] | b3
// A wave (64 lanes) processes 16 samples per step.  MFMA operand layout for
// 16x16x16 (verified by tests/test_gpu_mlp.py against a host product):
//   A[16][16]: lane l holds row l%16, k = 4*(l/16) + 0..3
//   B[16][16]: lane l holds col l%16, k = 4*(l/16) + 0..3
//   D[16][16]: lane l holds col l%16, row = 4*(l/16) + 0..3
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <stdexcept>
#include <string>
#include <vector>

#include "gpu_cdt_refine.h"
#include "mlp_infer.h"

namespace gcdt {

// Inference: the weights converted to BF16 once per block and kept in LDS,
// four waves per block, each wave taking 16 rows at a time; layer 2 on the
// 16x16x32 MFMA.  The gradient kernel's forward pass makes the same products
// and roundings (inputs, weights and hidden activations in BF16, FP32
// accumulate).
constexpr int INF_WAVES = 4;
__global__ __launch_bounds__(64 * INF_WAVES) void k_mlp_infer(const float *X, int n,
                                                              const float *P, float *y,
                                                              const int *dn, const int *dgo) {
  __shared__ MlpWeights w;
  __shared__ __align__(16) short h1[INF_WAVES][16 * H1_STRIDE];  // per wave: [row][k]
  if (dn) n = *dgo ? *dn : 0;
  if (n <= 0 || (int)blockIdx.x * INF_WAVES * 16 >= n) return;
  // Small passes are bound by this staging: 16.2 -> 5.5 us a launch in a
  // 41,003-point refinement with all of its loads in flight, together with
  // more blocks (infer_blocks).
  mlp_stage<64 * INF_WAVES>(P, w, (int)threadIdx.x);
  __syncthreads();
  const int wv = threadIdx.x / 64;
  for (int row0 = (blockIdx.x * INF_WAVES + wv) * 16; row0 < n;
       row0 += gridDim.x * INF_WAVES * 16) {
    mlp_rows16(X, n, row0, w, h1[wv], y);
    wave_sync();  // the activations are rewritten by the next rows
  }
}

// Mean-squared-error gradient over n samples, accumulated into G (MLP_NPARAM
// floats, zeroed by the caller) and the loss sum into *loss.
//
// A wave takes 16 rows at a time and keeps its share of every gradient in
// registers from tile to tile (the weight gradients as MFMA accumulators); the
// block sums its waves in LDS once and adds to G with one atomic per
// parameter.  Weights are converted to BF16 once per block.  200,003 rows: 515 -> 100 us,
// where every tile had added 85 values per lane to LDS and converted its
// weights again from global memory.
constexpr int GRAD_WAVES = 4, GRAD_BLOCKS = 256;
__global__ __launch_bounds__(64 * GRAD_WAVES) void k_mlp_grad(const float *X, const float *t,
                                                              int n, const float *P, float *G,
                                                              float *loss) {
  __shared__ MlpWeights w;
  __shared__ __align__(16) short w2n[MLP_H * W2T_STRIDE];          // W2 [k][c]
  __shared__ __align__(16) short hs[GRAD_WAVES][16 * H1_STRIDE];  // per wave: [row][unit]
  __shared__ float gsh[MLP_NPARAM];
  const int tid = threadIdx.x, wv = tid / 64, l = tid & 63, r = l % 16, kb = l / 16;
  mlp_stage<64 * GRAD_WAVES>(P, w, tid);
  for (int i = tid; i < MLP_H * MLP_H; i += 64 * GRAD_WAVES)
    w2n[(i / MLP_H) * W2T_STRIDE + i % MLP_H] = f2bf(P[OFF_W2 + i]);
  for (int k = tid; k < MLP_NPARAM; k += 64 * GRAD_WAVES) gsh[k] = 0.f;
  __syncthreads();
  short *H = hs[wv];
  const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
  floatx4 g1[4], g2[4][4];
  float gb1[4], gb2[4], gw3[4], gb3 = 0.f, lsum = 0.f;
  for (int a = 0; a < 4; a++) {
    g1[a] = zero;
    gb1[a] = gb2[a] = gw3[a] = 0.f;
    for (int b = 0; b < 4; b++) g2[a][b] = zero;
  }
  for (int row0 = (blockIdx.x * GRAD_WAVES + wv) * 16; row0 < n;
       row0 += gridDim.x * GRAD_WAVES * 16) {
    // ---- forward (D layout: lane l holds column l % 16, rows 4 (l / 16) + j) ----
    floatx4 h1[4], h2[4];
    bf16x4 ax0;
    {
      const int row = row0 + r;
      for (int j = 0; j < 4; j++)
        ax0[j] = row < n ? f2bf(X[(size_t)row * MLP_IN + 4 * kb + j]) : (short)0;
    }
    bf16x4 a1[4];  // H1 in BF16
    for (int cb = 0; cb < 4; cb++) {
      bf16x4 b;
      for (int j = 0; j < 4; j++) b[j] = w.w1[(4 * kb + j) * MLP_H + cb * 16 + r];
      floatx4 z = mfma(ax0, b, zero);
      const float bias = w.b1[cb * 16 + r];
      for (int j = 0; j < 4; j++) {
        z[j] = fmaxf(z[j] + bias, 0.f);
        a1[cb][j] = f2bf(z[j]);
        H[(4 * kb + j) * H1_STRIDE + cb * 16 + r] = a1[cb][j];
      }
      h1[cb] = z;
    }
    wave_sync();
    for (int cb = 0; cb < 4; cb++) {
      floatx4 z = zero;
      for (int kk = 0; kk < 2; kk++) {
        const shortx8 a2 =
            *reinterpret_cast<const shortx8 *>(&H[r * H1_STRIDE + kk * 32 + 8 * kb]);
        const shortx8 b2v = *reinterpret_cast<const shortx8 *>(
            &w.w2t[(cb * 16 + r) * W2T_STRIDE + kk * 32 + 8 * kb]);
        z = mfma32(a2, b2v, z);
      }
      const float bias = w.b2[cb * 16 + r];
      for (int j = 0; j < 4; j++) z[j] = fmaxf(z[j] + bias, 0.f);
      h2[cb] = z;
    }
    // ---- output, its error and layer 3 ----
    float dy[4];
    for (int j = 0; j < 4; j++) {
      float y = 0.f;
      for (int cb = 0; cb < 4; cb++) y += h2[cb][j] * w.w3[cb * 16 + r];
      for (int off = 8; off > 0; off >>= 1) y += __shfl_xor(y, off, 16);
      const int row = row0 + 4 * kb + j;
      const float e = row < n ? y + w.b3 - t[row] : 0.f;
      dy[j] = 2.f * e / (float)n;
      if (r == 0) lsum += e * e;
    }
    for (int cb = 0; cb < 4; cb++)
      for (int j = 0; j < 4; j++) gw3[cb] += h2[cb][j] * dy[j];
    if (r == 0) gb3 += dy[0] + dy[1] + dy[2] + dy[3];
    // ---- dH2 = dy W3 (.) relu', dW2 = H1^T dH2 (the D layout of 16 rows is
    // the A / B layout of a product over them) ----
    bf16x4 d2[4];
    wave_sync();  // H1 was read
    for (int cb = 0; cb < 4; cb++) {
      const float w3 = w.w3[cb * 16 + r];
      for (int j = 0; j < 4; j++) {
        const float d = h2[cb][j] > 0.f ? dy[j] * w3 : 0.f;
        gb2[cb] += d;
        d2[cb][j] = f2bf(d);
        H[(4 * kb + j) * H1_STRIDE + cb * 16 + r] = d2[cb][j];
      }
    }
    for (int mb = 0; mb < 4; mb++)
      for (int nb = 0; nb < 4; nb++) g2[mb][nb] = mfma(a1[mb], d2[nb], g2[mb][nb]);
    wave_sync();
    // ---- dH1 = dH2 W2^T (.) relu', dW1 = X^T dH1 ----
    bf16x4 ax;
    for (int j = 0; j < 4; j++) {
      const int row = row0 + 4 * kb + j;
      ax[j] = row < n ? f2bf(X[(size_t)row * MLP_IN + r]) : (short)0;
    }
    for (int cb = 0; cb < 4; cb++) {
      floatx4 z = zero;
      for (int kk = 0; kk < 2; kk++) {
        const shortx8 a2 =
            *reinterpret_cast<const shortx8 *>(&H[r * H1_STRIDE + kk * 32 + 8 * kb]);
        const shortx8 b2v = *reinterpret_cast<const shortx8 *>(
            &w2n[(cb * 16 + r) * W2T_STRIDE + kk * 32 + 8 * kb]);
        z = mfma32(a2, b2v, z);
      }
      bf16x4 b;
      for (int j = 0; j < 4; j++) {
        const float d = h1[cb][j] > 0.f ? z[j] : 0.f;
        gb1[cb] += d;
        b[j] = f2bf(d);
      }
      g1[cb] = mfma(ax, b, g1[cb]);
    }
    wave_sync();  // H is rewritten by the next rows
  }
  // ---- the block's sum ----
  for (int cb = 0; cb < 4; cb++) {
    for (int j = 0; j < 4; j++) {
      atomicAdd(&gsh[OFF_W1 + (4 * kb + j) * MLP_H + cb * 16 + r], g1[cb][j]);
      for (int mb = 0; mb < 4; mb++)
        atomicAdd(&gsh[OFF_W2 + (mb * 16 + 4 * kb + j) * MLP_H + cb * 16 + r], g2[mb][cb][j]);
    }
    atomicAdd(&gsh[OFF_B1 + cb * 16 + r], gb1[cb]);
    atomicAdd(&gsh[OFF_B2 + cb * 16 + r], gb2[cb]);
    atomicAdd(&gsh[OFF_W3 + cb * 16 + r], gw3[cb]);
  }
  if (r == 0) atomicAdd(&gsh[OFF_B3], gb3);
  for (int off = 32; off > 0; off >>= 1) lsum += __shfl_xor(lsum, off, 64);
  if (l == 0) atomicAdd(loss, lsum);
  __syncthreads();
  for (int k = tid; k < MLP_NPARAM; k += 64 * GRAD_WAVES)
    if (gsh[k] != 0.f) atomicAdd(&G[k], gsh[k]);
}

// Blocks of the gradient kernel for n > 0 rows.
static int grad_blocks(int n) {
  return std::min((n + 16 * GRAD_WAVES - 1) / (16 * GRAD_WAVES), GRAD_BLOCKS);
}

// Adam step on the FP32 master weights.
__global__ void k_adam(float *P, const float *G, float *m1, float *m2, int np,
                       float lr, float b1, float b2, float eps, int step) {
  int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= np) return;
  float g = G[k];
  float a = b1 * m1[k] + (1.f - b1) * g;
  float v = b2 * m2[k] + (1.f - b2) * g * g;
  m1[k] = a;
  m2[k] = v;
  float ah = a / (1.f - powf(b1, (float)step));
  float vh = v / (1.f - powf(b2, (float)step));
  P[k] -= lr * ah / (sqrtf(vh) + eps);
}

// Device MFMA layout probe: D = A(16x16) B(16x16) for host verification.
__global__ void k_mfma_probe(const float *A, const float *B, float *D) {
  int l = threadIdx.x, r = l % 16, kb = l / 16;
  bf16x4 a, b;
  for (int j = 0; j < 4; j++) {
    a[j] = f2bf(A[r * 16 + 4 * kb + j]);
    b[j] = f2bf(B[(4 * kb + j) * 16 + r]);
  }
  floatx4 z = {0.f, 0.f, 0.f, 0.f};
  z = mfma(a, b, z);
  for (int j = 0; j < 4; j++) D[(4 * kb + j) * 16 + r] = z[j];
}

// Device layout probe of the 16x16x32 MFMA: D = A(16x32) B(32x16).
__global__ void k_mfma_probe32(const float *A, const float *B, float *D) {
  int l = threadIdx.x, r = l % 16, kb = l / 16;
  shortx8 a, b;
  for (int j = 0; j < 8; j++) {
    a[j] = f2bf(A[r * 32 + 8 * kb + j]);
    b[j] = f2bf(B[(8 * kb + j) * 16 + r]);
  }
  floatx4 z = {0.f, 0.f, 0.f, 0.f};
  z = mfma32(a, b, z);
  for (int j = 0; j < 4; j++) D[(4 * kb + j) * 16 + r] = z[j];
}

static void hc(hipError_t e, const char *w) {
  if (e != hipSuccess) throw std::runtime_error(std::string(w) + ": " + hipGetErrorString(e));
}

// Inference inside the refinement: scores for n candidates on `stream`.
// Blocks of the inference kernel for n rows, each converting the weights
// once: a tile of 16 rows per wave until every CU has a block (a pass's few
// thousand rows are latency bound), then eight tiles per wave up to 1024.
static int infer_blocks(int n) {
  const int one = (n + 64 * 1 - 1) / (64 * 1);  // one tile of 16 rows per wave
  const int eight = (n + 64 * 8 - 1) / (64 * 8);
  return std::max(1, std::max(std::min(one, 256), std::min(eight, 1024)));
}

void mlp_forward_device(const float *dX, int n, const float *dP, float *dy,
                        hipStream_t stream) {
  if (n > 0) k_mlp_infer<<<infer_blocks(n), 64 * INF_WAVES, 0, stream>>>(dX, n, dP, dy, nullptr, nullptr);
  hc(hipGetLastError(), "mlp forward launch");
}

void mlp_forward_device_n(const float *dX, const int *dn, const int *dgo,
                          const float *dP, float *dy, int blocks,
                          hipStream_t stream) {
  k_mlp_infer<<<std::min(blocks, 1024), 64 * INF_WAVES, 0, stream>>>(dX, 0, dP, dy, dn, dgo);
  hc(hipGetLastError(), "mlp forward launch");
}

}  // namespace gcdt

using namespace gcdt;

static thread_local std::string g_mlp_err;

extern "C" {

int gcdt_mlp_nparam(void) { return MLP_NPARAM; }

// y[n] = MLP(X[n][16]) on the device.
int gcdt_mlp_forward(const float *X, int n, const float *params, float *y) {
  try {
    float *dX, *dP, *dy;
    hc(hipMalloc(&dX, sizeof(float) * (size_t)std::max(n, 1) * MLP_IN), "malloc");
    hc(hipMalloc(&dP, sizeof(float) * MLP_NPARAM), "malloc");
    hc(hipMalloc(&dy, sizeof(float) * (size_t)std::max(n, 1)), "malloc");
    hc(hipMemcpy(dX, X, sizeof(float) * (size_t)n * MLP_IN, hipMemcpyHostToDevice), "copy");
    hc(hipMemcpy(dP, params, sizeof(float) * MLP_NPARAM, hipMemcpyHostToDevice), "copy");
    if (n > 0) k_mlp_infer<<<infer_blocks(n), 64 * INF_WAVES>>>(dX, n, dP, dy, nullptr, nullptr);
    hc(hipGetLastError(), "launch");
    hc(hipDeviceSynchronize(), "sync");
    hc(hipMemcpy(y, dy, sizeof(float) * (size_t)n, hipMemcpyDeviceToHost), "copy");
    (void)hipFree(dX); (void)hipFree(dP); (void)hipFree(dy);
    return 0;
  } catch (const std::exception &e) {
    g_mlp_err = e.what();
    return -2;
  }
}

// Mean-squared-error gradient (grad[MLP_NPARAM]) and mean loss on the device.
int gcdt_mlp_grad(const float *X, const float *t, int n, const float *params,
                  float *grad, float *loss) {
  try {
    float *dX, *dt, *dP, *dG, *dl;
    hc(hipMalloc(&dX, sizeof(float) * (size_t)std::max(n, 1) * MLP_IN), "malloc");
    hc(hipMalloc(&dt, sizeof(float) * (size_t)std::max(n, 1)), "malloc");
    hc(hipMalloc(&dP, sizeof(float) * MLP_NPARAM), "malloc");
    hc(hipMalloc(&dG, sizeof(float) * MLP_NPARAM), "malloc");
    hc(hipMalloc(&dl, sizeof(float)), "malloc");
    hc(hipMemcpy(dX, X, sizeof(float) * (size_t)n * MLP_IN, hipMemcpyHostToDevice), "copy");
    hc(hipMemcpy(dt, t, sizeof(float) * (size_t)n, hipMemcpyHostToDevice), "copy");
    hc(hipMemcpy(dP, params, sizeof(float) * MLP_NPARAM, hipMemcpyHostToDevice), "copy");
    hc(hipMemset(dG, 0, sizeof(float) * MLP_NPARAM), "memset");
    hc(hipMemset(dl, 0, sizeof(float)), "memset");
    if (n > 0) k_mlp_grad<<<grad_blocks(n), 64 * GRAD_WAVES>>>(dX, dt, n, dP, dG, dl);
    hc(hipGetLastError(), "launch");
    hc(hipDeviceSynchronize(), "sync");
    hc(hipMemcpy(grad, dG, sizeof(float) * MLP_NPARAM, hipMemcpyDeviceToHost), "copy");
    float ls;
    hc(hipMemcpy(&ls, dl, sizeof(float), hipMemcpyDeviceToHost), "copy");
    *loss = ls / (float)std::max(n, 1);
    (void)hipFree(dX); (void)hipFree(dt); (void)hipFree(dP); (void)hipFree(dG); (void)hipFree(dl);
    return 0;
  } catch (const std::exception &e) {
    g_mlp_err = e.what();
    return -2;
  }
}

// Train params (in/out) with Adam on the device: mini-batches of `batch`
// samples drawn in a seeded shuffled order, `epochs` passes.  losses[epoch]
// receives the mean training loss of each epoch (may be NULL).
int gcdt_mlp_train(const float *X, const float *t, int n, int epochs, int batch,
                   float lr, unsigned long long seed, float *params,
                   float *losses) {
  try {
    if (n <= 0 || batch <= 0) throw std::runtime_error("empty training set");
    // shuffle once per epoch on the host (index permutation), gather on host
    std::vector<int> perm(n);
    for (int i = 0; i < n; i++) perm[i] = i;
    unsigned long long s = seed * 0x9E3779B97F4A7C15ull + 1;
    auto rnd = [&]() {
      s ^= s << 13;
      s ^= s >> 7;
      s ^= s << 17;
      return s;
    };
    float *dX, *dt, *dP, *dG, *dm1, *dm2, *dl;
    hc(hipMalloc(&dX, sizeof(float) * (size_t)n * MLP_IN), "malloc");
    hc(hipMalloc(&dt, sizeof(float) * (size_t)n), "malloc");
    hc(hipMalloc(&dP, sizeof(float) * MLP_NPARAM), "malloc");
    hc(hipMalloc(&dG, sizeof(float) * MLP_NPARAM), "malloc");
    hc(hipMalloc(&dm1, sizeof(float) * MLP_NPARAM), "malloc");
    hc(hipMalloc(&dm2, sizeof(float) * MLP_NPARAM), "malloc");
    hc(hipMalloc(&dl, sizeof(float)), "malloc");
    hc(hipMemcpy(dP, params, sizeof(float) * MLP_NPARAM, hipMemcpyHostToDevice), "copy");
    hc(hipMemset(dm1, 0, sizeof(float) * MLP_NPARAM), "memset");
    hc(hipMemset(dm2, 0, sizeof(float) * MLP_NPARAM), "memset");
    std::vector<float> hX((size_t)n * MLP_IN), ht(n);
    int step = 0;
    for (int ep = 0; ep < epochs; ep++) {
      for (int i = n - 1; i > 0; i--) std::swap(perm[i], perm[rnd() % (unsigned long long)(i + 1)]);
      for (int i = 0; i < n; i++) {
        std::memcpy(&hX[(size_t)i * MLP_IN], &X[(size_t)perm[i] * MLP_IN], sizeof(float) * MLP_IN);
        ht[i] = t[perm[i]];
      }
      hc(hipMemcpy(dX, hX.data(), sizeof(float) * (size_t)n * MLP_IN, hipMemcpyHostToDevice), "copy");
      hc(hipMemcpy(dt, ht.data(), sizeof(float) * (size_t)n, hipMemcpyHostToDevice), "copy");
      hc(hipMemset(dl, 0, sizeof(float)), "memset");
      double eloss = 0.0;
      for (int b0 = 0; b0 < n; b0 += batch) {
        int nb = std::min(batch, n - b0);
        hc(hipMemset(dG, 0, sizeof(float) * MLP_NPARAM), "memset");
        k_mlp_grad<<<grad_blocks(nb), 64 * GRAD_WAVES>>>(dX + (size_t)b0 * MLP_IN, dt + b0, nb, dP,
                                                         dG, dl);
        step++;
        k_adam<<<(MLP_NPARAM + 255) / 256, 256>>>(dP, dG, dm1, dm2, MLP_NPARAM, lr, 0.9f, 0.999f, 1e-8f, step);
      }
      hc(hipGetLastError(), "launch");
      float ls;
      hc(hipMemcpy(&ls, dl, sizeof(float), hipMemcpyDeviceToHost), "copy");
      eloss = ls;
      // k_mlp_grad accumulates e^2 / n_batch-weighted sums: report per-sample mean
      if (losses) losses[ep] = (float)(eloss / (double)n);
    }
    hc(hipMemcpy(params, dP, sizeof(float) * MLP_NPARAM, hipMemcpyDeviceToHost), "copy");
    (void)hipFree(dX); (void)hipFree(dt); (void)hipFree(dP); (void)hipFree(dG);
    (void)hipFree(dm1); (void)hipFree(dm2); (void)hipFree(dl);
    return 0;
  } catch (const std::exception &e) {
    g_mlp_err = e.what();
    return -2;
  }
}

// D = A B for 16x16 FP32 matrices rounded to BF16 (MFMA layout probe).
// D(16x16) = A(16x32) B(32x16) through the 16x16x32 MFMA (layout check).
int gcdt_mfma_probe32(const float *A, const float *B, float *D) {
  try {
    float *dA, *dB, *dD;
    hc(hipMalloc(&dA, 2048), "malloc");
    hc(hipMalloc(&dB, 2048), "malloc");
    hc(hipMalloc(&dD, 1024), "malloc");
    hc(hipMemcpy(dA, A, 2048, hipMemcpyHostToDevice), "copy");
    hc(hipMemcpy(dB, B, 2048, hipMemcpyHostToDevice), "copy");
    k_mfma_probe32<<<1, 64>>>(dA, dB, dD);
    hc(hipGetLastError(), "launch");
    hc(hipDeviceSynchronize(), "sync");
    hc(hipMemcpy(D, dD, 1024, hipMemcpyDeviceToHost), "copy");
    (void)hipFree(dA); (void)hipFree(dB); (void)hipFree(dD);
    return 0;
  } catch (const std::exception &e) {
    g_mlp_err = e.what();
    return -2;
  }
}

int gcdt_mfma_probe(const float *A, const float *B, float *D) {
  try {
    float *dA, *dB, *dD;
    hc(hipMalloc(&dA, 1024), "malloc");
    hc(hipMalloc(&dB, 1024), "malloc");
    hc(hipMalloc(&dD, 1024), "malloc");
    hc(hipMemcpy(dA, A, 1024, hipMemcpyHostToDevice), "copy");
    hc(hipMemcpy(dB, B, 1024, hipMemcpyHostToDevice), "copy");
    k_mfma_probe<<<1, 64>>>(dA, dB, dD);
    hc(hipGetLastError(), "launch");
    hc(hipDeviceSynchronize(), "sync");
    hc(hipMemcpy(D, dD, 1024, hipMemcpyDeviceToHost), "copy");
    (void)hipFree(dA); (void)hipFree(dB); (void)hipFree(dD);
    return 0;
  } catch (const std::exception &e) {
    g_mlp_err = e.what();
    return -2;
  }
}

const char *gcdt_mlp_last_error(void) { return g_mlp_err.c_str(); }

}  // extern "C"
