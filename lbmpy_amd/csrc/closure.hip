// Learned-closure kernels: feature extraction, batched MLP inference, one training step (forward,
// backward and weight gradients on BF16 MFMA with FP32 accumulation) and an Adam update that
// re-packs the BF16 weights.  The fused inference inside the cumulant sweep uses the same
// mlp_forward_wave (closure.h).
//
// Training loss over n samples:  L = (1/n) sum (softplus(o) - y)^2,  y = nu_t / nu_scale.
// Master parameters (FP32, flat): w1t[32][16] | w2t[32][32] | w3[32] | b1[32] | b2[32] | b3.
#include <string>

#include "lbm_common.h"
#include "closure.h"

namespace lbm355 {

constexpr int OFF_W1T = 0, OFF_W2T = 512, OFF_W3 = 1536, OFF_B1 = 1568, OFF_B2 = 1600, OFF_B3 = 1632;
constexpr int MASTER_SIZE = 1633;

__global__ void __launch_bounds__(256) features_kernel(const float* __restrict__ pi6, const float* __restrict__ rho,
                                                       int64_t n, float* __restrict__ x) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const float p[6] = {pi6[6 * i], pi6[6 * i + 1], pi6[6 * i + 2], pi6[6 * i + 3], pi6[6 * i + 4], pi6[6 * i + 5]};
    float f[CLOSURE_IN];
    closure_features(p, 1.f / rho[i], f);
#pragma unroll
    for (int k = 0; k < CLOSURE_IN; ++k) x[CLOSURE_IN * i + k] = f[k];
  }
}

// persistent waves over 64-sample tiles; lanes past n compute on zeros and store nothing
__global__ void __launch_bounds__(256) forward_kernel(const ClosureParams* __restrict__ P, const float* __restrict__ X,
                                                      int64_t n, float* __restrict__ out) {
  const int lane = threadIdx.x & 63;
  const int64_t wave = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int64_t nwaves = (int64_t)gridDim.x * (blockDim.x >> 6);
  const int64_t ntiles = (n + 63) / 64;
  for (int64_t tile = wave; tile < ntiles; tile += nwaves) {
    const int64_t i = tile * 64 + lane;
    const bool valid = i < n;
    float x[CLOSURE_IN];
#pragma unroll
    for (int k = 0; k < CLOSURE_IN; ++k) x[k] = valid ? X[CLOSURE_IN * i + k] : 0.f;
    const float o = mlp_forward_wave(P, x, nullptr, nullptr);
    if (valid) out[i] = o;
  }
}

__global__ void zero_kernel(float* __restrict__ p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.f;
}

// Orders a wavefront's LDS writes before its own lanes' reads.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ float half_wave_sum(float x) {   // over the 32 lanes of lane's half
#pragma unroll
  for (int o = 16; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  return x;
}

// Row stride of the per-block partial gradients: the 1633 gradient entries, the loss, and padding to 64-column blocks.
constexpr int LOSS_COL = MASTER_SIZE, PARTIAL_STRIDE = 1664;
constexpr int TRAIN_WAVES = 4;
constexpr int CELL_LD = 68;   // LDS row of 64 cells in BF16; 34 dwords keep the 8-byte reads of 32 rows apart

// Gradient of one minibatch: four wavefronts per block, each over tiles of 64 samples (index: the samples' rows, or null
// for the first n).  The weight gradients are MFMA products over the cells of a tile (K = cells), whose operands
// cross the lanes through LDS as the BF16 values the products take; the bias and output sums stay in FP32 registers.
// The block's four waves are summed in LDS and go to one row of `out`, summed by closure_reduce_kernel: in a fixed
// order, and without 1633 atomics of every wavefront to the same addresses.  Bound by the latency of one tile: 65536
// samples took 52 us with the atomics (and FP32 operands in LDS, 32 banks apart).
// ATOMIC: add to out[1633] and loss[0] instead, for callers that bring no memory for the rows.
template <bool ATOMIC>
__global__ void __launch_bounds__(64 * TRAIN_WAVES) train_kernel(const ClosureParams* __restrict__ P,
                                                                 const float* __restrict__ X,
                                                                 const float* __restrict__ Y,
                                                                 const int64_t* __restrict__ index, int64_t n,
                                                                 float inv_n, float* __restrict__ out,
                                                                 float* __restrict__ loss) {
  constexpr int OPERANDS = (3 * CLOSURE_H + CLOSURE_IN_PAD) * CELL_LD;
  __shared__ union {
    short cells[TRAIN_WAVES][OPERANDS];
    float sums[TRAIN_WAVES][MASTER_SIZE + 1];
  } lds;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int half = lane >> 5, col = lane & 31;
  short* const s_a1 = lds.cells[wv];
  short* const s_d2 = s_a1 + CLOSURE_H * CELL_LD;
  short* const s_d1 = s_d2 + CLOSURE_H * CELL_LD;
  short* const s_a0 = s_d1 + CLOSURE_H * CELL_LD;
  v16f gW1, gW2;
  float sb1[16], sb2[16], sw3[16], gb3 = 0.f, lsum = 0.f;
#pragma unroll
  for (int v = 0; v < 16; ++v) gW1[v] = gW2[v] = sb1[v] = sb2[v] = sw3[v] = 0.f;
  // W2 as an A operand [k1][k2] = w2t[k2][k1], per K block
  v4s w2ta[4];
#pragma unroll
  for (int kb = 0; kb < 4; ++kb)
#pragma unroll
    for (int t = 0; t < 4; ++t) w2ta[kb][t] = (short)P->w2t[8 * kb + 4 * half + t][col];
  float w3r[16];
#pragma unroll
  for (int v = 0; v < 16; ++v) w3r[v] = bf2f(P->w3[c_row(v, lane)]);

  const int64_t ntiles = (n + 63) / 64;
  for (int64_t tile = (int64_t)blockIdx.x * TRAIN_WAVES + wv; tile < ntiles; tile += (int64_t)gridDim.x * TRAIN_WAVES) {
    const int64_t i = tile * 64 + lane;
    const bool valid = i < n;
    const int64_t row = valid ? (index ? index[i] : i) : 0;
    float x[CLOSURE_IN];
#pragma unroll
    for (int k = 0; k < CLOSURE_IN; ++k) x[k] = valid ? X[CLOSURE_IN * row + k] : 0.f;
    const float y = valid ? Y[row] : 0.f;
    float h1[2][16], h2[2][16];
    const float o = mlp_forward_wave(P, x, h1, h2);
    const float diff = softplus(o) - y;
    const float g = valid ? 2.f * inv_n * diff * sigmoid(o) : 0.f;
    lsum += valid ? diff * diff : 0.f;
    gb3 += g;
    wave_lds_fence();   // the previous tile's operands have been read
#pragma unroll
    for (int f = 0; f < CLOSURE_IN_PAD; ++f)
      s_a0[f * CELL_LD + lane] = f < CLOSURE_IN ? (short)f2bf((x[f] - P->in_shift[f]) * P->in_scale[f]) : (short)0;
    const float g_other = __shfl_xor(g, 32, 64);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const float gc = (c == half) ? g : g_other;        // dL/do of cell 32c + col
      const int cell = 32 * c + col;
      v4s db[4];
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const float d2 = gc * w3r[v] * (1.f - h2[c][v] * h2[c][v]);
        const int at = c_row(v, lane) * CELL_LD + cell;
        const short d = (short)f2bf(d2);
        s_a1[at] = (short)f2bf(h1[c][v]);
        s_d2[at] = d;
        db[v >> 2][v & 3] = d;
        sb2[v] += d2;
        sw3[v] += gc * h2[c][v];
      }
      v16f acc;
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[v] = 0.f;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) acc = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(w2ta[kb], db[kb], acc, 0, 0, 0);
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const float d1 = acc[v] * (1.f - h1[c][v] * h1[c][v]);
        s_d1[c_row(v, lane) * CELL_LD + cell] = (short)f2bf(d1);
        sb1[v] += d1;
      }
    }
    wave_lds_fence();
    // weight gradients: K = the 64 cells of the tile, 8 blocks of 8
    auto cells_of = [&](const short* m, int unit, int kb) {
      v4s r;
      __builtin_memcpy(&r, __builtin_assume_aligned(m + unit * CELL_LD + 8 * kb + 4 * half, 8), sizeof r);
      return r;
    };
#pragma unroll
    for (int kb = 0; kb < 8; ++kb) {
      gW2 = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(cells_of(s_d2, col, kb), cells_of(s_a1, col, kb), gW2, 0, 0, 0);
      // the inputs fill 16 of the product's 32 columns; the others repeat them and are not read
      gW1 = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(cells_of(s_d1, col, kb), cells_of(s_a0, col & 15, kb), gW1, 0, 0,
                                                     0);
    }
  }
  __syncthreads();
  float* const mine = lds.sums[wv];
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int row = c_row(v, lane);
    mine[OFF_W2T + row * CLOSURE_H + col] = gW2[v];
    if (col < CLOSURE_IN_PAD) mine[OFF_W1T + row * CLOSURE_IN_PAD + col] = gW1[v];
    const float b1 = half_wave_sum(sb1[v]), b2 = half_wave_sum(sb2[v]), w3 = half_wave_sum(sw3[v]);
    if (col == v) {
      mine[OFF_B1 + row] = b1;
      mine[OFF_B2 + row] = b2;
      mine[OFF_W3 + row] = w3;
    }
  }
  gb3 = half_wave_sum(gb3);
  lsum = half_wave_sum(lsum);
  gb3 += __shfl_xor(gb3, 32, 64);
  lsum += __shfl_xor(lsum, 32, 64);
  if (lane == 0) {
    mine[OFF_B3] = gb3;
    mine[LOSS_COL] = lsum * inv_n;
  }
  __syncthreads();
  for (int i = threadIdx.x; i <= LOSS_COL; i += 64 * TRAIN_WAVES) {
    const float s = (lds.sums[0][i] + lds.sums[1][i]) + (lds.sums[2][i] + lds.sums[3][i]);
    if (!ATOMIC)
      out[(int64_t)blockIdx.x * PARTIAL_STRIDE + i] = s;
    else
      atomicAdd(i < LOSS_COL ? out + i : loss, s);
  }
}

// Adam (Kingma & Ba 2015) on the FP32 master parameters, then BF16 re-pack into the device block.
// The padded layer-1 inputs 10..15 stay zero.
struct AdamArgs {
  float *w, *m, *v;
  float lr, beta1, beta2, eps, bc1, bc2;
  ClosureParams* P;
};
// Contraction is spelt out, so that both kernels round alike.
__device__ __forceinline__ void adam_update(const AdamArgs& a, int i, float gi) {
#pragma clang fp contract(off)
  float* const w = a.w;
  ClosureParams* const P = a.P;
  if (i < OFF_W2T && (i % CLOSURE_IN_PAD) >= CLOSURE_IN) gi = 0.f;
  const float mi = __builtin_fmaf(a.beta1, a.m[i], (1.f - a.beta1) * gi);
  const float vi = __builtin_fmaf(a.beta2, a.v[i], (1.f - a.beta2) * gi * gi);
  a.m[i] = mi;
  a.v[i] = vi;
  float wi = w[i] - a.lr * (mi / a.bc1) / (__builtin_sqrtf(vi / a.bc2) + a.eps);
  if (i < OFF_W2T && (i % CLOSURE_IN_PAD) >= CLOSURE_IN) wi = 0.f;
  w[i] = wi;
  if (i < OFF_W2T) P->w1t[i / CLOSURE_IN_PAD][i % CLOSURE_IN_PAD] = f2bf(wi);
  else if (i < OFF_W3) P->w2t[(i - OFF_W2T) / CLOSURE_H][(i - OFF_W2T) % CLOSURE_H] = f2bf(wi);
  else if (i < OFF_B1) P->w3[i - OFF_W3] = f2bf(wi);
  else if (i < OFF_B2) P->b1[i - OFF_B1] = wi;
  else if (i < OFF_B3) P->b2[i - OFF_B2] = wi;
  else P->b3 = wi;
}

__global__ void adam_kernel(AdamArgs a, const float* __restrict__ g) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < MASTER_SIZE) adam_update(a, i, g[i]);
}

// Sums the rows of the per-block partial gradients, 64 columns per block, 16 rows at a time.  ADAM: applies them to the
// master parameters; otherwise they go to grad[1633].  The loss goes to loss[0].
template <bool ADAM>
__global__ void __launch_bounds__(1024) closure_reduce_kernel(const float* __restrict__ partials, int rows, AdamArgs a,
                                                              float* __restrict__ grad, float* __restrict__ loss) {
  __shared__ float part[16][64];
  const int col = threadIdx.x & 63, first = threadIdx.x >> 6;
  const int i = blockIdx.x * 64 + col;
  float s = 0.f;
#pragma unroll 4
  for (int r = first; r < rows; r += 16) s += partials[(int64_t)r * PARTIAL_STRIDE + i];
  part[first][col] = s;
  __syncthreads();
  if (first != 0 || i > LOSS_COL) return;
  s = 0.f;
#pragma unroll
  for (int k = 0; k < 16; ++k) s += part[k][col];
  if (i == LOSS_COL)
    loss[0] = s;
  else if (ADAM)
    adam_update(a, i, s);
  else
    grad[i] = s;
}

}  // namespace lbm355

using namespace lbm355;

namespace {
int cerr(int code, const std::string& msg) { return lbm355_set_error(code, msg.c_str()); }
int launched() {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return cerr(LBM355_ERR_LAUNCH, std::string("launch failed: ") + hipGetErrorString(e));
  return LBM355_OK;
}
// Blocks of a minibatch's gradient: one tile per wavefront up to `most` blocks, whose rows the sum then reads.
constexpr int TRAIN_MAX_BLOCKS = 512;
int train_grid(int64_t n, int most) {
  const int64_t b = ((n + 63) / 64 + TRAIN_WAVES - 1) / TRAIN_WAVES;
  return (int)(b < most ? b : most);
}
int grid_for(int64_t n, int per_block) {
  const int64_t b = (n + per_block - 1) / per_block;
  return (int)(b < 4096 ? (b > 0 ? b : 1) : 4096);
}
}  // namespace

extern "C" {

int64_t lbm355_closure_params_size(void) { return (int64_t)sizeof(ClosureParams); }
int32_t lbm355_closure_master_size(void) { return MASTER_SIZE; }

int lbm355_closure_features(const float* pi_neq, const float* density, int64_t n, float* features, void* stream) {
  if (!pi_neq || !density || !features || n < 0) return cerr(LBM355_ERR_ARG, "bad closure_features arguments");
  if (n == 0) return LBM355_OK;
  hipLaunchKernelGGL(features_kernel, dim3(grid_for(n, 256)), dim3(256), 0, (hipStream_t)stream, pi_neq, density, n,
                     features);
  return launched();
}

int lbm355_closure_forward(const void* params, const float* features, int64_t n, float* out, void* stream) {
  if (!params || !features || !out || n < 0) return cerr(LBM355_ERR_ARG, "bad closure_forward arguments");
  if (n == 0) return LBM355_OK;
  hipLaunchKernelGGL(forward_kernel, dim3(grid_for(n, 256)), dim3(256), 0, (hipStream_t)stream,
                     (const ClosureParams*)params, features, n, out);
  return launched();
}

int lbm355_closure_train_step(const void* params, const float* features, const float* targets, int64_t n,
                              float* grad, float* loss, int32_t blocks, void* stream) {
  if (!params || !features || !targets || !grad || !loss || n <= 0 || blocks <= 0)
    return cerr(LBM355_ERR_ARG, "bad closure_train_step arguments");
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(zero_kernel, dim3((MASTER_SIZE + 255) / 256), dim3(256), 0, s, grad, MASTER_SIZE);
  hipLaunchKernelGGL(zero_kernel, dim3(1), dim3(64), 0, s, loss, 1);
  hipLaunchKernelGGL(train_kernel<true>, dim3(train_grid(n, (blocks + TRAIN_WAVES - 1) / TRAIN_WAVES)),
                     dim3(64 * TRAIN_WAVES), 0, s, (const ClosureParams*)params, features, targets,
                     (const int64_t*)nullptr, n, 1.f / (float)n, grad, loss);
  return launched();
}

int64_t lbm355_closure_workspace_floats(void) { return (int64_t)TRAIN_MAX_BLOCKS * PARTIAL_STRIDE; }

int lbm355_closure_gradient(const void* params, const float* features, const float* targets, int64_t n, float* grad,
                            float* loss, float* workspace, void* stream) {
  if (!params || !features || !targets || !grad || !loss || !workspace || n <= 0)
    return cerr(LBM355_ERR_ARG, "bad closure_gradient arguments");
  hipStream_t s = (hipStream_t)stream;
  const int grid = train_grid(n, TRAIN_MAX_BLOCKS);
  hipLaunchKernelGGL(train_kernel<false>, dim3(grid), dim3(64 * TRAIN_WAVES), 0, s, (const ClosureParams*)params, features,
                     targets, (const int64_t*)nullptr, n, 1.f / (float)n, workspace, (float*)nullptr);
  hipLaunchKernelGGL(closure_reduce_kernel<false>, dim3(PARTIAL_STRIDE / 64), dim3(1024), 0, s, (const float*)workspace,
                     grid, AdamArgs{}, grad, loss);
  return launched();
}

int lbm355_closure_train_epoch(void* params, float* master, float* m, float* v, const float* features,
                               const float* targets, const int64_t* order, int64_t n, int64_t batch, float lr,
                               float beta1, float beta2, float eps, int32_t steps_done, float* losses, float* workspace,
                               void* stream) {
  if (!params || !master || !m || !v || !features || !targets || !order || !losses || !workspace || n < 0 || batch < 1 ||
      steps_done < 0)
    return cerr(LBM355_ERR_ARG, "bad closure_train_epoch arguments");
  hipStream_t s = (hipStream_t)stream;
  int32_t step = steps_done;
  for (int64_t first = 0; first < n; first += batch) {
    const int64_t k = n - first < batch ? n - first : batch;
    const int grid = train_grid(k, TRAIN_MAX_BLOCKS);
    ++step;
    const AdamArgs a = {master, m, v, lr, beta1, beta2, eps, 1.f - powf(beta1, (float)step),
                        1.f - powf(beta2, (float)step), (ClosureParams*)params};
    hipLaunchKernelGGL(train_kernel<false>, dim3(grid), dim3(64 * TRAIN_WAVES), 0, s, (const ClosureParams*)params,
                       features, targets, order + first, k, 1.f / (float)k, workspace, (float*)nullptr);
    hipLaunchKernelGGL(closure_reduce_kernel<true>, dim3(PARTIAL_STRIDE / 64), dim3(1024), 0, s, (const float*)workspace,
                       grid, a, (float*)nullptr, losses + (step - steps_done - 1));
    const int rc = launched();
    if (rc) return rc;
  }
  return LBM355_OK;
}

int lbm355_closure_adam(float* master, const float* grad, float* m, float* v, float lr, float beta1, float beta2,
                        float eps, int32_t step, void* params, void* stream) {
  if (!master || !grad || !m || !v || !params || step < 1) return cerr(LBM355_ERR_ARG, "bad closure_adam arguments");
  const AdamArgs a = {master, m, v, lr, beta1, beta2, eps, 1.f - powf(beta1, (float)step), 1.f - powf(beta2, (float)step),
                      (ClosureParams*)params};
  hipLaunchKernelGGL(adam_kernel, dim3((MASTER_SIZE + 255) / 256), dim3(256), 0, (hipStream_t)stream, a, grad);
  return launched();
}

}  // extern "C"
