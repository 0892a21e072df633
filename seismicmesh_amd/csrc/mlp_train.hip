// Forward and backward pass of the surrogate's training (FP32), fused around
// one matrix-core product.
//
// A step of `rows` network evaluations (a sample and its 2 dim shifted
// copies each) is 3 products a hidden layer: Z_l = A_{l-1} W_l^T forward,
// dA_{l-1} = dZ_l W_l and dW_l = dZ_l^T A_{l-1} backward.  k_gemm32 computes
// all three with v_mfma_f32_32x32x2_f32 (FP32 operands and accumulation) and
// takes the elementwise work into its epilogue: bias + SiLU forward (Z and A
// are written, nothing is read back), the SiLU derivative and the bias
// gradient's column sums backward (dA is never stored).  The narrow ends --
// 2 or 3 inputs, 1 output -- are plain streaming kernels.  Sums over rows go
// through per-workgroup partials added in a fixed order by one launch at the
// end (k_sum_parts), so a gradient does not depend on scheduling.
//
// Bound: the matrix cores for large batches (68 GFLOP a step of 8192
// samples; FP32 products run at 157 TFLOP/s there against 79 on the vector
// ALUs without packed instructions).  Measured on MI355X, 8192 samples, 3
// hidden layers, eikonal term: 9.02 ms before (128 x 128 tiles on the
// vector ALUs, 128-wide tiles also for the one-row products, separate
// elementwise passes), 0.90 ms now; the gradient's error against 64 bits, over
// three draws of weights and samples, 5.3e-6 to 6.3e-6 before, 1.0e-6 to
// 1.5e-6 now.
#include <algorithm>

#include "common.h"
#include "mlp_gemm.h"

namespace smk {
namespace {

constexpr int kW = kTrainWidth;
// rows of a pass (samples and their shifted copies): what the products take,
// 1 TB of workspace for three hidden layers
constexpr int64_t kMaxRows = (int64_t)1 << 27;
// hidden layers (inference takes fewer)
constexpr int kMaxLayers = 1024;

// x' of network row b * n + i: sample i scaled to the box, shifted along one
// axis for b > 0 (sm_mlp_make_inputs)
struct Inputs {
  const double *x;
  double shift[3], scale[3];
  float eik_h;
  int64_t n;
  int dim;
  __device__ inline void get(int64_t row, float *q) const {
    const int b = (int)(row / n);
    const int64_t i = row - (int64_t)b * n;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      if (c >= dim) break;
      float v = (float)((x[i * dim + c] - shift[c]) * scale[c]);
      if (b > 0 && c == (b - 1) / 2) v += (b % 2 == 1) ? eik_h : -eik_h;
      q[c] = v;
    }
  }
};

// Z0 = X W_in^T + b_in, A0 = silu(Z0): four features a lane, a row a wave.
// Bound by the two writes.
__global__ __launch_bounds__(256) void k_train_input(Inputs in, int64_t rows, const float *w,
                                                     const float *b, float *Z, float *A) {
  const int lane = threadIdx.x % 64, f = 4 * lane;
  float wv[4][3], bv[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    bv[j] = b[f + j];
#pragma unroll
    for (int c = 0; c < 3; ++c) wv[j][c] = c < in.dim ? w[(f + j) * in.dim + c] : 0.0f;
  }
  const int64_t nw = (int64_t)gridDim.x * 4;
  for (int64_t r = (int64_t)blockIdx.x * 4 + threadIdx.x / 64; r < rows; r += nw) {
    float q[3] = {0.0f, 0.0f, 0.0f};
    in.get(r, q);
    float z[4], a[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float s = wv[j][0] * q[0];
      s = fmaf(wv[j][1], q[1], s);
      s = fmaf(wv[j][2], q[2], s);
      z[j] = s + bv[j];
      a[j] = train_silu(z[j]);
    }
    *reinterpret_cast<float4 *>(Z + r * kW + f) = make_float4(z[0], z[1], z[2], z[3]);
    *reinterpret_cast<float4 *>(A + r * kW + f) = make_float4(a[0], a[1], a[2], a[3]);
  }
}

// y = A w_out + b_out: a row a wave
__global__ __launch_bounds__(256) void k_train_output(int64_t rows, const float *A,
                                                      const float *w, const float *b, float *y) {
  const int lane = threadIdx.x % 64;
  float wv[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) wv[j] = w[4 * lane + j];
  const float bo = b[0];
  const int64_t nw = (int64_t)gridDim.x * 4;
  for (int64_t r = (int64_t)blockIdx.x * 4 + threadIdx.x / 64; r < rows; r += nw) {
    const float4 a = *reinterpret_cast<const float4 *>(A + r * kW + 4 * lane);
    float s = a.x * wv[0];
    s = fmaf(a.y, wv[1], s);
    s = fmaf(a.z, wv[2], s);
    s = fmaf(a.w, wv[3], s);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (lane == 0) y[r] = s + bo;
  }
}

// dZ_L = gy w_out^T silu'(Z_L) with the partials, per chunk of rows, of
// dw_out = gy^T A_L, db_L = 1^T dZ_L and db_out = 1^T gy
__global__ __launch_bounds__(256) void k_train_output_back(int64_t rows, int64_t chunk,
                                                           const float *gy, const float *w,
                                                           const float *Z, const float *A,
                                                           float *dZ, float *p_w, float *p_b,
                                                           float *p_o) {
  __shared__ float red[4][2][kW];
  __shared__ float redo[4];
  const int lane = threadIdx.x % 64, wv = threadIdx.x / 64, f = 4 * lane;
  const float4 w4 = *reinterpret_cast<const float4 *>(w + f);
  const float wo[4] = {w4.x, w4.y, w4.z, w4.w};
  float sw[4] = {0, 0, 0, 0}, sb[4] = {0, 0, 0, 0}, so = 0.0f;
  const int64_t b = (int64_t)blockIdx.x * chunk, e = min(rows, b + chunk);
  for (int64_t r = b + wv; r < e; r += 4) {
    const float g = gy[r];
    const float4 z4 = *reinterpret_cast<const float4 *>(Z + r * kW + f);
    const float4 a4 = *reinterpret_cast<const float4 *>(A + r * kW + f);
    const float z[4] = {z4.x, z4.y, z4.z, z4.w}, a[4] = {a4.x, a4.y, a4.z, a4.w};
    float d[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float s = train_sigmoid(z[j]);
      d[j] = g * wo[j] * s * (1.0f + z[j] * (1.0f - s));
      sw[j] = fmaf(g, a[j], sw[j]);
      sb[j] += d[j];
    }
    so += g;
    *reinterpret_cast<float4 *>(dZ + r * kW + f) = make_float4(d[0], d[1], d[2], d[3]);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    red[wv][0][f + j] = sw[j];
    red[wv][1][f + j] = sb[j];
  }
  if (lane == 0) redo[wv] = so;
  __syncthreads();
  const int c = threadIdx.x;
  p_w[(int64_t)blockIdx.x * kW + c] =
      (red[0][0][c] + red[1][0][c]) + (red[2][0][c] + red[3][0][c]);
  p_b[(int64_t)blockIdx.x * kW + c] =
      (red[0][1][c] + red[1][1][c]) + (red[2][1][c] + red[3][1][c]);
  if (c == 0) p_o[blockIdx.x] = (redo[0] + redo[1]) + (redo[2] + redo[3]);
}

// partials, per chunk of rows, of dW_in = dZ_0^T X ([feature][dim])
__global__ __launch_bounds__(256) void k_train_input_back(Inputs in, int64_t rows, int64_t chunk,
                                                          const float *dZ, float *p_w) {
  __shared__ float red[4][3][kW];
  const int lane = threadIdx.x % 64, wv = threadIdx.x / 64, f = 4 * lane;
  float s[4][3] = {};
  const int64_t b = (int64_t)blockIdx.x * chunk, e = min(rows, b + chunk);
  for (int64_t r = b + wv; r < e; r += 4) {
    float q[3] = {0.0f, 0.0f, 0.0f};
    in.get(r, q);
    const float4 d4 = *reinterpret_cast<const float4 *>(dZ + r * kW + f);
    const float d[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int c = 0; c < 3; ++c) s[j][c] = fmaf(d[j], q[c], s[j][c]);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int c = 0; c < 3; ++c) red[wv][c][f + j] = s[j][c];
  __syncthreads();
  const int ft = threadIdx.x;
  for (int c = 0; c < in.dim; ++c)
    p_w[((int64_t)blockIdx.x * kW + ft) * in.dim + c] =
        (red[0][c][ft] + red[1][c][ft]) + (red[2][c][ft] + red[3][c][ft]);
}

// out[c] = sum over p of part[p * cols + c], in a fixed order, for a list of
// jobs: 64 columns a workgroup, 16 interleaved partial sums a column.
struct SumJob {
  const float *part;
  float *out;
  int32_t parts, cols;
  int32_t block0;
};
// jobs of one launch (of arguments: 32 bytes each); three layers take 10
constexpr int kMaxJobs = 36;
struct SumJobs {
  SumJob j[kMaxJobs];
  int n;
};
__global__ __launch_bounds__(1024) void k_sum_parts(SumJobs jobs) {
  __shared__ float red[16][64];
  int k = 0;
  while (k + 1 < jobs.n && (int)blockIdx.x >= jobs.j[k + 1].block0) ++k;
  const SumJob j = jobs.j[k];
  const int lane = threadIdx.x % 64, g = threadIdx.x / 64;
  const int c = ((int)blockIdx.x - j.block0) * 64 + lane;
  float s = 0.0f;
  if (c < j.cols)
    for (int p = g; p < j.parts; p += 16) s += j.part[(int64_t)p * j.cols + c];
  red[g][lane] = s;
  __syncthreads();
  if (g == 0 && c < j.cols) {
    float t = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) t += red[i][lane];
    j.out[c] = t;
  }
}

// sizes of a step and the layout of its workspace (floats)
struct Plan {
  int64_t rows, chunk;
  int nchunk, nsplit, colparts;
  bool small;
  int64_t Z, A, dZ0, dZ1, y, gy, p_dw, p_db, p_wo, p_bo, p_wi, total;
};
Plan make_plan(int64_t n, int dim, int hidden, bool eik) {
  Plan p;
  p.rows = n * (eik ? 2 * dim + 1 : 1);
  p.small = p.rows < 128 * 128;
  const int tile = p.small ? 64 : 128;
  p.colparts = (int)((p.rows + tile - 1) / tile);
  // rows per partial: enough workgroups for the chip, few enough partials
  p.chunk = std::max<int64_t>(16, (p.rows + 1023) / 1024);
  p.nchunk = (int)((p.rows + p.chunk - 1) / p.chunk);
  p.nsplit = (int)std::min<int64_t>(128, std::max<int64_t>(1, p.rows / (p.small ? 64 : 256)));
  int64_t o = 0;
  const auto take = [&](int64_t k) {
    const int64_t at = o;
    o += (k + 63) / 64 * 64;
    return at;
  };
  p.Z = take((hidden + 1) * p.rows * kW);
  p.A = take((hidden + 1) * p.rows * kW);
  p.dZ0 = take(p.rows * kW);
  p.dZ1 = take(p.rows * kW);
  p.y = take(p.rows);
  p.gy = take(p.rows);
  p.p_dw = take((int64_t)hidden * p.nsplit * kW * kW);
  p.p_db = take((int64_t)(hidden + 1) * std::max(p.colparts, p.nchunk) * kW);
  p.p_wo = take((int64_t)p.nchunk * kW);
  p.p_bo = take(p.nchunk);
  p.p_wi = take((int64_t)p.nchunk * kW * dim);
  p.total = o;
  return p;
}

}  // namespace
}  // namespace smk

using namespace smk;

extern "C" size_t sm_mlp_loss_grad_workspace(int64_t n, int in_dim, int hidden, float eik_h) {
  if (n <= 0 || n > kMaxRows / 7 || (in_dim != 2 && in_dim != 3) || hidden < 0 ||
      hidden > kMaxLayers)
    return 0;
  return (size_t)make_plan(n, in_dim, hidden, eik_h > 0.0f).total * sizeof(float);
}

extern "C" int sm_mlp_loss_grad(int64_t n, int in_dim, int hidden, const double *x,
                                const float *t, const double *shift, const double *scale,
                                float eik_h, float lam, float trunc, const float *params,
                                float *grad, float *part, void *ws, size_t ws_bytes,
                                void *stream) {
  SM_CHECK(n > 0 && n <= kMaxRows / 7 && (in_dim == 2 || in_dim == 3) && hidden >= 0 &&
               hidden <= kMaxLayers,
           SM_ERR_ARG, "mlp_loss_grad: bad size");
  SM_CHECK(x && t && shift && scale && params && grad && part && ws, SM_ERR_ARG,
           "mlp_loss_grad: null pointer");
  SM_CHECK(eik_h >= 0.0f && (lam == 0.0f || eik_h > 0.0f) && trunc >= 0.0f, SM_ERR_ARG,
           "mlp_loss_grad: the eikonal term needs eik_h > 0, the truncation be >= 0");
  SM_CHECK(((uintptr_t)params & 15) == 0 && ((uintptr_t)ws & 15) == 0, SM_ERR_ARG,
           "mlp_loss_grad: parameters and workspace must be 16-byte aligned");
  const Plan p = make_plan(n, in_dim, hidden, eik_h > 0.0f);
  SM_CHECK(ws_bytes >= (size_t)p.total * sizeof(float), SM_ERR_CAPACITY,
           "mlp_loss_grad: workspace %zu < %zu bytes", ws_bytes,
           (size_t)p.total * sizeof(float));
  hipStream_t s = stream_of(stream);
  float *w = reinterpret_cast<float *>(ws);
  // flat parameters: w_in, b_in, w_hid, b_hid, w_out, b_out
  const int64_t o_bin = (int64_t)kW * in_dim, o_wh = o_bin + kW,
                o_bh = o_wh + (int64_t)hidden * kW * kW, o_wo = o_bh + (int64_t)hidden * kW,
                o_bo = o_wo + kW;
  Inputs in;
  in.x = x;
  for (int c = 0; c < 3; ++c) {
    in.shift[c] = c < in_dim ? shift[c] : 0.0;
    in.scale[c] = c < in_dim ? scale[c] : 0.0;
  }
  in.eik_h = eik_h;
  in.n = n;
  in.dim = in_dim;
  const int64_t rows = p.rows, layer = rows * kW;
  const unsigned gr = (unsigned)std::min<int64_t>(2048, (rows + 3) / 4);
  float *Z = w + p.Z, *A = w + p.A;
  hipLaunchKernelGGL(k_train_input, dim3(gr), dim3(256), 0, s, in, rows, params, params + o_bin, Z,
                     A);
  for (int l = 1; l <= hidden; ++l) {
    GemmArgs g;
    g.M = rows;
    g.N = kW;
    g.K = kW;
    g.A = A + (l - 1) * layer;
    g.lda = kW;
    g.B = params + o_wh + (int64_t)(l - 1) * kW * kW;
    g.ldb = kW;
    g.C = Z + l * layer;
    g.ldc = kW;
    g.C2 = A + l * layer;
    g.vec = params + o_bh + (int64_t)(l - 1) * kW;
    int rc = gemm32(kEpiSilu, true, true, g, p.small, s);
    if (rc) return rc;
  }
  float *y = w + p.y, *gy = w + p.gy;
  hipLaunchKernelGGL(k_train_output, dim3(gr), dim3(256), 0, s, rows, A + hidden * layer,
                     params + o_wo, params + o_bo, y);
  SM_LAUNCH_CHECK();
  int rc = sm_mlp_sdf_loss(n, in_dim, y, t, eik_h, lam, trunc, gy, part, stream);
  if (rc) return rc;
  SumJobs jobs;
  jobs.n = 0;
  int blocks = 0;
  const auto flush = [&]() {
    if (jobs.n) hipLaunchKernelGGL(k_sum_parts, dim3(blocks), dim3(1024), 0, s, jobs);
    jobs.n = blocks = 0;
  };
  const auto sum = [&](const float *pp, int parts, int cols, float *out) {
    jobs.j[jobs.n++] = SumJob{pp, out, parts, cols, blocks};
    blocks += (cols + 63) / 64;
  };
  const int64_t dbs = (int64_t)std::max(p.colparts, p.nchunk) * kW;
  float *dz = w + p.dZ0, *dz2 = w + p.dZ1;
  hipLaunchKernelGGL(k_train_output_back, dim3(p.nchunk), dim3(256), 0, s, rows, p.chunk, gy,
                     params + o_wo, Z + hidden * layer, A + hidden * layer, dz, w + p.p_wo,
                     w + p.p_db + hidden * dbs, w + p.p_bo);
  SM_LAUNCH_CHECK();
  sum(w + p.p_wo, p.nchunk, kW, grad + o_wo);
  sum(w + p.p_bo, p.nchunk, 1, grad + o_bo);
  int dbparts = p.nchunk;
  for (int l = hidden; l >= 1; --l) {
    sum(w + p.p_db + l * dbs, dbparts, kW, grad + o_bh + (int64_t)(l - 1) * kW);
    // dW_l = dZ_l^T A_{l-1}
    GemmArgs g;
    g.M = kW;
    g.N = kW;
    g.K = rows;
    g.A = dz;
    g.lda = kW;
    g.B = A + (l - 1) * layer;
    g.ldb = kW;
    g.C = w + p.p_dw + (int64_t)(l - 1) * p.nsplit * kW * kW;
    g.ldc = kW;
    g.nsplit = p.nsplit;
    if ((rc = gemm32(kEpiPart, false, false, g, p.small, s))) return rc;
    sum(g.C, gemm32_splits(g), kW * kW, grad + o_wh + (int64_t)(l - 1) * kW * kW);
    // dZ_{l-1} = (dZ_l W_l) silu'(Z_{l-1}), and its column sums
    GemmArgs h;
    h.M = rows;
    h.N = kW;
    h.K = kW;
    h.A = dz;
    h.lda = kW;
    h.B = params + o_wh + (int64_t)(l - 1) * kW * kW;
    h.ldb = kW;
    h.C = dz2;
    h.ldc = kW;
    h.C2 = w + p.p_db + (l - 1) * dbs;
    h.vec = Z + (l - 1) * layer;
    if ((rc = gemm32(kEpiSiluBack, true, false, h, p.small, s))) return rc;
    dbparts = p.colparts;
    std::swap(dz, dz2);
    // a deep network: more sums than one launch takes (the partials of every
    // layer have their own place)
    if (jobs.n + 4 > kMaxJobs) flush();
  }
  sum(w + p.p_db, dbparts, kW, grad + o_bin);
  hipLaunchKernelGGL(k_train_input_back, dim3(p.nchunk), dim3(256), 0, s, in, rows, p.chunk, dz,
                     w + p.p_wi);
  sum(w + p.p_wi, p.nchunk, kW * in_dim, grad);
  flush();
  SM_LAUNCH_CHECK();
  return SM_OK;
}
