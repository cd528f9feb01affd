// Learned scheduler: the 12 -> 32 -> 32 -> 9 MLP that predicts, for each
// batched-step action, the log of the time to finish the wave. Forward,
// backward, gradient reduction and Adam are hand-written kernels; the batch
// kernel evaluates the trained network (mlp.hpp) at every step decision.
//
// There is no counterpart in the reference, whose visits always expand both
// frontiers top-down (bernaschi/.../make_stcon.c:960-1200); the network only
// reorders that work, so verdicts and distances are unchanged.
//
// Parameter layout (FC_SCHED_PARAMS floats):
//   W1[32][12] b1[32] W2[32][32] b2[32] W3[9][32] b3[9].
// Loss over n rows with row weights w_r (all 1 unless given):
//   L = 0.5 * sum_r w_r * sum_a (y[r][a] - target[r][a])^2 / sum_r w_r.
#include "engine.hpp"

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

#include "mlp.hpp"

namespace fcd {

constexpr int kP = kMlpParams;
constexpr int kOffW1 = 0;
constexpr int kOffB1 = kOffW1 + kHidden * kFeatures;
constexpr int kOffW2 = kOffB1 + kHidden;
constexpr int kOffB2 = kOffW2 + kHidden * kHidden;
constexpr int kOffW3 = kOffB2 + kHidden;
constexpr int kOffB3 = kOffW3 + kActions * kHidden;
static_assert(kOffB3 + kActions == kP, "parameter layout");

// Activations and row gradients are kept column-major (column c of an array
// with K columns at [c * np], np = n rounded up to kRowPad), so that the
// parameter kernel streams its columns along the rows.
constexpr int kRowPad = 64;
constexpr int kRowsPerBlock = 16;  // rows of one block of mlp_rows_kernel, half a wave each
constexpr int kRowThreads = kRowsPerBlock * kHidden;
inline size_t padded_rows(int n) { return ((size_t)n + kRowPad - 1) / kRowPad * kRowPad; }

// Forward pass of every row and, when T is given, the backward pass down to
// the per-row layer gradients. Half a wave takes a row, lane j its hidden
// unit j: the lane holds unit j's weights in registers (loaded once per
// block, from the canonical layout for the backward pass and from the
// mlp_t_index one, wt, for the forward pass, so that lanes read consecutive
// words), and the activations of the other units come from LDS as
// broadcasts. Each sum runs over its inputs in ascending order. 1,796
// rows take 6.6 us, bound by the weights' loads and the chain of 117
// dependent FMAs; one thread per row, each weight a scalar load, took 31 us. A block
// stages 16 rows' results in LDS and writes each column's 64 bytes together.
// Wr (nullable: all 1) holds the row weights and inv_wsum is 1 / sum_r w_r.
__global__ __launch_bounds__(kRowThreads) void mlp_rows_kernel(const float* __restrict__ w, const float* __restrict__ wt,
                                                       const float* __restrict__ X, const float* __restrict__ T,
                                                       const float* __restrict__ Wr, float inv_wsum, int n, int np,
                                                       float* __restrict__ Y, float* __restrict__ H1,
                                                       float* __restrict__ H2, float* __restrict__ D1,
                                                       float* __restrict__ D2, float* __restrict__ DY,
                                                       float* __restrict__ err) {
  constexpr int kCols = 4 * kHidden + kActions;
  __shared__ __align__(16) float s_b[kRowsPerBlock][kHidden];  // a half-wave's broadcast vector
  __shared__ float s_out[kCols][kRowsPerBlock + 1];
  const int j = (int)threadIdx.x & (kHidden - 1), k = (int)threadIdx.x / kHidden;  // unit, row of the block
  const int a = j < kActions ? j : 0;
  float w1[kFeatures], w2[kHidden], w3[kHidden], v2[kHidden], v3[kActions];
#pragma unroll
  for (int i = 0; i < kFeatures; ++i) w1[i] = wt[kOffW1 + i * kHidden + j];
#pragma unroll
  for (int i = 0; i < kHidden; ++i) w2[i] = wt[kOffW2 + i * kHidden + j];
#pragma unroll
  for (int i = 0; i < kHidden; ++i) w3[i] = wt[kOffW3 + i * kActions + a];
  if (T) {
#pragma unroll
    for (int k = 0; k < kHidden; ++k) v2[k] = w[kOffW2 + k * kHidden + j];
#pragma unroll
    for (int k = 0; k < kActions; ++k) v3[k] = w[kOffW3 + k * kHidden + j];
  }
  const float b1 = w[kOffB1 + j], b2 = w[kOffB2 + j], b3 = w[kOffB3 + a];
  float* sb = s_b[k];
  // s = fma(m[i], vector[i], s) for i = 0 .. N-1, the vector from LDS
  auto dot = [&](const float* m, auto count, float s) {
    constexpr int N = decltype(count)::value;
#pragma unroll
    for (int i = 0; i < N; i += 4) {
      const float4 b = *reinterpret_cast<const float4*>(sb + i);
      s = __fmaf_rn(m[i], b.x, s);
      if (i + 1 < N) s = __fmaf_rn(m[i + 1], b.y, s);
      if (i + 2 < N) s = __fmaf_rn(m[i + 2], b.z, s);
      if (i + 3 < N) s = __fmaf_rn(m[i + 3], b.w, s);
    }
    return s;
  };
  using N12 = std::integral_constant<int, kFeatures>;
  using N32 = std::integral_constant<int, kHidden>;
  using N9 = std::integral_constant<int, kActions>;
  // the wave's lanes write and read their half's vector in program order
  auto put = [&](float v) {
    __builtin_amdgcn_wave_barrier();
    sb[j] = v;
    __builtin_amdgcn_wave_barrier();
  };
  const int r0 = (int)blockIdx.x * kRowsPerBlock;
  const int r = r0 + k;
  const bool on = r < n;
  put(on && j < kFeatures ? X[(size_t)r * kFeatures + j] : 0.f);
  float s = dot(w1, N12{}, b1);
  const float h1 = s > 0.f ? s : 0.f;
  put(h1);
  s = dot(w2, N32{}, b2);
  const float h2 = s > 0.f ? s : 0.f;
  put(h2);
  const float y = dot(w3, N32{}, b3);
  if (on && j < kActions) Y[(size_t)r * kActions + j] = y;
  if (!T) return;  // for every thread of the launch alike
  const float wr = on && Wr ? Wr[r] : 1.f;
  const float scale = wr * inv_wsum;
  const float d = on && j < kActions ? y - T[(size_t)r * kActions + j] : 0.f;
  const float dy = d * scale;
  put(d);
  if (j == 0 && on) {
    float e = 0.f;
    for (int i = 0; i < kActions; ++i) e = __fmaf_rn(sb[i], sb[i], e);
    err[r] = 0.5f * wr * e;
  }
  put(dy);
  s = dot(v3, N9{}, 0.f);
  const float d2 = h2 > 0.f ? s : 0.f;
  put(d2);
  s = dot(v2, N32{}, 0.f);
  const float d1 = h1 > 0.f ? s : 0.f;
  s_out[j][k] = h1;
  s_out[kHidden + j][k] = h2;
  s_out[2 * kHidden + j][k] = d1;
  s_out[3 * kHidden + j][k] = d2;
  if (j < kActions) s_out[4 * kHidden + j][k] = dy;
  __syncthreads();
  for (int i = (int)threadIdx.x; i < kCols * kRowsPerBlock; i += kRowThreads) {
    const int c = i / kRowsPerBlock, q = i % kRowsPerBlock;
    float* dst = c < kHidden       ? H1 + (size_t)c * np
                 : c < 2 * kHidden ? H2 + (size_t)(c - kHidden) * np
                 : c < 3 * kHidden ? D1 + (size_t)(c - 2 * kHidden) * np
                 : c < 4 * kHidden ? D2 + (size_t)(c - 3 * kHidden) * np
                                   : DY + (size_t)(c - 4 * kHidden) * np;
    dst[r0 + q] = s_out[c][q];  // np covers the whole block of rows
  }
}

// Adam (Kingma & Ba 2015) with bias correction: c1, c2 = 1 - beta^t.
struct AdamStep {
  float* w;   // canonical parameters; null: the gradient only
  float* wt;  // the same in mlp_t_index order
  float* m;
  float* v;
  float lr, beta1, beta2, eps, c1, c2;
};

// The gradient of every parameter, summed over the rows in row order
// (deterministic), and the parameter's Adam step. A block's first wave holds
// 64 parameters (one chain of n dependent FMAs a lane, which sets the time:
// the rows' order is part of the result); its columns (at most 34: the
// upstream gradients' and the inputs') come through LDS in tiles of 256
// rows, which the other seven waves fetch a tile ahead, and a lane reads four
// rows of a column at once. The bias gradients take a column of ones: an FMA with
// 1 is the plain sum. 31 blocks; 1,796 rows take 13.7 us with the Adam
// step. One thread per parameter reading both columns from memory row by row
// took 590 us, with Adam (4.6 us) and an unread loss (4.5 us) as launches of
// their own: an epoch went from 0.63 ms to 20 us.
constexpr int kGradTile = 256;
constexpr int kGradThreads = 512;
constexpr int kGradCols = 35;  // 2 + 32 columns and the ones
constexpr int kGradBlocks = 16 + 7 + 5 + 3;

__global__ __launch_bounds__(kGradThreads) void mlp_grad_kernel(const float* __restrict__ XT, const float* __restrict__ H1,
                                                       const float* __restrict__ H2, const float* __restrict__ D1,
                                                       const float* __restrict__ D2, const float* __restrict__ DY,
                                                       int n, int np, float* __restrict__ grad, AdamStep ad) {
  constexpr int kStride = kGradTile + 4;
  constexpr int kBuf = kGradCols * kStride;
  __shared__ __align__(16) float s_col[2 * kBuf];
  // This block's parameters: na upstream columns from A, nb input columns
  // from B (0: a bias), parameter of (ca, cb) = base + ca * nb + cb.
  const int b = (int)blockIdx.x;
  const float *A, *B;
  int ca0, na, nb, base;
  if (b < 16) {
    A = D2, B = H1, ca0 = 2 * b, na = 2, nb = kHidden, base = kOffW2;
  } else if (b < 23) {
    ca0 = 5 * (b - 16);
    A = D1, B = XT, na = kHidden - ca0 < 5 ? kHidden - ca0 : 5, nb = kFeatures, base = kOffW1;
  } else if (b < 28) {
    ca0 = 2 * (b - 23);
    A = DY, B = H2, na = kActions - ca0 < 2 ? kActions - ca0 : 2, nb = kHidden, base = kOffW3;
  } else {
    const int k = b - 28;
    A = k == 0 ? D1 : k == 1 ? D2 : DY;
    B = nullptr, ca0 = 0, na = k == 2 ? kActions : kHidden, nb = 0, base = k == 0 ? kOffB1 : k == 1 ? kOffB2 : kOffB3;
  }
  const int cols = na + nb;
  const int lane = (int)threadIdx.x & 63;
  const int per = nb ? nb : 1;  // parameters of one upstream column
  const int lca = lane / per, lcb = lane % per;
  const bool mine = threadIdx.x < 64 && lca < na;
  const int oa = (mine ? lca : 0) * kStride, ob = (nb ? na + lcb : kGradCols - 1) * kStride;
  if (!nb)
    for (int i = (int)threadIdx.x; i < 2 * kGradTile; i += kGradThreads)
      s_col[(i / kGradTile) * kBuf + (kGradCols - 1) * kStride + i % kGradTile] = 1.f;
  // waves 1.. copy the columns' rows [t0, t0 + kGradTile) into buffer d
  constexpr int kLoaders = kGradThreads - 64;
  constexpr int kPer = ((kGradCols - 1) * kGradTile / 4 + kLoaders - 1) / kLoaders;
  auto fetch = [&](int t0, float* d) {
    float4 pre[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int i = k * kLoaders + (int)threadIdx.x - 64, c = i / (kGradTile / 4), r = t0 + 4 * (i % (kGradTile / 4));
      pre[k] = make_float4(0.f, 0.f, 0.f, 0.f);
      if (c < cols && r < np)
        pre[k] = *reinterpret_cast<const float4*>((c < na ? A + (size_t)(ca0 + c) * np : B + (size_t)(c - na) * np) + r);
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int i = k * kLoaders + (int)threadIdx.x - 64, c = i / (kGradTile / 4), r = 4 * (i % (kGradTile / 4));
      if (c < cols) *reinterpret_cast<float4*>(d + c * kStride + r) = pre[k];
    }
  };
  float s = 0.f;
  if (threadIdx.x >= 64) fetch(0, s_col);
  int buf = 0;
  for (int t0 = 0; t0 < n; t0 += kGradTile, buf ^= 1) {
    __syncthreads();
    if (threadIdx.x >= 64) {
      if (t0 + kGradTile < n) fetch(t0 + kGradTile, s_col + (buf ^ 1) * kBuf);
      continue;
    }
    const float* sa = s_col + buf * kBuf + oa;
    const float* sb = s_col + buf * kBuf + ob;
    const int m = n - t0 < kGradTile ? n - t0 : kGradTile;
    // two sets of registers: one set's rows are read while the other's are summed
    constexpr int kStep = 16, kQ = kStep / 4;
    float4 x0[kQ], y0[kQ], x1[kQ], y1[kQ];
    auto read = [&](float4* x, float4* y, int at) {
#pragma unroll
      for (int q = 0; q < kQ; ++q) {
        x[q] = *reinterpret_cast<const float4*>(sa + at + 4 * q);
        y[q] = *reinterpret_cast<const float4*>(sb + at + 4 * q);
      }
    };
    auto sum = [&](const float4* x, const float4* y) {
#pragma unroll
      for (int q = 0; q < kQ; ++q) {
        s = __fmaf_rn(x[q].x, y[q].x, s);
        s = __fmaf_rn(x[q].y, y[q].y, s);
        s = __fmaf_rn(x[q].z, y[q].z, s);
        s = __fmaf_rn(x[q].w, y[q].w, s);
      }
    };
    const int full = m / (2 * kStep) * (2 * kStep);
    int r = 0;
    if (full) read(x0, y0, 0);
    for (; r < full; r += 2 * kStep) {
      read(x1, y1, r + kStep);
      sum(x0, y0);
      read(x0, y0, r + 2 * kStep < full ? r + 2 * kStep : r);
      sum(x1, y1);
    }
    for (; r < m; ++r) s = __fmaf_rn(sa[r], sb[r], s);
  }
  if (!mine) return;
  const int p = base + (ca0 + lca) * per + lcb;
  grad[p] = s;
  if (!ad.w) return;
  const float gi = s;
  const float mi = ad.beta1 * ad.m[p] + (1.f - ad.beta1) * gi;
  const float vi = ad.beta2 * ad.v[p] + (1.f - ad.beta2) * gi * gi;
  ad.m[p] = mi;
  ad.v[p] = vi;
  const float mh = mi / ad.c1, vh = vi / ad.c2;
  const float wn = ad.w[p] - ad.lr * mh / (sqrtf(vh) + ad.eps);
  ad.w[p] = wn;
  ad.wt[mlp_t_index(p)] = wn;
}

// Deterministic sum of the per-row (weighted) errors times inv_wsum (one block).
__global__ __launch_bounds__(256) void mlp_loss_kernel(const float* __restrict__ err, int n, float inv_wsum,
                                                       float* __restrict__ out) {
  __shared__ float part[256];
  float s = 0.f;
  for (int r = (int)threadIdx.x; r < n; r += 256) s += err[r];
  part[threadIdx.x] = s;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) part[threadIdx.x] += part[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = part[0] * inv_wsum;
}

// Device buffers of one training / gradient call.
struct MlpBuffers {
  float *X = nullptr, *XT = nullptr, *T = nullptr, *Y = nullptr, *H1 = nullptr, *H2 = nullptr, *D1 = nullptr, *D2 = nullptr,
        *DY = nullptr, *err = nullptr, *w = nullptr, *wt = nullptr, *g = nullptr, *m = nullptr, *v = nullptr, *loss = nullptr,
        *wr = nullptr;
  float inv_wsum = 1.f;  // 1 / sum of the row weights
  ~MlpBuffers() {
    for (float* p : {X, XT, T, Y, H1, H2, D1, D2, DY, err, w, wt, g, m, v, loss, wr}) (void)hipFree(p);
  }
  // Uploads row weights (null: every row weighs 1) and sets inv_wsum.
  fc_status set_weights(const float* weight, int n, hipStream_t s) {
    double sum = 0.0;
    if (weight) {
      for (int r = 0; r < n; ++r) {
        if (!(weight[r] >= 0.f) || !std::isfinite(weight[r]))
          return fc::fail(FC_ERR_INVALID, "scheduler row weight %d is negative or not finite", r);
        sum += weight[r];
      }
      if (!(sum > 0.0)) return fc::fail(FC_ERR_INVALID, "scheduler row weights sum to zero");
      if (fcd::dev_malloc((void**)&wr, sizeof(float) * (size_t)n) != hipSuccess)
        return fc::fail(FC_ERR_NOMEM, "scheduler buffers: device allocation failed");
      FC_HIP(hipMemcpyAsync(wr, weight, sizeof(float) * (size_t)n, hipMemcpyHostToDevice, s));
    } else {
      sum = (double)n;
    }
    inv_wsum = (float)(1.0 / sum);
    return FC_OK;
  }
  fc_status alloc(int n, bool train) {
    auto A = [](float** p, size_t cnt) { return fcd::dev_malloc((void**)p, sizeof(float) * (cnt ? cnt : 1)); };
    const size_t N = (size_t)n, P = padded_rows(n);
    if (A(&X, N * kFeatures) != hipSuccess || A(&XT, P * kFeatures) != hipSuccess || A(&T, N * kActions) != hipSuccess ||
        A(&Y, N * kActions) != hipSuccess || A(&H1, P * kHidden) != hipSuccess || A(&H2, P * kHidden) != hipSuccess ||
        A(&D1, P * kHidden) != hipSuccess || A(&D2, P * kHidden) != hipSuccess || A(&DY, P * kActions) != hipSuccess ||
        A(&err, N) != hipSuccess || A(&w, kP) != hipSuccess || A(&wt, kP) != hipSuccess || A(&g, kP) != hipSuccess ||
        A(&loss, 1) != hipSuccess)
      return fc::fail(FC_ERR_NOMEM, "scheduler buffers: device allocation failed");
    if (train && (A(&m, kP) != hipSuccess || A(&v, kP) != hipSuccess))
      return fc::fail(FC_ERR_NOMEM, "scheduler buffers: device allocation failed");
    return FC_OK;
  }
};

static hipError_t launch_rows(const MlpBuffers& b, int n, bool backward, hipStream_t s) {
  const int blocks = (n + kRowsPerBlock - 1) / kRowsPerBlock;
  hipLaunchKernelGGL(mlp_rows_kernel, dim3(blocks), dim3(kRowThreads), 0, s, b.w, b.wt, b.X, backward ? b.T : nullptr, b.wr,
                     b.inv_wsum, n, (int)padded_rows(n), b.Y, b.H1, b.H2, b.D1, b.D2, b.DY, b.err);
  return hipGetLastError();
}

static hipError_t launch_grad(const MlpBuffers& b, int n, const AdamStep& ad, hipStream_t s) {
  hipLaunchKernelGGL(mlp_grad_kernel, dim3(kGradBlocks), dim3(kGradThreads), 0, s, b.XT, b.H1, b.H2, b.D1, b.D2, b.DY, n,
                     (int)padded_rows(n), b.g, ad);
  return hipGetLastError();
}

static hipError_t launch_loss(const MlpBuffers& b, int n, hipStream_t s) {
  hipLaunchKernelGGL(mlp_loss_kernel, dim3(1), dim3(256), 0, s, b.err, n, b.inv_wsum, b.loss);
  return hipGetLastError();
}

// The rows' features, row-major for the forward pass and column-major for
// the gradient (pageable host memory: the caller synchronises before x goes).
static fc_status upload_features(const MlpBuffers& b, const float* x, int n, std::vector<float>& xt, hipStream_t s) {
  const size_t np = padded_rows(n);
  xt.assign(np * kFeatures, 0.f);
  for (int r = 0; r < n; ++r)
    for (int i = 0; i < kFeatures; ++i) xt[(size_t)i * np + (size_t)r] = x[(size_t)r * kFeatures + i];
  FC_HIP(hipMemcpyAsync(b.X, x, sizeof(float) * (size_t)n * kFeatures, hipMemcpyHostToDevice, s));
  FC_HIP(hipMemcpyAsync(b.XT, xt.data(), sizeof(float) * xt.size(), hipMemcpyHostToDevice, s));
  return FC_OK;
}

// Seeded Xavier-uniform initialisation (weights), zero biases.
static void init_params(uint64_t seed, std::vector<float>& w) {
  w.assign(kP, 0.f);
  uint64_t st = seed * 0x9E3779B97F4A7C15ull + 1;
  auto uni = [&]() {
    st += 0x9E3779B97F4A7C15ull;
    uint64_t z = st;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (double)(z >> 11) * (1.0 / 9007199254740992.0);
  };
  auto fill = [&](int off, int fan_out, int fan_in) {
    const double lim = std::sqrt(6.0 / (double)(fan_in + fan_out));
    for (int i = 0; i < fan_out * fan_in; ++i) w[off + i] = (float)((2.0 * uni() - 1.0) * lim);
  };
  fill(kOffW1, kHidden, kFeatures);
  fill(kOffW2, kHidden, kHidden);
  fill(kOffW3, kActions, kHidden);
}

static fc_status set_params_device(fc_graph* g, const std::vector<float>& w) {
  g->h_mlp = w;
  // the batch kernel reads a second copy in its wave-friendly layout
  std::vector<float> wt((size_t)kP);
  for (int i = 0; i < kP; ++i) wt[(size_t)mlp_t_index(i)] = w[(size_t)i];
  FC_HIP(hipMemcpyAsync(g->d_mlp, g->h_mlp.data(), sizeof(float) * (size_t)kP, hipMemcpyHostToDevice, g->stream));
  FC_HIP(hipMemcpyAsync(g->d_mlp + kP, wt.data(), sizeof(float) * (size_t)kP, hipMemcpyHostToDevice, g->stream));
  FC_HIP(hipStreamSynchronize(g->stream));
  g->mlp_set = true;
  return FC_OK;
}

}  // namespace fcd

using namespace fcd;

// Parameters live on the device (read by the batch kernel's learned policy)
// with a host copy. Passing params == NULL and n == 0 removes them, which
// makes the learned policy unavailable again.
extern "C" fc_status fc_sched_set_params(fc_graph* g, const float* params, int32_t n) {
  fc::clear_error();
  if (!g) return fc::fail(FC_ERR_INVALID, "fc_sched_set_params: null graph");
  if (!params && n == 0) {
    g->mlp_set = false;
    return FC_OK;
  }
  if (!params || n != kP) return fc::fail(FC_ERR_INVALID, "fc_sched_set_params: expected %d parameters", kP);
  for (int32_t i = 0; i < n; ++i)
    if (!std::isfinite(params[i])) return fc::fail(FC_ERR_INVALID, "fc_sched_set_params: parameter %d is not finite", i);
  return set_params_device(g, std::vector<float>(params, params + n));
}

extern "C" fc_status fc_sched_get_params(fc_graph* g, float* params, int32_t n) {
  fc::clear_error();
  if (!g || !params) return fc::fail(FC_ERR_INVALID, "fc_sched_get_params: null argument");
  if (n != kP) return fc::fail(FC_ERR_INVALID, "fc_sched_get_params: expected %d parameters", kP);
  if (!g->mlp_set) return fc::fail(FC_ERR_INVALID, "fc_sched_get_params: no scheduler parameters are set");
  std::copy(g->h_mlp.begin(), g->h_mlp.end(), params);
  return FC_OK;
}

static fc_status check_rows(fc_graph* g, const float* x, int32_t n, const char* fn) {
  if (!g || (n > 0 && !x)) return fc::fail(FC_ERR_INVALID, "%s: null argument", fn);
  if (n <= 0) return fc::fail(FC_ERR_INVALID, "%s: need at least one row", fn);
  if (!g->mlp_set) return fc::fail(FC_ERR_INVALID, "%s: no scheduler parameters are set", fn);
  return FC_OK;
}

extern "C" fc_status fc_sched_forward(fc_graph* g, const float* x, int32_t n, float* y_out) {
  fc::clear_error();
  fc_status st = check_rows(g, x, n, "fc_sched_forward");
  if (st != FC_OK) return st;
  if (!y_out) return fc::fail(FC_ERR_INVALID, "fc_sched_forward: null output");
  MlpBuffers b;
  if ((st = b.alloc(n, false)) != FC_OK) return st;
  FC_HIP(hipMemcpyAsync(b.X, x, sizeof(float) * (size_t)n * kFeatures, hipMemcpyHostToDevice, g->stream));
  FC_HIP(hipMemcpyAsync(b.w, g->d_mlp, sizeof(float) * kP, hipMemcpyDeviceToDevice, g->stream));
  FC_HIP(hipMemcpyAsync(b.wt, g->d_mlp + kP, sizeof(float) * kP, hipMemcpyDeviceToDevice, g->stream));
  FC_HIP(launch_rows(b, n, false, g->stream));
  FC_HIP(hipMemcpyAsync(y_out, b.Y, sizeof(float) * (size_t)n * kActions, hipMemcpyDeviceToHost, g->stream));
  FC_HIP(hipStreamSynchronize(g->stream));
  return FC_OK;
}

extern "C" fc_status fc_sched_gradient(fc_graph* g, const float* x, const float* target, const float* weight,
                                       int32_t n, float* loss_out, float* grad_out) {
  fc::clear_error();
  fc_status st = check_rows(g, x, n, "fc_sched_gradient");
  if (st != FC_OK) return st;
  if (!target || !grad_out) return fc::fail(FC_ERR_INVALID, "fc_sched_gradient: null argument");
  MlpBuffers b;
  if ((st = b.alloc(n, false)) != FC_OK) return st;
  if ((st = b.set_weights(weight, n, g->stream)) != FC_OK) return st;
  std::vector<float> xt;
  if ((st = upload_features(b, x, n, xt, g->stream)) != FC_OK) return st;
  FC_HIP(hipMemcpyAsync(b.T, target, sizeof(float) * (size_t)n * kActions, hipMemcpyHostToDevice, g->stream));
  FC_HIP(hipMemcpyAsync(b.w, g->d_mlp, sizeof(float) * kP, hipMemcpyDeviceToDevice, g->stream));
  FC_HIP(hipMemcpyAsync(b.wt, g->d_mlp + kP, sizeof(float) * kP, hipMemcpyDeviceToDevice, g->stream));
  FC_HIP(launch_rows(b, n, true, g->stream));
  FC_HIP(launch_grad(b, n, AdamStep{}, g->stream));
  FC_HIP(launch_loss(b, n, g->stream));
  float loss = 0.f;
  FC_HIP(hipMemcpyAsync(grad_out, b.g, sizeof(float) * kP, hipMemcpyDeviceToHost, g->stream));
  FC_HIP(hipMemcpyAsync(&loss, b.loss, sizeof(float), hipMemcpyDeviceToHost, g->stream));
  FC_HIP(hipStreamSynchronize(g->stream));
  if (loss_out) *loss_out = loss;
  return FC_OK;
}

// Training targets of a trace row: log(cost) minus its mean over the actions.
static bool row_targets(const fc_trace_row& r, float* tgt) {
  double lc[kActions], mean = 0.0;
  for (int a = 0; a < kActions; ++a) {
    if (!(r.cost_us[a] > 0.f) || !std::isfinite(r.cost_us[a])) return false;
    lc[a] = std::log((double)r.cost_us[a]);
    mean += lc[a];
  }
  mean /= kActions;
  for (int a = 0; a < kActions; ++a) tgt[a] = (float)(lc[a] - mean);
  return true;
}

extern "C" fc_status fc_sched_train(fc_graph* g, const fc_trace_row* rows, int32_t n_rows, int32_t epochs, float lr,
                                    uint64_t seed, int32_t weighting, float* final_loss) {
  fc::clear_error();
  if (!g || (n_rows > 0 && !rows)) return fc::fail(FC_ERR_INVALID, "fc_sched_train: null argument");
  if (n_rows <= 0 || epochs <= 0 || !(lr > 0.f))
    return fc::fail(FC_ERR_INVALID, "fc_sched_train: need rows, epochs > 0 and lr > 0");
  if (weighting != FC_SCHED_WEIGHT_UNIFORM && weighting != FC_SCHED_WEIGHT_TIME)
    return fc::fail(FC_ERR_INVALID, "fc_sched_train: unknown weighting %d", weighting);
  std::vector<float> X, T, Wt;
  X.reserve((size_t)n_rows * kFeatures);
  T.reserve((size_t)n_rows * kActions);
  int32_t n = 0;
  for (int32_t i = 0; i < n_rows; ++i) {
    float tg[kActions];
    if (!row_targets(rows[i], tg)) continue;
    for (int k = 0; k < kFeatures; ++k) {
      if (!std::isfinite(rows[i].features[k])) return fc::fail(FC_ERR_INVALID, "fc_sched_train: row %d feature %d", i, k);
      X.push_back(rows[i].features[k]);
    }
    T.insert(T.end(), tg, tg + kActions);
    Wt.push_back(*std::min_element(rows[i].cost_us, rows[i].cost_us + kActions));
    ++n;
  }
  if (n == 0) return fc::fail(FC_ERR_INVALID, "fc_sched_train: no row has positive finite costs");
  if (weighting == FC_SCHED_WEIGHT_TIME) {  // each row's best remaining time over the mean of those
    double mean = 0.0;
    for (float v : Wt) mean += v;
    mean /= (double)n;
    for (float& v : Wt) v = (float)((double)v / mean);
  }
  std::vector<float> w;
  init_params(seed, w);
  MlpBuffers b;
  fc_status st = b.alloc(n, true);
  if (st != FC_OK) return st;
  if ((st = b.set_weights(weighting == FC_SCHED_WEIGHT_TIME ? Wt.data() : nullptr, n, g->stream)) != FC_OK) return st;
  std::vector<float> xt, wt((size_t)kP);
  for (int i = 0; i < kP; ++i) wt[(size_t)mlp_t_index(i)] = w[(size_t)i];
  if ((st = upload_features(b, X.data(), n, xt, g->stream)) != FC_OK) return st;
  FC_HIP(hipMemcpyAsync(b.wt, wt.data(), sizeof(float) * kP, hipMemcpyHostToDevice, g->stream));
  FC_HIP(hipMemcpyAsync(b.T, T.data(), sizeof(float) * T.size(), hipMemcpyHostToDevice, g->stream));
  FC_HIP(hipMemcpyAsync(b.w, w.data(), sizeof(float) * kP, hipMemcpyHostToDevice, g->stream));
  FC_HIP(hipMemsetAsync(b.m, 0, sizeof(float) * kP, g->stream));
  FC_HIP(hipMemsetAsync(b.v, 0, sizeof(float) * kP, g->stream));
  const float beta1 = 0.9f, beta2 = 0.999f, eps = 1e-8f;
  double c1 = 1.0, c2 = 1.0;
  for (int32_t e = 0; e < epochs; ++e) {
    FC_HIP(launch_rows(b, n, true, g->stream));
    c1 *= beta1;
    c2 *= beta2;
    FC_HIP(launch_grad(b, n, AdamStep{b.w, b.wt, b.m, b.v, lr, beta1, beta2, eps, (float)(1.0 - c1), (float)(1.0 - c2)},
                       g->stream));
  }
  // loss of the final parameters
  FC_HIP(launch_rows(b, n, true, g->stream));
  FC_HIP(launch_loss(b, n, g->stream));
  float loss = 0.f;
  FC_HIP(hipMemcpyAsync(w.data(), b.w, sizeof(float) * kP, hipMemcpyDeviceToHost, g->stream));
  FC_HIP(hipMemcpyAsync(&loss, b.loss, sizeof(float), hipMemcpyDeviceToHost, g->stream));
  FC_HIP(hipStreamSynchronize(g->stream));
  for (float v : w)
    if (!std::isfinite(v)) return fc::fail(FC_ERR_INVALID, "fc_sched_train: training diverged (lower lr)");
  if (final_loss) *final_loss = loss;
  return set_params_device(g, w);
}
