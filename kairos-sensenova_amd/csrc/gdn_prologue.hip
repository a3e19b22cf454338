// Prologue of the GatedDeltaNet layer: the inputs of the chunked op.
//
// 1. Short causal convolution over time, per channel (ShortConvolution /
//    causal_conv1d, fla modules/convolution.py:410-458, kernel :54-141), with
//    the layer's SiLU (layers/gated_deltanet.py:176-189,235-253):
//      y[t, d] = act( sum_{i<W} w[d, i] x~[t - W + 1 + i, d] + bias[d] )
//    where x~ is x inside the sequence and, before its first token, the cache
//    [N, D, W] of the previous call (slot W-1 = most recent input) or zeros.
//    fp32 accumulation, y rounded once to x's dtype.  Optionally the rounded y
//    is then L2-normalised per head of hd channels (y / sqrt(sum y^2 + 1e-6),
//    fla modules/l2norm.py:115-118), the q/k normalisation the layer asks the
//    chunked op for (use_qk_l2norm_in_kernel=True, gated_deltanet.py:283):
//    fusing it here saves the op a read and a write of q and k.
// 2. The final cache: the last W entries of [cache, x] per sequence
//    (causal_conv1d_update_states, convolution.py:539-602).
// 3. The gates (gated_deltanet.py:265-271): g = -exp(A_log) softplus(a + dt_bias)
//    in fp32 (softplus threshold 20), beta = sigmoid(b) in b's dtype (times 2
//    with allow_neg_eigval).
//
// Layout of the convolution: lane = 8 consecutive channels (one 16-byte bf16
// load), wave = 512 channels of a run of 4 or 8 consecutive tokens, whose rows
// and W - 1 halo rows it loads together.  Every kernel here is HBM-bound.
#include <algorithm>

#include "gdn_common.hpp"
#include "gdn_kernels.h"

namespace kgdn {

namespace {

constexpr int kConvWaves = 4;
// From this many (token, 512-channel group) rows on a wave takes eight tokens, below it four: the halo read
// again is smaller, but fewer waves are in flight.  Measured in bf16, four against eight tokens: 18.9 / 19.6
// us at 31,200 rows, 22.6 / 23.1 at 40,950, 29.9 / 28.9 at 65,520, 43.6 / 41.6 at 81,900, 159 / 146 at
// 327,600; in fp32 76.1 / 73.5 at 81,900, 82 / 74 at 200,000, 277 / 264 at 327,600.  Two tokens gain at most
// 0.4 us on the smallest inputs and lose from 10,000 rows on.  In bf16 with the L2 norm four everywhere: eight
// need 181 VGPRs, two waves a SIMD (181 / 163 us at 327,600 rows, 49 / 43 at 81,900).
constexpr int64_t kConvRows8 = 49152;

__device__ __forceinline__ float sigmoid_f(float z) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-z * 1.4426950408889634f));
}

// 8 channels of a runtime-typed per-channel parameter array (fp32 or bf16)
__device__ __forceinline__ void ld_chan8(const void* p, int64_t i, int dt, float (&out)[8]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) out[e] = ld_scalar(p, i + e, dt);
}

template <typename TX>
__device__ __forceinline__ void ld_row8(const TX* p, float (&out)[8]) {
  const Vec8<TX> v = ld8<TX>(p);
#pragma unroll
  for (int e = 0; e < 8; ++e) out[e] = vget<TX>(v, e);
}

// Sequence containing flattened token t: [bos, eos) and its index.
__device__ __forceinline__ void seq_of(int64_t t, const ConvArgs& a, int& n, int64_t& bos, int64_t& eos) {
  if (a.cu == nullptr) {
    n = (int)(t / a.T);
    bos = (int64_t)n * a.T;
    eos = bos + a.T;
    return;
  }
  int lo = 0, hi = a.N - 1;                        // last n with cu[n] <= t
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (a.cu[mid] <= t) lo = mid; else hi = mid - 1;
  }
  while (lo + 1 < a.N && a.cu[lo + 1] <= t) ++lo;  // skip empty sequences ending at t
  n = lo;
  bos = a.cu[lo];
  eos = a.cu[lo + 1];
}

// A wave takes R consecutive tokens of 512 channels.  Bound by HBM on large inputs and by the latency of
// one wave on small ones, so a wave sends all its R + W - 1 row loads at once: walking a run of 64 rows
// with the window in registers, each row waited for in turn, took 52 us at T = 1560, D = 5120 (now 12.5)
// and 304 us at T = 32760, D = 10240 (now 277 us = 4.8 TB/s; a plain copy reaches 5.1).  The halo rows are
// read again by the next wave, the workgroup's next, from the caches.  With the L2 norm the tokens' sums are
// reduced together: at T = 32760, D = 5120 in bf16 224 us one after another, 163 so (166 the 64-row walk).
template <typename TX, int W, int HL, int R>
__global__ __launch_bounds__(WAVE * kConvWaves) void conv1d_rows_kernel(ConvArgs a, int64_t n_runs, int fold_state) {
  // the workgroup's waves take consecutive runs of one channel group, which share their halo rows
  const unsigned ncg = (a.D + 511) / 512, block = blockIdx.y * gridDim.x + blockIdx.x;
  const int64_t run = (int64_t)(block / ncg) * kConvWaves + threadIdx.x / WAVE;
  if (run >= n_runs) return;
  const int c0 = (int)(block % ncg) * 512 + 8 * lane_id();
  const bool ok = c0 < a.D;
  const int cc = ok ? c0 : 0;                        // lanes past D load channel 0 and store nothing
  const int64_t t_begin = run * R;
  const int64_t t_stop = min(t_begin + (int64_t)R, a.total_tokens);
  const TX* x = static_cast<const TX*>(a.x);
  TX* y = static_cast<TX*>(a.y);
  constexpr int P = W - 1;
  // rows t_begin - P .. t_begin + R - 1, clamped into the tensor (a clamped row reaches no output)
  Vec8<TX> row[R + P];
#pragma unroll
  for (int i = 0; i < R + P; ++i) {
    const int64_t s = t_begin - P + i;
    row[i] = ld8<TX>(x + (s < 0 ? 0 : s < t_stop ? s : t_stop - 1) * a.D + cc);
  }
  float wt[W][8], bias[8];
#pragma unroll
  for (int q = 0; q < W; ++q) {
    float w8[8];
    if (a.w_dtype == DT_F32) ld_row8<float>(static_cast<const float*>(a.w) + (int64_t)cc * W + 8 * q, w8);
    else ld_row8<bf16>(static_cast<const bf16*>(a.w) + (int64_t)cc * W + 8 * q, w8);
#pragma unroll
    for (int e = 0; e < 8; ++e) wt[(8 * q + e) % W][(8 * q + e) / W] = w8[e];
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) bias[e] = 0.f;
  if (a.bias) ld_chan8(a.bias, cc, a.w_dtype, bias);

  int n;
  int64_t bos, eos;
  seq_of(t_begin, a, n, bos, eos);
  // the cache of sequence n, read where a window starts before the sequence: all loads in one batch
  float hc[8 * W];
  auto load_cache = [&]() {
#pragma unroll
    for (int f = 0; f < 8 * W; ++f) hc[f] = 0.f;
    if (a.h0) {
      const TX* h = static_cast<const TX*>(a.h0) + ((int64_t)n * a.D + cc) * W;
#pragma unroll
      for (int f = 0; f < 8 * W; ++f) hc[f] = to_f32(h[f]);
    }
  };
  if (t_begin - P < bos) load_cache();
  Vec8<TX> o[R];
  float ss[R] = {};
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int64_t t = t_begin + r;
    if (t >= t_stop) break;
    if (t >= eos) {
      seq_of(t, a, n, bos, eos);
      load_cache();
    }
    float in[W][8];                                  // x~[t - P + i]
#pragma unroll
    for (int i = 0; i < W; ++i)
#pragma unroll
      for (int e = 0; e < 8; ++e) in[i][e] = vget<TX>(row[r + i], e);
#pragma unroll
    for (int d = 0; d < P; ++d)                      // the sequence's d-th token: P - d inputs from the cache
      if (t - bos == d) {
#pragma unroll
        for (int i = 0; i < P - d; ++i)
#pragma unroll
          for (int e = 0; e < 8; ++e) in[i][e] = hc[e * W + d + 1 + i];
      }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float acc = bias[e];
#pragma unroll
      for (int i = 0; i < W; ++i) acc = fmaf(wt[i][e], in[i][e], acc);
      if (a.silu) acc = acc * sigmoid_f(acc);
      acc = round_to<TX>(acc);
      vset<TX>(o[r], e, acc);
      if constexpr (HL > 0) ss[r] = fmaf(acc, acc, ss[r]);
    }
    if (!ok) continue;
    if constexpr (HL == 0) st8<TX>(y + t * a.D + c0, o[r]);
    if (fold_state && t == eos - 1) {                // the final cache: the last token's own window
      TX* ht = static_cast<TX*>(a.ht) + ((int64_t)n * a.D + c0) * W;
#pragma unroll
      for (int f = 0; f < 8 * W; ++f) ht[f] = from_f32<TX>(in[f % W][f / W]);
    }
  }
  if constexpr (HL > 0) {                            // per-head L2 norm over HL lanes of 8 channels
#pragma unroll
    for (int off = HL / 2; off > 0; off >>= 1)
#pragma unroll
      for (int r = 0; r < R; ++r) ss[r] += __shfl_xor(ss[r], off, HL);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int64_t t = t_begin + r;
      const float r1 = 1.0f / __builtin_sqrtf(ss[r] + 1e-6f);
      if (t >= t_stop || !ok) break;
#pragma unroll
      for (int e = 0; e < 8; ++e) vset<TX>(o[r], e, vget<TX>(o[r], e) * r1);
      st8<TX>(y + t * a.D + c0, o[r]);
    }
  }
}

// final cache [N, D, W]: entry w = x~[eos - W + w] (x inside the sequence, else the old cache
// slot w + T, else zero), one thread per (sequence, channel)
template <typename TX>
__global__ __launch_bounds__(256) void conv_state_kernel(ConvArgs a) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)a.N * a.D) return;
  const int n = (int)(i / a.D), d = (int)(i % a.D);
  const int64_t bos = a.cu ? a.cu[n] : (int64_t)n * a.T;
  const int64_t eos = a.cu ? a.cu[n + 1] : bos + a.T;
  const int64_t T = eos - bos;
  const TX* x = static_cast<const TX*>(a.x);
  TX* ht = static_cast<TX*>(a.ht);
  for (int w = 0; w < a.W; ++w) {
    const int64_t s = eos - a.W + w;
    TX v = from_f32<TX>(0.f);
    if (s >= bos) v = x[s * a.D + d];
    else if (a.h0 && w + T < a.W) v = from_f32<TX>(ld_scalar(a.h0, i * a.W + w + T, a.x_dtype));
    ht[i * a.W + w] = v;
  }
}

__device__ __forceinline__ float softplus_f(float x) {   // torch softplus, beta 1, threshold 20
  return x > 20.f ? x : log1pf(expf(x));
}

template <typename TB>
__global__ __launch_bounds__(256) void gates_kernel(GateArgs a) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= a.rows * a.HV) return;
  const int h = (int)(i % a.HV);
  const float av = ld_scalar(a.a, i, a.a_dtype) + ld_scalar(a.dt_bias, h, a.p_dtype);
  a.g[i] = -expf(ld_scalar(a.A_log, h, a.p_dtype)) * softplus_f(av);
  const float bv = ld_scalar(a.b, i, a.b_dtype);
  float beta = round_to<TB>(1.0f / (1.0f + expf(-bv)));
  if (a.neg_eigval) beta *= 2.f;                    // exact in either dtype
  static_cast<TB*>(a.beta)[i] = from_f32<TB>(beta);
}

// fp32 copy of n values of a runtime-typed array (the folded convolution reads fp32 taps)
__global__ __launch_bounds__(256) void to_f32_kernel(const void* src, int dt, float* dst, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) dst[i] = ld_scalar(src, i, dt);
}

template <typename TX, int W, int HL, int R>
int launch_conv_rows(const ConvArgs& a, bool fold, hipStream_t s) {
  const int64_t n_runs = (a.total_tokens + R - 1) / R;
  const int64_t blocks = (n_runs + kConvWaves - 1) / kConvWaves * ((a.D + 511) / 512);
  // a row of the grid holds fewer than 2^32 threads, which 2^29 tokens of 8 channels exceed
  const int64_t row = std::min<int64_t>(blocks, 1 << 22), rows = (blocks + row - 1) / row;
  hipLaunchKernelGGL((conv1d_rows_kernel<TX, W, HL, R>), dim3((unsigned)row, (unsigned)rows), dim3(WAVE * kConvWaves),
                     0, s, a, n_runs, (int)fold);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

template <typename TX, int W>
int launch_conv_w(const ConvArgs& a, bool fold, hipStream_t s) {
  const bool r8 = a.total_tokens * ((a.D + 511) / 512) >= kConvRows8;
  switch (a.head_lanes) {
#define KGDN_CONV_CASE(HL)                                                  \
    case HL:                                                                \
      if constexpr (W == 4 && (HL == 0 || sizeof(TX) == 4))                 \
        if (r8) return launch_conv_rows<TX, W, HL, 8>(a, fold, s);          \
      return launch_conv_rows<TX, W, HL, 4>(a, fold, s);
    KGDN_CONV_CASE(0) KGDN_CONV_CASE(8) KGDN_CONV_CASE(16) KGDN_CONV_CASE(32) KGDN_CONV_CASE(64)
#undef KGDN_CONV_CASE
    default: return -2;
  }
}

template <typename TX>
int launch_conv_t(const ConvArgs& a, hipStream_t s) {
  // fixed-length sequences: the wave of a sequence's last token writes its final cache; a varlen batch may
  // hold empty sequences, which no wave visits
  const bool fold = a.ht != nullptr && a.cu == nullptr && a.total_tokens > 0;
  if (a.total_tokens > 0) {
    int rc = -2;
    switch (a.W) {
      case 1: rc = launch_conv_w<TX, 1>(a, fold, s); break;
      case 2: rc = launch_conv_w<TX, 2>(a, fold, s); break;
      case 3: rc = launch_conv_w<TX, 3>(a, fold, s); break;
      case 4: rc = launch_conv_w<TX, 4>(a, fold, s); break;
      default: return -2;
    }
    if (rc || fold) return rc;
  }
  return launch_conv_state(a, s);
}

}  // namespace

int launch_conv1d(const ConvArgs& a, hipStream_t s) {
  if (a.x_dtype == DT_BF16) return launch_conv_t<bf16>(a, s);
  if (a.x_dtype == DT_F32) return launch_conv_t<float>(a, s);
  return -2;
}

int launch_conv_state(const ConvArgs& a, hipStream_t s) {
  if (!a.ht || a.N <= 0) return 0;
  const int64_t total = (int64_t)a.N * a.D;
  if (a.x_dtype == DT_BF16)
    hipLaunchKernelGGL(conv_state_kernel<bf16>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, a);
  else if (a.x_dtype == DT_F32)
    hipLaunchKernelGGL(conv_state_kernel<float>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, a);
  else
    return -2;
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_to_f32(const void* src, int dtype, float* dst, int64_t n, hipStream_t s) {
  if (n <= 0) return 0;
  hipLaunchKernelGGL(to_f32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, src, dtype, dst, n);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_gates(const GateArgs& a, hipStream_t s) {
  const int64_t total = a.rows * a.HV;
  if (total == 0) return 0;
  const dim3 grid((unsigned)((total + 255) / 256));
  if (a.b_dtype == DT_BF16) hipLaunchKernelGGL(gates_kernel<bf16>, grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL(gates_kernel<float>, grid, dim3(256), 0, s, a);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace kgdn
