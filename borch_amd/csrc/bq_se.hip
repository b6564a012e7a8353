// Squeeze-excite gates in f32 for a channels-last activation (EfficientNet's MBConv):
//   pooled[n, c] = (sum over the HW pixels of x[n, p, c]) * (1 / HW)
//   z[n, j]      = silu(b1[j] + sum_c w1[j, c] * pooled[n, c])        (j < S, the squeeze width)
//   gate[n, c]   = sigmoid(b2[c] + sum_j w2t[j, c] * z[n, j])   (w2t: the expand weight transposed)
// the operation of borch's CPU runner "se" node (borch-ts/src/cpu/runner.ts:256-268:
// meanRows, gemmBiasAct(swish), gemmBiasAct(sigmoid); lib.rs:222-244 mean_rows). The gate
// multiplies the activation inside the next conv's quantizer (bq_quantize_nhwc_chscale)
// instead of the runner's scaleRows pass. Two kernels: partial sums (and maxima) over row
// chunks (the bandwidth pass), then one workgroup per image finishes the mean and runs the
// small MLP. Every sum has a fixed order: results do not depend on scheduling.
//
// The excite also gives the quantizer of the product its dynamic scale without a pass over
// x: the gate is positive and f32 rounding is monotonic, so over the pixels of (n, c)
// max |fl(x * g)| = fl(max |x| * g). The partial pass keeps max |x| per chunk and channel;
// the gate workgroup of each image writes the maximum of fl(max|x| * g) over its channels.
#include <algorithm>

#include "bq_common.h"

namespace bq {

constexpr int SE_THREADS = 256;     // the partial-sum pass
constexpr int GATE_THREADS = 1024;  // the per-image pass: 16 waves cover the squeeze outputs and channels

__device__ __forceinline__ float sigmoid_f(float v) {
  return __builtin_amdgcn_rcpf(__fadd_rn(1.0f, __builtin_amdgcn_exp2f(__fmul_rn(v, -1.4426950408889634f))));
}

// Block (n, chunk): rows [chunk * rows_per, ...) of image n; thread t sums channel group
// g = t % G (4 channels) over the rows r = t / G, t / G + TR, ... of the chunk (TR = 256 / G
// row lanes, G >= 1 groups a pass, more passes when C / 4 > 256), eight rows' loads issued
// before they are added in row order; the TR row-lane sums of a group are then added in
// lane order through LDS. partial[(n * chunks + chunk) * C + c]; with `pmax`, max |x| of the
// same rows at the same index.
__global__ __launch_bounds__(SE_THREADS) void se_partial_kernel(const float* __restrict__ x, int HW, int C,
                                                                int chunks, int rows_per,
                                                                float* __restrict__ partial,
                                                                float* __restrict__ pmax) {
  __shared__ float4 red[SE_THREADS];
  __shared__ float4 redm[SE_THREADS];
  const int n = blockIdx.x / chunks, chunk = blockIdx.x - n * chunks;
  const int r0 = chunk * rows_per, r1 = min(HW, r0 + rows_per);
  const int groups = C / 4;
  const int G = min(groups, SE_THREADS);
  const int TR = SE_THREADS / G;
  const int t = threadIdx.x;
  const int lane_r = t / G, g0 = t - lane_r * G;
  const float* xn = x + (size_t)n * HW * C;
  constexpr int U = 8;
  for (int gb = 0; gb < groups; gb += G) {
    const int g = gb + g0;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f), mx = acc;
    if (lane_r < TR && g < groups) {
      const float* xg = xn + g * 4;
      for (int r = r0 + lane_r; r < r1; r += U * TR) {
        float4 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int rr = r + u * TR;
          v[u] = rr < r1 ? *reinterpret_cast<const float4*>(xg + (size_t)rr * C) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          acc.x = __fadd_rn(acc.x, v[u].x); acc.y = __fadd_rn(acc.y, v[u].y);
          acc.z = __fadd_rn(acc.z, v[u].z); acc.w = __fadd_rn(acc.w, v[u].w);
          mx.x = fmaxf(mx.x, fabsf(v[u].x)); mx.y = fmaxf(mx.y, fabsf(v[u].y));
          mx.z = fmaxf(mx.z, fabsf(v[u].z)); mx.w = fmaxf(mx.w, fabsf(v[u].w));
        }
      }
    }
    red[t] = acc;
    redm[t] = mx;
    __syncthreads();
    if (t < G && gb + t < groups) {
      float4 s = red[t], m = redm[t];
      for (int k = 1; k < TR; ++k) {
        const float4 v = red[k * G + t], w = redm[k * G + t];
        s.x = __fadd_rn(s.x, v.x); s.y = __fadd_rn(s.y, v.y);
        s.z = __fadd_rn(s.z, v.z); s.w = __fadd_rn(s.w, v.w);
        m.x = fmaxf(m.x, w.x); m.y = fmaxf(m.y, w.y); m.z = fmaxf(m.z, w.z); m.w = fmaxf(m.w, w.w);
      }
      const size_t o = ((size_t)n * chunks + chunk) * C + (gb + t) * 4;
      *reinterpret_cast<float4*>(partial + o) = s;
      if (pmax) *reinterpret_cast<float4*>(pmax + o) = m;
    }
    __syncthreads();
  }
}

// 16 bytes of a buffer, zeros past its end (SE_OOB and up), without a branch a load.
constexpr uint32_t SE_OOB = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t se_rsrc(const float* base, size_t floats) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), (short)0, (int)(floats * 4), 0x00020000);
}
__device__ __forceinline__ float4 se_load(__amdgpu_buffer_rsrc_t r, bool in, int float4s) {
  return __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, in ? (uint32_t)float4s * 16u : SE_OOB, 0, 0));
}
__device__ __forceinline__ float4 add4(float4 a, float4 b) {
  return make_float4(__fadd_rn(a.x, b.x), __fadd_rn(a.y, b.y), __fadd_rn(a.z, b.z), __fadd_rn(a.w, b.w));
}
__device__ __forceinline__ float4 max4(float4 a, float4 b) {
  return make_float4(fmaxf(a.x, b.x), fmaxf(a.y, b.y), fmaxf(a.z, b.z), fmaxf(a.w, b.w));
}
__device__ __forceinline__ float4 fma4(float a, float4 b, float4 c) {
  return make_float4(__fmaf_rn(a, b.x, c.x), __fmaf_rn(a, b.y, c.y), __fmaf_rn(a, b.z, c.z), __fmaf_rn(a, b.w, c.w));
}

// One block per image: pooled and max |x| per channel (in LDS), z = silu(W1 pooled + b1)
// (one wave per output j, its lanes over c, a wave tree), gate = sigmoid(W2 z + b2) from the
// transposed expand weight w2t [S, C]. With `amax`: max over c of fl(max|x[n, :, c]| *
// gate[n, c]) into amax[n]. (Splitting the squeeze and the excite into two wider kernels was
// slower on every B0 layer: each small launch pays its own latency chain.)
//
// The chain of memory round trips bounds it, at most a block an image being in flight. So the
// weights come as 16-byte loads, all that a thread needs of a layer at once (up to 15 of w1,
// issued before the pooled sums they wait for, and 16 of w2t, before the barrier on z). More
// than 4 chunks or 16 terms are split over up to R row lanes a channel group of 4 (thread t:
// group t % G, row lane t / G), which meet through LDS in lane order; fewer are not, a meeting
// costing what a round trip does. Loads that no lane needs are skipped: out of range they cost
// the address unit as much (1.5-2.5 us at C <= 480).
// A call's two kernels at 32 images: C = 1152 at 7x7 19.6 -> 15.0 us, 672 at 14x14 15.2 -> 12.9,
// 480 11.5 -> 10.2, C <= 240 the same (144 at 28x28, whose 6 chunks meet, 8.7 -> 9.6), against
// 4-byte loads in batches of 20 and 32 and one thread a channel.
__global__ __launch_bounds__(GATE_THREADS) void se_gate_kernel(const float* __restrict__ partial,
                                                             const float* __restrict__ pmax, int chunks, int HW,
                                                             int C, int S, int R, const float* __restrict__ w1,
                                                             const float* __restrict__ b1,
                                                             const float* __restrict__ w2t,
                                                             const float* __restrict__ b2, float* __restrict__ gate,
                                                             float* __restrict__ amax) {
  extern __shared__ __attribute__((aligned(16))) float sm[];  // pooled [C], xmax [C], red [R > 1: 2][R][C], z [S]
  __shared__ float wmax[GATE_THREADS / 64];
  constexpr int WAVES = GATE_THREADS / 64;
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  const int G = C / 4, GW = min(G, GATE_THREADS);
  float4* const pooled = reinterpret_cast<float4*>(sm);
  float4* const xmax = pooled + G;
  float4* const red = xmax + G;  // R > 1 only (then G <= GATE_THREADS / 2: one pass over the groups)
  float* const z = sm + 2 * C + (R > 1 ? 2 * R * C : 0);
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int rl = t / GW, g0 = t - rl * GW;
  const int n = blockIdx.x;
  const float inv = __fdiv_rn(1.0f, (float)HW);

  constexpr int JW = 3, CU = 5;
  const __amdgpu_buffer_rsrc_t r1 = se_rsrc(w1, (size_t)S * C);
  float4 wv[JW][CU];
  auto load_w1 = [&](int jb, int cb) {  // outputs jb + 16 q, channel groups cb + 64 u
#pragma unroll
    for (int q = 0; q < JW; ++q)
#pragma unroll
      for (int u = 0; u < CU; ++u) {
        const int j = jb + WAVES * q, c4 = cb + 64 * u;
        wv[q][u] = zero;
        if (j < S && cb - lane + 64 * u < G) wv[q][u] = se_load(r1, c4 < G, j * G + c4);  // uniform
      }
  };
  load_w1(wave, lane);
  __builtin_amdgcn_sched_barrier(0);

  const int KL = min(R, (chunks + 3) / 4);  // row lanes that the chunks need
  const size_t image = (size_t)n * chunks * C;
  const __amdgpu_buffer_rsrc_t rs = se_rsrc(partial + image, (size_t)chunks * C);
  const __amdgpu_buffer_rsrc_t rm = se_rsrc(amax ? pmax + image : partial, amax ? (size_t)chunks * C : 0);
  for (int gb = 0; gb < G; gb += GW) {
    const int g = gb + g0;
    const bool mine = rl < KL && g < G;
    float4 s = zero, m = zero;
    for (int kb = 0; mine && kb < chunks; kb += 4 * KL) {  // four chunks' loads in flight, added in order
      float4 v[4], w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int k = kb + rl + u * KL;
        v[u] = w[u] = zero;
        if (kb + u * KL < chunks) {  // uniform
          v[u] = se_load(rs, k < chunks, k * G + g);
          w[u] = se_load(rm, k < chunks, k * G + g);
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        s = add4(s, v[u]);
        m = max4(m, w[u]);
      }
    }
    if (KL > 1) {  // uniform
      if (mine) {
        red[rl * G + g] = s;
        red[(R + rl) * G + g] = m;
      }
      __syncthreads();
      if (mine && rl == 0)
        for (int k = 1; k < KL; ++k) {
          s = add4(s, red[k * G + g]);
          m = max4(m, red[(R + k) * G + g]);
        }
    }
    if (mine && rl == 0) {
      pooled[g] = make_float4(__fmul_rn(s.x, inv), __fmul_rn(s.y, inv), __fmul_rn(s.z, inv), __fmul_rn(s.w, inv));
      xmax[g] = m;
    }
  }
  __syncthreads();

  // z: lane l of a wave takes channel groups l, l + 64, ... in order, then a fixed-order wave sum
  for (int jb = wave; jb < S; jb += WAVES * JW) {
    float acc[JW];
#pragma unroll
    for (int q = 0; q < JW; ++q) acc[q] = 0.f;
    for (int cb = lane; cb - lane < G; cb += 64 * CU) {
      if (jb != wave || cb != lane) load_w1(jb, cb);
#pragma unroll
      for (int u = 0; u < CU; ++u) {
        if (cb - lane + 64 * u >= G) break;  // uniform
        const float4 pv = cb + 64 * u < G ? pooled[cb + 64 * u] : zero;
#pragma unroll
        for (int q = 0; q < JW; ++q) {
          const float4 w = wv[q][u];
          acc[q] = __fmaf_rn(w.w, pv.w, __fmaf_rn(w.z, pv.z, __fmaf_rn(w.y, pv.y, __fmaf_rn(w.x, pv.x, acc[q]))));
        }
      }
    }
#pragma unroll
    for (int q = 0; q < JW; ++q) {
      const int j = jb + WAVES * q;
      const float v = wave_sum_fixed(acc[q]);  // the whole wave is here (the loop is per wave)
      if (lane == 0 && j < S) z[j] = silu(__fadd_rn(v, b1 ? b1[j] : 0.f));
    }
  }

  constexpr int JU = 16;
  const int JL = min(R, (S + JU - 1) / JU);  // row lanes that the terms need
  const __amdgpu_buffer_rsrc_t r2 = se_rsrc(w2t, (size_t)S * C);
  float4 ev[JU];
  auto load_w2 = [&](int jb, int g) {  // terms jb + rl + JL v
#pragma unroll
    for (int v = 0; v < JU; ++v) {
      const int j = jb + rl + JL * v;
      ev[v] = zero;
      if (jb + JL * v < S) ev[v] = se_load(r2, j < S, j * G + g);  // uniform
    }
  };
  if (rl < JL) load_w2(0, g0);
  __builtin_amdgcn_sched_barrier(0);
  __syncthreads();
  float peak = 0.f;
  for (int gb = 0; gb < G; gb += GW) {
    const int g = gb + g0;
    const bool mine = rl < JL && g < G;
    float4 acc = zero;
    for (int jb = 0; mine && jb < S; jb += JL * JU) {
      if (jb || gb) load_w2(jb, g);
#pragma unroll
      for (int v = 0; v < JU; ++v) {
        const int j = jb + rl + JL * v;
        if (jb + JL * v < S) acc = fma4(j < S ? z[j] : 0.f, ev[v], acc);
      }
    }
    if (JL > 1) {  // uniform
      if (mine) red[rl * G + g] = acc;
      __syncthreads();
      if (mine && rl == 0)
        for (int k = 1; k < JL; ++k) acc = add4(acc, red[k * G + g]);
    }
    if (mine && rl == 0) {
      const float a[4] = {acc.x, acc.y, acc.z, acc.w};
      const float4 x4 = xmax[g];
      const float xm[4] = {x4.x, x4.y, x4.z, x4.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int c = 4 * g + e;
        const float y = sigmoid_f(b2 ? __fadd_rn(a[e], b2[c]) : a[e]);
        gate[(size_t)n * C + c] = y;
        peak = fmaxf(peak, __fmul_rn(xm[e], y));
      }
    }
  }
  if (amax) {  // uniform
    peak = wave_max(peak);
    if (lane == 0) wmax[wave] = peak;
    __syncthreads();
    if (t == 0) {
      float r = wmax[0];
#pragma unroll
      for (int w = 1; w < WAVES; ++w) r = fmaxf(r, wmax[w]);
      amax[n] = r;
    }
  }
}

// Row lanes a channel group: the threads over the groups, at most 16 (each adds an LDS read to
// the meeting), one where their sums would not fit beside the rest in 64 KB of LDS.
static size_t gate_lds(int64_t C, int64_t S, int R) { return (size_t)(2 * C + S + (R > 1 ? 2 * R * C : 0)) * sizeof(float); }
static int gate_lanes(int64_t C, int64_t S) {
  const int R = (int)std::min<int64_t>(GATE_THREADS / std::min<int64_t>(C / 4, GATE_THREADS), 16);
  return gate_lds(C, S, R) + 1024 <= 64 * 1024 ? R : 1;
}

static int se_chunks(int64_t HW, int64_t C) {
  int64_t k = HW * C / 16384;
  k = std::min<int64_t>(k, std::min<int64_t>(HW, 64));
  return (int)std::max<int64_t>(k, 1);
}

// A classifier head in f32, beside the int8 path: the global average pool of a channels-last
// activation x [N, HW, C] and the Linear after it, out[n, o] = b[o] + sum_c pooled[n, c] *
// w[o, c] with pooled[n, c] = (sum over the HW pixels of x[n, p, c], in pixel order) / HW.
// One workgroup per image: the pooled vector in LDS, then a wave per output, its lanes over
// c in order and a fixed-order wave sum. For the small heads (O * C <= 65536: CIFAR
// ResNet-18's 512 -> 10) where the pool and the GEMM would be two launches of a few
// microseconds each.
constexpr int HEAD_THREADS = 256;

__global__ __launch_bounds__(HEAD_THREADS) void avgpool_linear_kernel(const float* __restrict__ x, int HW, int C,
                                                                      const float* __restrict__ w,
                                                                      const float* __restrict__ b, int O,
                                                                      float* __restrict__ out) {
  extern __shared__ float pooled[];
  const int n = blockIdx.x;
  const float* xn = x + (size_t)n * HW * C;
  // eight loads in flight before their adds / FMAs (in order): a loop of dependent round trips
  // would cost one each
  constexpr int U = 8;
  for (int c = threadIdx.x; c < C; c += HEAD_THREADS) {
    float s = 0.f;
    for (int p0 = 0; p0 < HW; p0 += U) {
      float v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = p0 + u < HW ? xn[(size_t)(p0 + u) * C + c] : 0.f;
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (p0 + u < HW) s = __fadd_rn(s, v[u]);
    }
    pooled[c] = __fdiv_rn(s, (float)HW);
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int o = wave; o < O; o += HEAD_THREADS / 64) {
    const float* wo = w + (size_t)o * C;
    float acc = 0.f;
    for (int c0 = lane; c0 < C; c0 += 64 * U) {
      float v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = c0 + 64 * u < C ? wo[c0 + 64 * u] : 0.f;
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (c0 + 64 * u < C) acc = __fmaf_rn(pooled[c0 + 64 * u], v[u], acc);
    }
    const float v = wave_sum_fixed(acc);  // the whole wave is here (the loop is per wave)
    if (lane == 0) out[(size_t)n * O + o] = b ? __fadd_rn(v, b[o]) : v;
  }
}

}  // namespace bq

using namespace bq;

extern "C" {

size_t bq_se_gate_ws_bytes(int64_t N, int64_t HW, int64_t C) {
  if (N < 0 || HW < 1 || C < 0) return 0;
  return 2 * (size_t)N * se_chunks(HW, C) * C * sizeof(float);  // partial sums, then partial maxima
}

int64_t bq_se_gate_absmax_parts(int64_t N, int64_t C) {
  if (N < 0 || C < 1) return set_error(BQ_ERR_ARG, "bq_se_gate_absmax_parts: bad sizes");
  return N;
}

int bq_se_gate_nhwc(const float* x, int64_t N, int64_t HW, int64_t C, const float* w1, const float* b1, int64_t S,
                    const float* w2t, const float* b2, float* gate, float* absmax_parts, void* ws, size_t ws_bytes,
                    bq_stream_t stream) {
  const char* what = "bq_se_gate_nhwc";
  if (N < 0 || HW < 1 || C < 4 || S < 1) return set_error(BQ_ERR_ARG, "%s: bad sizes", what);
  if (C % 4) return set_error(BQ_ERR_UNSUPPORTED, "%s: C=%lld is not a multiple of 4", what, (long long)C);
  if (N * HW * C >= ((int64_t)1 << 40) || HW > 0x7fffffff || C > 65536 || S > 65536)
    return set_error(BQ_ERR_ARG, "%s: size too large", what);
  if (N == 0) return BQ_OK;
  if (!x || !w1 || !w2t || !gate) return set_error(BQ_ERR_ARG, "%s: null pointer", what);
  if ((uintptr_t)x & 15) return set_error(BQ_ERR_ARG, "%s: x must be 16-byte aligned", what);
  const int chunks = se_chunks(HW, C);
  const size_t need = bq_se_gate_ws_bytes(N, HW, C);
  if (!ws || ws_bytes < need) return set_error(BQ_ERR_ARG, "%s: workspace %zu bytes, need %zu", what, ws_bytes, need);
  if ((uintptr_t)ws & 15) return set_error(BQ_ERR_ARG, "%s: workspace must be 16-byte aligned", what);
  if ((2 * C + S) * sizeof(float) > 64 * 1024) return set_error(BQ_ERR_UNSUPPORTED, "%s: 2 C + S too large", what);
  float* partial = (float*)ws;
  float* pmax = partial + (size_t)N * chunks * C;
  hipStream_t st = (hipStream_t)stream;
  const int rows_per = (int)((HW + chunks - 1) / chunks);
  se_partial_kernel<<<(unsigned)(N * chunks), SE_THREADS, 0, st>>>(x, (int)HW, (int)C, chunks, rows_per, partial,
                                                                   absmax_parts ? pmax : nullptr);
  if (int r = check_launch(what)) return r;
  const int R = gate_lanes(C, S);
  se_gate_kernel<<<(unsigned)N, GATE_THREADS, gate_lds(C, S, R), st>>>(partial, pmax, chunks, (int)HW, (int)C, (int)S, R,
                                                                       w1, b1, w2t, b2, gate, absmax_parts);
  return check_launch(what);
}

int bq_avgpool_linear_f32(const float* x, int64_t N, int64_t HW, int64_t C, const float* w, const float* b,
                          int64_t O, float* out, bq_stream_t stream) {
  const char* what = "bq_avgpool_linear_f32";
  if (N < 0 || HW < 1 || C < 1 || O < 1) return set_error(BQ_ERR_ARG, "%s: bad sizes", what);
  if (O * C > 65536 || C > 16384) return set_error(BQ_ERR_UNSUPPORTED, "%s: O * C = %lld (at most 65536)", what,
                                                   (long long)(O * C));
  if (N * HW * C >= ((int64_t)1 << 31) || N > 0x7fffffff) return set_error(BQ_ERR_ARG, "%s: size too large", what);
  if (N == 0) return BQ_OK;
  if (!x || !w || !out) return set_error(BQ_ERR_ARG, "%s: null pointer", what);
  avgpool_linear_kernel<<<(unsigned)N, HEAD_THREADS, (size_t)C * sizeof(float), (hipStream_t)stream>>>(
      x, (int)HW, (int)C, w, b, (int)O, out);
  return check_launch(what);
}

}  // extern "C"
