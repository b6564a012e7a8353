// Weight-only int8 (W8A32): f32 activations against an int8 weight with one f32 scale per
// output channel; the effective weight is f32(q) * scale (one rounding), the products are
// accumulated in f32 (FMA). The reference's `matmul(..., weightInt8)` (borch-ts/src/
// kernels.ts:2695-2708) for streamed/windowed weights, and its `dequantInt8` unpack pass
// (kernels.ts:1264-1274).
//
// gemv_w8a32_kernel (M <= 4, the decode shape; the MFMA kernels below take more rows):
// HBM-bound on the int8 weight — a quarter of the f32 bytes. Each wave owns RPW weight rows; a row is read as contiguous 1 KB
// wave-loads (64 lanes x 16 bytes) and every load of the wave's rows is issued before any
// arithmetic; each lane multiplies its 16 weights against the matching 16 activations
// (L1/L2-resident, reused across the wave's rows) and the wave reduces the lane sums.
#include <algorithm>

#include "bq_bf16x3.h"
#include "bq_common.h"

namespace bq {

// bq_gemm_ws_bytes(): 1024 tile counters, zero between launches, then the partial sums.
constexpr size_t W8_CNT_BYTES = 4096;
constexpr size_t W8_WS_BYTES = W8_CNT_BYTES + (size_t)416 * 4096 * 4;
constexpr uint32_t W_OOB = 0x80000000u;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t w_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

constexpr int WA_WAVES = 8;
constexpr int WA_MMAX = 16;  // activation rows bq_gemv_w8a32 takes
constexpr int WA_MPW = 4;    // activation rows the per-wave kernel takes (4096 x 4096, M = 2 / 4: 7.9 / 10.5 us)
constexpr int WA_XLDS = 16384;       // f32 activations staged through registers (64 KB of LDS)
constexpr int WA_XLDS_BIG = 32768;   // staged by a load loop after the weights (128 KB of LDS)

// The activation rows (M rows of KC * 1024 floats, K padded to whole 1 KB weight chunks) are
// staged in LDS once per workgroup and every wave reads them from there (XN = WA_XLDS: their
// loads issued before the weights' and held in registers, so that the wait for them is not a
// wait for the weights; WA_XLDS_BIG, three and four rows above 4096 values: by a loop after
// the weight loads). The register staging: one row of 4096 at 7.6 -> 7.3 us, four at 12.3 -> 11.5 us.
// CO: the products chunk by chunk as each weight chunk lands (M = 1: one row of 4096 at
// 7.0 -> 6.5 us); else row by row once every chunk has landed (M = 2..4: 8.0 / 9.0 / 10.1
// us, 0.1-0.8 us less than chunk by chunk).
template <int KC, int RPW, int XN = WA_XLDS, bool CO = false>
__global__ __launch_bounds__(WA_WAVES * 64) void gemv_w8a32_kernel(const float* __restrict__ x, const int8_t* W,
                                                                   int M, int N, int K, const float* __restrict__ sW,
                                                                   const float* __restrict__ bias,
                                                                   const float* __restrict__ res, int act,
                                                                   float* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) float xs[XN];
  constexpr int T = WA_WAVES * 64;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int row0 = (blockIdx.x * WA_WAVES + wave) * RPW;
  const int nrows = max(0, min(RPW, N - row0));  // 0 past N: every weight load out of range
  const __amdgpu_buffer_rsrc_t rw = w_rsrc(W + (size_t)min(row0, N) * K, (uint32_t)(nrows * K));
  // the activations' loads first: the wait for them (before the LDS writes) then does not
  // wait for the weight loads issued after them
  constexpr bool XREG = XN <= WA_XLDS;  // staged through registers
  constexpr int XR = XREG ? XN / 4 / T : 1;
  float4 xr[XR];
  const int k4 = K / 4;
  const int n4 = M * k4;
  if constexpr (XREG) {
#pragma unroll
    for (int r = 0; r < XR; ++r) {
      const int i = tid + r * T;
      xr[r] = i < n4 ? reinterpret_cast<const float4*>(x)[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }
  float sc[RPW];  // before the weights: the first products then wait for chunk 0 only
#pragma unroll
  for (int j = 0; j < RPW; ++j) sc[j] = j < nrows ? sW[row0 + j] : 0.f;
  v4i w[RPW][KC];
  // chunk-major, the order the products use them: chunk c waits for its own loads only
#pragma unroll
  for (int c = 0; c < KC; ++c)
#pragma unroll
    for (int j = 0; j < RPW; ++j) {
      const int k = c * 1024 + lane * 16;
      w[j][c] = load_nt16(rw, k < K ? (uint32_t)(j * K + k) : W_OOB);
    }
  __builtin_amdgcn_sched_barrier(0);
  // Row m's float4 number c*256 + l*4 + t (the t-th of lane l's four in 1 KB chunk c) is
  // stored at float4 (m*KC + c)*256 + t*64 + l, so the four reads of a chunk each take
  // 64 consecutive float4s across the wave (no bank conflicts).
  if constexpr (XREG) {
#pragma unroll
    for (int rr = 0; rr < XR; ++rr) {
      const int i = tid + rr * T;
      if (i < n4) {
        const int m = i / k4;
        const int r = i - m * k4;
        const int dst = (m * KC + (r >> 8)) * 256 + (r & 3) * 64 + ((r >> 2) & 63);
        reinterpret_cast<float4*>(xs)[dst] = xr[rr];
      }
    }
  } else {
    for (int i = tid; i < n4; i += T) {
      const int m = i / k4;
      const int r = i - m * k4;
      const int dst = (m * KC + (r >> 8)) * 256 + (r & 3) * 64 + ((r >> 2) & 63);
      reinterpret_cast<float4*>(xs)[dst] = reinterpret_cast<const float4*>(x)[i];
    }
  }
  __syncthreads();
  if constexpr (CO) {
    // Chunk by chunk, as the loads arrive: the chunk's effective weights f32(q) * scale, then
    // every row's FMAs against them (each output accumulates chunk by chunk, byte by byte).
    float acc[WA_MPW][RPW];
#pragma unroll
    for (int m = 0; m < WA_MPW; ++m)
#pragma unroll
      for (int j = 0; j < RPW; ++j) acc[m][j] = 0.f;
#pragma unroll
    for (int c = 0; c < KC; ++c) {
      const int k = c * 1024 + lane * 16;
      if (c * 1024 >= K) break;  // uniform
      float wf[RPW][16];
#pragma unroll
      for (int j = 0; j < RPW; ++j)
#pragma unroll
        for (int q = 0; q < 16; ++q)
          wf[j][q] = __fmul_rn((float)(int)(int8_t)((uint32_t)w[j][c][q >> 2] >> ((q & 3) * 8)), sc[j]);
#pragma unroll
      for (int m = 0; m < WA_MPW; ++m) {
        if (m >= M) break;  // uniform
        const float4* xp = reinterpret_cast<const float4*>(xs) + (m * KC + c) * 256 + lane;
        float xv[16];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float4 v = k < K ? xp[t * 64] : make_float4(0.f, 0.f, 0.f, 0.f);
          xv[t * 4] = v.x; xv[t * 4 + 1] = v.y; xv[t * 4 + 2] = v.z; xv[t * 4 + 3] = v.w;
        }
#pragma unroll
        for (int j = 0; j < RPW; ++j)
#pragma unroll
          for (int q = 0; q < 16; ++q) acc[m][j] = __fmaf_rn(xv[q], wf[j][q], acc[m][j]);
      }
    }
#pragma unroll
    for (int m = 0; m < WA_MPW; ++m) {
      if (m >= M) break;
#pragma unroll
      for (int j = 0; j < RPW; ++j) {
        const float s = wave_sum_fixed(acc[m][j]);  // every lane is here
        const int n = row0 + j;
        if (lane == 0 && j < nrows) {
          float v = bias ? __fadd_rn(s, bias[n]) : s;
          if (res) v = __fadd_rn(v, res[(size_t)m * N + n]);
          out[(size_t)m * N + n] = activate(v, act);
        }
      }
    }
  } else {
    for (int m = 0; m < M; ++m) {
      float acc[RPW];
#pragma unroll
      for (int j = 0; j < RPW; ++j) acc[j] = 0.f;
#pragma unroll
      for (int c = 0; c < KC; ++c) {
        const int k = c * 1024 + lane * 16;
        if (k >= K) break;
        const float4* xp = reinterpret_cast<const float4*>(xs) + (m * KC + c) * 256 + lane;
        float xv[16];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float4 v = xp[t * 64];
          xv[t * 4] = v.x; xv[t * 4 + 1] = v.y; xv[t * 4 + 2] = v.z; xv[t * 4 + 3] = v.w;
        }
#pragma unroll
        for (int j = 0; j < RPW; ++j)
#pragma unroll
          for (int q = 0; q < 16; ++q) {
            const int b = (int)(int8_t)((uint32_t)w[j][c][q >> 2] >> ((q & 3) * 8));
            acc[j] = __fmaf_rn(xv[q], __fmul_rn((float)b, sc[j]), acc[j]);
          }
      }
#pragma unroll
      for (int j = 0; j < RPW; ++j) {
        const float s = wave_sum_fixed(acc[j]);  // every lane is here
        const int n = row0 + j;
        if (lane == 0 && j < nrows) {
          float v = bias ? __fadd_rn(s, bias[n]) : s;
          if (res) v = __fadd_rn(v, res[(size_t)m * N + n]);
          out[(size_t)m * N + n] = activate(v, act);
        }
      }
    }
  }
}

// gemv_w8a32_mfma_kernel (5 <= M <= 16, short K): the products on v_mfma_f32_16x16x4_f32. A
// workgroup owns 16 weight rows; its waves split K into 64-byte chunks (wave w takes
// chunks w, w + 8, ...). Lane l holds 16 bytes of weight row l % 16 at K offset
// 64 c + 16 (l / 16) and the 16 matching floats of activation row l % 16 (zero for rows
// >= M); MFMA j of a chunk multiplies byte j of every lane's piece, so the MFMA's K index
// l / 16 stands for K offset 64 c + 16 (l / 16) + j in both operands. The effective weight
// is f32(q) * scale (one rounding, as in the kernel above); the f32 sums take another
// order, within the same f32-accumulation bound. The per-wave kernel above reads every
// activation row in every wave and does M FMAs a weight on the VALU: at M = 8, 17.3 us for
// a 4096 x 4096 weight. Partial 16 x 16 blocks meet through LDS in wave order.
constexpr int WM_ROWS = 16;
template <int CPW>  // 64-byte chunks a wave: K <= CPW * 8 * 64
__global__ __launch_bounds__(WA_WAVES * 64) void gemv_w8a32_mfma_kernel(const float* __restrict__ x, const int8_t* W,
                                                                        int M, int N, int K,
                                                                        const float* __restrict__ sW,
                                                                        const float* __restrict__ bias,
                                                                        const float* __restrict__ res, int act,
                                                                        float* __restrict__ out) {
  __shared__ float red[WA_WAVES][WM_ROWS][16];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int n0 = blockIdx.x * WM_ROWS;
  const int nrows = min(WM_ROWS, N - n0);
  const int r = lane & 15;        // weight row (A operand) and activation row (B operand) of this lane
  const int kq = (lane >> 4) * 16;  // this lane's 16-byte piece of a 64-byte chunk
  const __amdgpu_buffer_rsrc_t rw = w_rsrc(W + (size_t)n0 * K, (uint32_t)(nrows * K));  // rows past N read 0
  const bool xrow = r < M;
  // The activations in batches of up to 8 chunks (64 floats a lane in registers). The scale
  // and the first batch are issued before the weights, so that chunk c's MFMAs wait for
  // weight chunk c only (the counter drains in issue order), not for the whole stream.
  constexpr int XB = CPW < 8 ? CPW : 8;
  float4 xv[XB][4];
  auto load_x = [&](int b0) {
#pragma unroll
    for (int c = 0; c < XB; ++c) {
      const int k = (wave + WA_WAVES * (b0 + c)) * 64 + kq;
#pragma unroll
      for (int t = 0; t < 4; ++t)
        xv[c][t] = xrow && k < K ? *reinterpret_cast<const float4*>(x + (size_t)r * K + k + 4 * t)
                                 : make_float4(0.f, 0.f, 0.f, 0.f);
    }
  };
  const float sc = r < nrows ? sW[n0 + r] : 0.f;
  load_x(0);
  v4i w[CPW];
#pragma unroll
  for (int c = 0; c < CPW; ++c) {
    const int k = (wave + WA_WAVES * c) * 64 + kq;
    w[c] = load_nt16(rw, k < K ? (uint32_t)(r * K + k) : W_OOB);
  }
  __builtin_amdgcn_sched_barrier(0);  // every load above is issued before the first MFMA
  v4f acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int b0 = 0; b0 < CPW; b0 += XB) {
    if ((wave + WA_WAVES * b0) * 64 >= K) break;  // uniform across the wave
    if (b0 > 0) load_x(b0);
#pragma unroll
    for (int c = 0; c < XB; ++c) {
      if ((wave + WA_WAVES * (b0 + c)) * 64 >= K) break;  // uniform across the wave
      const float xs[16] = {xv[c][0].x, xv[c][0].y, xv[c][0].z, xv[c][0].w, xv[c][1].x, xv[c][1].y,
                            xv[c][1].z, xv[c][1].w, xv[c][2].x, xv[c][2].y, xv[c][2].z, xv[c][2].w,
                            xv[c][3].x, xv[c][3].y, xv[c][3].z, xv[c][3].w};
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const float wf = __fmul_rn((float)(int)(int8_t)((uint32_t)w[b0 + c][j >> 2] >> ((j & 3) * 8)), sc);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wf, xs[j], acc, 0, 0, 0);
      }
    }
  }
  // result register i of lane l: weight row 4 (l / 16) + i, activation row l % 16
#pragma unroll
  for (int i = 0; i < 4; ++i) red[wave][(lane >> 4) * 4 + i][lane & 15] = acc[i];
  __syncthreads();
  if (tid < WM_ROWS * 16) {
    const int row = tid >> 4;
    const int m = tid & 15;
    if (m < M && row < nrows) {
      float s = red[0][row][m];
#pragma unroll
      for (int wv = 1; wv < WA_WAVES; ++wv) s = __fadd_rn(s, red[wv][row][m]);
      float v = bias ? __fadd_rn(s, bias[n0 + row]) : s;
      if (res) v = __fadd_rn(v, res[(size_t)m * N + n0 + row]);
      out[(size_t)m * N + n0 + row] = activate(v, act);
    }
  }
}

// ------------------------------------------------- W8A32 above the decode rows: bf16 MFMA
//
// out[m, n] = act(fl(fl(acc[m, n] * s[n]) + bias[n]) + res[m, n]) with acc[m, n] =
// sum_k x[m, k] * q[n, k] accumulated in f32. The bf16 MFMA runs 16 times the f32 MFMA rate
// on this chip, and every product fits it exactly: q (|q| <= 127: 7 bits) is exact in bf16,
// and x is the exact sum of three bf16 pieces (bq_bf16x3.h), so each x * q is three exact
// products (at most 15 significant bits) that three v_mfma_f32_16x16x32_bf16 add into one f32
// accumulator: the accumulation is the only rounding before the per-channel scale, applied
// once to the sum. The reference's order (the effective weight f32(q) * s rounded per element,
// then f32 FMAs, kernels.ts:2695-2708) and this one are both within the f32-accumulation
// bound (K + 2) 2^-24 sum |x * w| of the exact result on the effective weights.
//
// The weight is the MFMA's first operand, so a lane's four results are four consecutive
// outputs of one row (16-byte stores). K goes in chunks of 64. x is loaded so that the four
// lanes g = l / 16 of a row take 64 contiguous bytes a load: lane (r = l % 16, g) holds values
// 16 t + 4 g + (0..3), t = 0..3, of row r's chunk, and MFMA step h takes t = 2 h and 2 h + 1 in
// both operands (the contracted index permuted alike in both).

constexpr int W8_WAVES = 8;  // waves of a K-split workgroup

struct W8P {
  const float* x;    // [M, K]
  const int8_t* W;   // [N, K]
  int M, N, K;
  const float* sW;   // [N]
  const float* bias; // [N] or null
  const float* res;  // [M, N] or null
  int act;
  float* out;        // [M, N]
};

// Outputs of one row that a wave takes again over the effective weights f32(q) * s: lane l's
// n .. n + 3 for the lanes of `again`, 64 lanes a sum (in a fixed order). Lanes l, l + 16, l + 32 and
// l + 48 hold the same row m; `row` is what is known of it from an earlier call (0 nothing, 1 no
// NaN, 2 a NaN). A NaN in x decides its whole row, so a row is searched for one first, and only
// rows without pay for sums: a batch that has gone NaN costs one more read of x (256 x 4096 x 4096
// 0.044 ms -> 0.09, where a lane summed each output alone 7.5), an infinity in every row the sums
// (6304 x 768 x 3072 0.11 -> 2.4 ms, 34 so).
struct W8Again {
  v4f y;
  int row;
};
__device__ __attribute__((noinline)) W8Again w8_again(const float* x, const int8_t* W, int N, int K, int m, int n, v4f y,
                                                      v4f s, int row, uint64_t again) {
  const int lane = threadIdx.x & 63;
  for (int r = 0; r < 16; ++r) {  // uniform, as every test below but the last of each row
    uint64_t todo = again & (0x0001000100010001ull << r);
    if (!todo) continue;
    const float* xr = x + (size_t)__shfl(m, __builtin_ffsll((long long)todo) - 1) * K;
    int known = __shfl(row, r);
    if (known == 0) {
      bool nan = false;
      for (int k = lane * 4; k < K; k += 256) {
        const float4 v = *reinterpret_cast<const float4*>(xr + k);
        nan = nan || __builtin_isnan(v.x) || __builtin_isnan(v.y) || __builtin_isnan(v.z) || __builtin_isnan(v.w);
      }
      known = __ballot(nan) ? 2 : 1;
    }
    if ((lane & 15) == r) row = known;
    for (; todo; todo &= todo - 1) {
      const int l = __builtin_ffsll((long long)todo) - 1;
      const int nl = __shfl(n, l);
      float a[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) a[e] = known == 2 ? __builtin_nanf("") : 0.f;
      if (known != 2) {
        float sc[4];
        const int8_t* w[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          sc[e] = __shfl(s[e], l);
          w[e] = W + (size_t)min(nl + e, N - 1) * K;
        }
        for (int k = lane * 4; k < K; k += 256) {
          const float4 v = *reinterpret_cast<const float4*>(xr + k);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint32_t q = *reinterpret_cast<const uint32_t*>(w[e] + k);
            a[e] = __fmaf_rn(v.x, __fmul_rn((float)(int8_t)(q & 0xff), sc[e]), a[e]);
            a[e] = __fmaf_rn(v.y, __fmul_rn((float)(int8_t)((q >> 8) & 0xff), sc[e]), a[e]);
            a[e] = __fmaf_rn(v.z, __fmul_rn((float)(int8_t)((q >> 16) & 0xff), sc[e]), a[e]);
            a[e] = __fmaf_rn(v.w, __fmul_rn((float)(int8_t)(q >> 24), sc[e]), a[e]);
          }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) a[e] = wave_sum_fixed(a[e]);
      }
      if (lane == l) y = (v4f){a[0], a[1], a[2], a[3]};
    }
  }
  return W8Again{y, row};
}

typedef float v4f_u __attribute__((ext_vector_type(4), aligned(4)));

// Outputs n .. n + 3 of row m from their sums; the whole wave calls it. An output whose scaled
// sum is not finite is taken again over the effective weights f32(q) * s: the split leaves NaN
// where x is infinite or rounds to a bf16 infinity, the sum of x * q can overflow where that of
// x * (q * s) does not (x = 3e36, q = 127, s = 1 / 127), and an infinite scale makes NaN of a zero
// weight. So an infinity, a NaN or an overflow comes out as f32 arithmetic on the effective
// weights gives it. So is a sum below K * 2^-103, zero aside: values below 2^-109 lose up to 2^-134
// in the split, so a larger sum at most 127 K 2^-134 < 2^-24 of itself. `row`: w8_again's, 0 where
// the lane's row is another than in the last call.
__device__ __forceinline__ void w8_store4(const W8P& p, int m, int n, v4f v, int& row) {
  const bool in = m < p.M && n < p.N;
  const size_t o = (size_t)m * p.N + n;
  v4f s = {0.f, 0.f, 0.f, 0.f}, bias = s, res = s;  // loaded together, before the test that needs the scales
  const bool whole = n + 3 < p.N;  // 16-byte accesses, which need 4-byte alignment only
  if (in) {
    if (whole) {
      s = *reinterpret_cast<const v4f_u*>(p.sW + n);
      if (p.bias) bias = *reinterpret_cast<const v4f_u*>(p.bias + n);
      if (p.res) res = *reinterpret_cast<const v4f_u*>(p.res + o);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < p.N) {
          s[e] = p.sW[n + e];
          if (p.bias) bias[e] = p.bias[n + e];
          if (p.res) res[e] = p.res[o + e];
        }
    }
  }
  uint32_t least = ~0u;  // |sum| as an integer, 0 as the largest
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    least = min(least, (__float_as_uint(v[e]) & 0x7fffffffu) - 1u);
    v[e] = __fmul_rn(v[e], s[e]);
  }
  const bool lost = least < __float_as_uint((float)p.K * 0x1p-103f) - 1u;
  const uint64_t again = __ballot(in && (lost || !__builtin_isfinite(v[0] + v[1] + v[2] + v[3])));
  if (again) {
    const W8Again a = w8_again(p.x, p.W, p.N, p.K, m, n, v, s, row, again);
    v = a.y;
    row = a.row;
  }
  if (!in) return;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (p.bias) v[e] = __fadd_rn(v[e], bias[e]);
    if (p.res) v[e] = __fadd_rn(v[e], res[e]);
    v[e] = activate(v[e], p.act);
  }
  if (whole) {
    *reinterpret_cast<v4f_u*>(p.out + o) = v;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < p.N) p.out[o + e] = v[e];
  }
}

// A lane's 16 contiguous weights (words t = 0..3 of group g: values 16 g + 4 t + (0..3)) into
// the order x is held in (word t of group g: values 16 t + 4 g + (0..3)): the 4 x 4 transpose
// of words and lane groups, by two exchanges of half waves and two of 16-lane rows.
__device__ __forceinline__ v4i w8_transpose(v4i w) {
  typedef unsigned int v2u __attribute__((ext_vector_type(2)));
  const v2u a = __builtin_amdgcn_permlane32_swap((uint32_t)w[0], (uint32_t)w[2], false, false);
  const v2u b = __builtin_amdgcn_permlane32_swap((uint32_t)w[1], (uint32_t)w[3], false, false);
  const v2u c = __builtin_amdgcn_permlane16_swap(a[0], b[0], false, false);
  const v2u d = __builtin_amdgcn_permlane16_swap(a[1], b[1], false, false);
  return (v4i){(int)c[0], (int)c[1], (int)d[0], (int)d[1]};
}

// Few rows: a workgroup owns 16 FM x 16 FN outputs over one of S slices of K, and its waves
// split the slice (wave w takes chunks w, w + WAVES, ...), each straight from memory into
// registers, PF chunks ahead; the waves' partial blocks meet through LDS in wave order, the
// slices' through the workspace in slice order (TURNS, without a workspace: this workgroup takes
// every slice in turn, which gives the same sums). As in the int8 GEMM's K split, no workgroup waits for
// another: a tile's last one (its counter) adds the slices, runs the epilogue and clears the
// counter; partials are device-scope relaxed atomics, complete before the counter's increment.
//
// What bounds it is the bytes a CU pulls through its L1, x above all (four bytes a value
// against the weight's one): 16 rows of 4096 are 256 KB in every workgroup of a grid that only
// splits N. Slices of K cut that, for the 2-3 us that the exchange of partials takes: 16 rows
// against a 4096 x 4096 weight 13.5 us unsliced, 11.1 us as 64 tiles of 16 x 64 in 4 slices
// (f32 MFMA on the unsplit rows, as below but for this K: 15.4 us). Against 32 x 64 tiles
// staged through LDS: M = 17 35.8 -> 13.0 us, M = 64 36.0 -> 19.0, M = 256 44.7 -> 36.8.
template <int FM, int FN, int PF, bool TURNS, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void w8a32_ksplit_kernel(W8P p, int S, int* cnt, uint64_t* part) {
  constexpr int T = WAVES * 64, ITEMS = FM * FN * 64, PER = (ITEMS + T - 1) / T;
  constexpr int G = TURNS ? (FM * FN == 1 ? 8 : 2) : 1;  // slices whose blocks meet at a time
  __shared__ __attribute__((aligned(16))) v4f red[G * WAVES * ITEMS];
  __shared__ int s_last;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int K = p.K;
  const int groups = TURNS ? 1 : S;  // workgroups of a tile
  const int id = xcd_order(blockIdx.x, gridDim.x);
  const int tiles_m = (p.M + 16 * FM - 1) / (16 * FM), tiles_n = (p.N + 16 * FN - 1) / (16 * FN);
  int bm, bn;
  tile_of(id / groups, tiles_m, tiles_n, bm, bn);
  const int slice = id % groups;
  const int m0 = bm * 16 * FM, n0 = bn * 16 * FN;
  const __amdgpu_buffer_rsrc_t rx = w_rsrc(p.x, (uint32_t)((size_t)p.M * K * 4));
  const __amdgpu_buffer_rsrc_t rw = w_rsrc(p.W, (uint32_t)((size_t)p.N * K));
  uint32_t xo[FM], wo[FN];  // byte offsets of this lane's rows; a row past the edge stays out of range
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int m = m0 + 16 * i + r;
    xo[i] = m < p.M ? (uint32_t)(m * K + 4 * g) * 4u : W_OOB;
  }
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int n = n0 + 16 * j + r;
    wo[j] = n < p.N ? (uint32_t)(n * K + 16 * g) : W_OOB;
  }
  float4 xb[PF][FM][4];
  v4i wb[PF][FN];
  auto load_x = [&](int s, int c) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int t = 0; t < 4; ++t)
        xb[s][i][t] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(
                                                     rx, c * 64 + 16 * t < K ? xo[i] + (c * 64 + 16 * t) * 4 : W_OOB, 0, 0));
  };
  auto load_w = [&](int s, int j, int c) {
    const uint32_t off = c * 64 + 16 * g < K ? wo[j] + c * 64 : W_OOB;
    wb[s][j] = FM == 1 ? load_nt16(rw, off) : __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rw, off, 0, 0));
  };
  v4f acc[FM][FN];
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
  };
  // A chunk's products, its registers taking chunk `next` (`more`: there is one) as they fall free.
  auto products = [&](int s, bool more, int next) __attribute__((always_inline)) {
    Split8 a[2][FM];  // x is split first
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < FM; ++i) a[h][i] = split8(xb[s][i][2 * h], xb[s][i][2 * h + 1]);
    if (more) {
      load_x(s, next);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const v4i w = w8_transpose(wb[s][j]);
      if (more) load_w(s, j, next);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const v8bf b = i8x8_bf16((uint32_t)w[2 * h], (uint32_t)w[2 * h + 1]);
#pragma unroll
        for (int i = 0; i < FM; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a[h][i].p3, acc[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < FM; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a[h][i].p2, acc[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < FM; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a[h][i].p1, acc[i][j], 0, 0, 0);
      }
    }
  };
  auto put = [&](int at) {  // this wave's blocks, as those of slice `at` of the G
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) red[(((at * WAVES + wave) * FM + i) * FN + j) * 64 + lane] = acc[i][j];
  };
  v4f sum[PER];
  auto meet = [&](int n, bool first) {  // n slices' blocks, the waves of each in order
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int e = tid + u * T;
      if (ITEMS % T == 0 || e < ITEMS)
        for (int at = 0; at < n; ++at) {
          const v4f* from = red + at * WAVES * ITEMS + e;
          v4f v = from[0];
#pragma unroll
          for (int w = 1; w < WAVES; ++w) v += from[w * ITEMS];
          sum[u] = first && at == 0 ? v : sum[u] + v;
        }
    }
  };
  const int KT = (K + 63) / 64, per = (KT + S - 1) / S;
  clear();
  if constexpr (TURNS) {
    // every slice in this workgroup, the loads running on from one slice into the next; all waves
    // have chunks in every slice but, maybe, the last (slices hold at least a chunk a wave)
    int q = 0, c = wave, nq = 0, nc = wave;  // the chunk at hand and the next one to load
    auto forth = [&](int& sl, int& ch) {
      ch += WAVES;
      if (ch >= min(KT, (sl + 1) * per)) ch = ++sl * per + wave;
    };
    const auto valid = [&](int sl, int ch) { return sl < S && ch < min(KT, (sl + 1) * per); };
#pragma unroll
    for (int s = 0; s < PF; ++s) {
      if (!valid(nq, nc)) break;  // uniform across the wave, as below
#pragma unroll
      for (int j = 0; j < FN; ++j) load_w(s, j, nc);
      load_x(s, nc);
      forth(nq, nc);
    }
    __builtin_amdgcn_sched_barrier(0);
    while (valid(q, c)) {
#pragma unroll
      for (int s = 0; s < PF; ++s) {
        if (!valid(q, c)) break;
        products(s, valid(nq, nc), nc);
        if (valid(nq, nc)) forth(nq, nc);
        const int was = q;
        forth(q, c);
        if (q != was && q < S) {  // slice `was` is done and another follows
          put(was % G);
          clear();
          if (was % G == G - 1) {
            __syncthreads();
            meet(G, was < G);
            __syncthreads();
          }
        }
      }
    }
    put((S - 1) % G);
    __syncthreads();
    meet((S - 1) % G + 1, S <= G);
  } else {
    const int c_begin = slice * per, c_end = min(KT, c_begin + per);
#pragma unroll
    for (int s = 0; s < PF; ++s) {
      const int c = c_begin + wave + s * WAVES;
      if (c >= c_end) break;  // uniform across the wave
#pragma unroll
      for (int j = 0; j < FN; ++j) load_w(s, j, c);
      load_x(s, c);
    }
    __builtin_amdgcn_sched_barrier(0);  // every load above is issued before the first product
    for (int c0 = c_begin + wave; c0 < c_end; c0 += WAVES * PF) {
#pragma unroll
      for (int s = 0; s < PF; ++s) {
        const int c = c0 + s * WAVES, next = c + WAVES * PF;
        if (c >= c_end) break;
        products(s, next < c_end, next);
      }
    }
    put(0);
    __syncthreads();
    meet(1, true);
  }
  if (groups > 1) {
    const int tile = bm * tiles_n + bn;
    uint64_t* const mine = part + (size_t)(tile * S + slice) * ITEMS * 2;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int e = tid + u * T;
      if (ITEMS % T == 0 || e < ITEMS)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          __hip_atomic_store(mine + h * ITEMS + e,
                             (uint64_t)__float_as_uint(sum[u][2 * h]) | (uint64_t)__float_as_uint(sum[u][2 * h + 1]) << 32,
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every partial store of this lane has completed
    __syncthreads();
    if (tid == 0)
      s_last = __hip_atomic_fetch_add(cnt + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == S - 1;
    __syncthreads();
    if (!s_last) return;  // uniform across the workgroup
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int e = tid + u * T;
      if (ITEMS % T == 0 || e < ITEMS) {
        v4f v = {0.f, 0.f, 0.f, 0.f};
        const uint64_t* from = part + (size_t)tile * S * ITEMS * 2 + e;
        for (int s0 = 0; s0 < S; s0 += 4) {  // four slices' loads in flight
          uint64_t w[4][2];
#pragma unroll
          for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int h = 0; h < 2; ++h)
              w[s][h] = s0 + s < S ? __hip_atomic_load(const_cast<uint64_t*>(from) + (size_t)((s0 + s) * 2 + h) * ITEMS,
                                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                                   : 0;
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            if (s0 + s >= S) break;
            const v4f x = {__uint_as_float((uint32_t)w[s][0]), __uint_as_float((uint32_t)(w[s][0] >> 32)),
                           __uint_as_float((uint32_t)w[s][1]), __uint_as_float((uint32_t)(w[s][1] >> 32))};
            v = s0 + s ? v + x : x;
          }
        }
        sum[u] = v;
      }
    }
    if (tid == 0) __hip_atomic_store(cnt + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    const int e = tid + u * T;
    const int l = e & 63, j = (e >> 6) % FN, i = (e >> 6) / FN;
    int row = 0;
    if (ITEMS % T == 0 || e < ITEMS) w8_store4(p, m0 + 16 * i + (l & 15), n0 + 16 * j + 4 * (l >> 4), sum[u], row);
  }
}

// Many rows: a workgroup of WAVES waves owns 16 FM WAVES x 16 FN outputs, each wave 16 FM
// rows over all the columns. A wave's rows are its own, so x goes straight from memory into
// registers and is split there once; the weight chunk, which the waves share, is expanded
// to bf16 once a workgroup into one of two LDS buffers (128-byte rows, 16-byte pieces XORed by
// row bits so that a fragment read's 16 rows cover all 64 banks), one barrier a chunk: the next
// chunk's weights are expanded and stored between this chunk's MFMAs. 16 rows a wave keep the
// registers at 128, four waves a SIMD, whose splits (5.5 VALU a value of x) then run under each
// other's MFMAs; 32 rows a wave (two waves a SIMD) measured 10-40% slower, and so did
// fragments read one at a time or all eight ahead. Against x staged through LDS as its three
// planes: 6304 x 3072 x 768 114 -> 99 us, 6304 x 768 x 3072 138 -> 104, 2048^3 72 -> 53,
// 4096^3 380 -> 334 us (1.23 PFLOP/s of bf16 products; a bf16 library product of 8192^3
// runs at 1.13 here). MFMAs and splits alone would take about half of it.
__device__ __forceinline__ int w8_lds_off(int row, int c) { return row * 128 + ((c ^ ((row >> 1) & 7)) << 4); }

template <int FM, int FN, int WAVES>
__global__ __launch_bounds__(WAVES * 64, 4) void w8a32_tile_kernel(W8P p) {
  constexpr int BM = 16 * FM * WAVES, BN = 16 * FN, T = WAVES * 64;
  constexpr int RW = BN * 4 / T;  // 16-byte weight pieces a thread and chunk
  static_assert(RW * T == BN * 4, "whole pieces");
  constexpr int STAGE = BN * 128;
  __shared__ __attribute__((aligned(16))) unsigned char lds[2 * STAGE];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int K = p.K, KT = (K + 63) / 64;
  int bm, bn;
  tile_of(xcd_order(blockIdx.x, gridDim.x), (p.M + BM - 1) / BM, (p.N + BN - 1) / BN, bm, bn);
  const int m0 = bm * BM + wave * 16 * FM, n0 = bn * BN;
  const __amdgpu_buffer_rsrc_t rx = w_rsrc(p.x, (uint32_t)((size_t)p.M * K * 4));
  const __amdgpu_buffer_rsrc_t rw = w_rsrc(p.W, (uint32_t)((size_t)p.N * K));
  uint32_t xo[FM];  // byte offset of this lane's row and quad; a row past M stays out of range
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int m = m0 + 16 * i + r;
    xo[i] = m < p.M ? (uint32_t)(m * K + 4 * g) * 4u : W_OOB;
  }
  float4 xb[2][FM][4];
  v4i wq[RW];
  auto load_x = [&](int s, int c) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int t = 0; t < 4; ++t)
        xb[s][i][t] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(
                                                     rx, c * 64 + 16 * t < K ? xo[i] + (c * 64 + 16 * t) * 4 : W_OOB, 0, 0));
  };
  auto load_w = [&](int c) {
#pragma unroll
    for (int e = 0; e < RW; ++e) {
      const int i = tid + e * T, n = n0 + (i >> 2), k = c * 64 + (i & 3) * 16;
      const uint32_t off = n < p.N && k < K ? (uint32_t)(n * K + k) : W_OOB;
      wq[e] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rw, off, 0, 0));
    }
  };
  auto store_w = [&](int buf) {
    unsigned char* st = lds + buf * STAGE;
#pragma unroll
    for (int e = 0; e < RW; ++e) {
      const int i = tid + e * T, row = i >> 2, t = i & 3;  // values 16 t + 4 g + (0..3): group g's half t % 2 of step t / 2
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<uint2*>(st + w8_lds_off(row, 2 * q + (t >> 1)) + (t & 1) * 8) = i8x4_bf16((uint32_t)wq[e][q]);
    }
  };
  v4f acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
  load_w(0);
  load_x(0, 0);
  store_w(0);
  load_w(1);  // past K: zeros
  auto chunk = [&](int c, int s) {
    __syncthreads();  // chunk c's weights are stored; nobody reads the other buffer any more
    load_x(s ^ 1, c + 1);
    __builtin_amdgcn_sched_barrier(0);  // issued here, not sunk to its use
    const unsigned char* st = lds + (c & 1) * STAGE;
    constexpr int NB = 4;  // weight fragments read ahead of their products
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      v8bf b[NB];
      Split8 a[FM];
#pragma unroll
      for (int j0 = 0; j0 < FN; j0 += NB) {
#pragma unroll
        for (int j = 0; j < NB; ++j) b[j] = *reinterpret_cast<const v8bf*>(st + w8_lds_off(16 * (j0 + j) + r, 2 * g + h));
        if (j0 == 0) {
#pragma unroll
          for (int i = 0; i < FM; ++i) a[i] = split8(xb[s][i][2 * h], xb[s][i][2 * h + 1]);
        }
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int i = 0; i < FM; ++i)
            acc[i][j0 + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a[i].p3, acc[i][j0 + j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int i = 0; i < FM; ++i)
            acc[i][j0 + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a[i].p2, acc[i][j0 + j], 0, 0, 0);
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int i = 0; i < FM; ++i)
            acc[i][j0 + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[j], a[i].p1, acc[i][j0 + j], 0, 0, 0);
      }
      if (h == 0) {
        store_w((c & 1) ^ 1);
        load_w(c + 2);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  for (int c = 0; c < KT; c += 2) {
    chunk(c, 0);
    if (c + 1 < KT) chunk(c + 1, 1);
  }
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    int row = 0;
#pragma unroll
    for (int j = 0; j < FN; ++j) w8_store4(p, m0 + 16 * i + r, n0 + 16 * j + 4 * g, acc[i][j], row);
  }
}

// w[n, k] = f32(q[n, k]) * s[n] (one rounding), four elements a thread.
__global__ __launch_bounds__(256) void dequant_i8_kernel(const int8_t* __restrict__ q, int64_t N, int64_t K,
                                                         const float* __restrict__ s, float* __restrict__ w) {
  const int64_t total = N * K;
  for (int64_t e = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4; e < total; e += (int64_t)gridDim.x * 256 * 4) {
    if (e + 3 < total && (K & 3) == 0) {
      const uint32_t v = *reinterpret_cast<const uint32_t*>(q + e);
      const float sc = s[e / K];
      *reinterpret_cast<float4*>(w + e) =
          make_float4(__fmul_rn((float)(int8_t)(v & 0xff), sc), __fmul_rn((float)(int8_t)((v >> 8) & 0xff), sc),
                      __fmul_rn((float)(int8_t)((v >> 16) & 0xff), sc), __fmul_rn((float)(int8_t)(v >> 24), sc));
    } else {
      for (int64_t i = e; i < e + 4 && i < total; ++i) w[i] = __fmul_rn((float)q[i], s[i / K]);
    }
  }
}

// The per-wave kernel (M <= WA_MPW, K <= 8192): KC the weight chunks of a row; the activations
// through registers where they fit (all but three and four rows above 4096 values).
static void launch_gemv_w8a32(const float* x, const int8_t* W, int m, int n, int k, const float* sW,
                              const float* bias, const float* res, int act, float* out, hipStream_t st) {
  constexpr int RPW = 2;
  const unsigned grid = (unsigned)((n + WA_WAVES * RPW - 1) / (WA_WAVES * RPW));
  auto go = [&](auto kernel) {
    kernel<<<grid, WA_WAVES * 64, 0, st>>>(x, W, m, n, k, sW, bias, res, act, out);
  };
  if (k <= 1024) m == 1 ? go(gemv_w8a32_kernel<1, RPW, WA_XLDS, true>) : go(gemv_w8a32_kernel<1, RPW>);
  else if (k <= 2048) m == 1 ? go(gemv_w8a32_kernel<2, RPW, WA_XLDS, true>) : go(gemv_w8a32_kernel<2, RPW>);
  else if (k <= 4096) m == 1 ? go(gemv_w8a32_kernel<4, RPW, WA_XLDS, true>) : go(gemv_w8a32_kernel<4, RPW>);
  else if (m == 1) go(gemv_w8a32_kernel<8, RPW, WA_XLDS, true>);
  else if (m == 2) go(gemv_w8a32_kernel<8, RPW>);
  else go(gemv_w8a32_kernel<8, RPW, WA_XLDS_BIG>);
}

struct W8Ws {
  void* ptr;
  size_t bytes;
};
// Slices of K of an output block of 16 fm rows: up to 256 workgroups, each slice at least a chunk a wave.
static int w8a32_slices(const W8P& p, int fm, int fn) {
  const int64_t tiles = (int64_t)((p.M + 16 * fm - 1) / (16 * fm)) * ((p.N + 16 * fn - 1) / (16 * fn));
  const int KT = (p.K + 63) / 64;
  int S = std::max(1, std::min((int)(256 / tiles), KT / W8_WAVES));
  const int per = std::max(1, (KT + S - 1) / S);  // K = 0 has one empty slice
  S = std::max(1, (KT + per - 1) / per);  // no empty slice
  const bool fits = (size_t)tiles * S * fm * fn * 1024 <= W8_WS_BYTES - W8_CNT_BYTES && tiles * 4 <= (int64_t)W8_CNT_BYTES;
  return fits ? S : 1;
}
template <int FM, int FN, int PF, bool TURNS = false, int WAVES = W8_WAVES>
static void launch_w8a32_blocks(const W8P& p, int S, const W8Ws& ws, hipStream_t st) {
  const unsigned tiles = (unsigned)(((p.M + 16 * FM - 1) / (16 * FM)) * ((p.N + 16 * FN - 1) / (16 * FN)));
  const bool split = !TURNS && S > 1;
  w8a32_ksplit_kernel<FM, FN, PF, TURNS, WAVES><<<split ? tiles * S : tiles, WAVES * 64, 0, st>>>(
      p, S, split ? static_cast<int*>(ws.ptr) : nullptr,
      split ? reinterpret_cast<uint64_t*>(static_cast<char*>(ws.ptr) + W8_CNT_BYTES) : nullptr);
}
// Without a workspace the slices run in turn, in blocks small enough for the chip (the block's
// shape does not change an output's sum, the slices do). 5 to 16 rows: one 16 x 16 block a
// workgroup, chunks loaded one ahead, or two where slices give the waves unequal counts (16 x
// 4096 x 4096 12.8 us against 13.9, 5 x 768 x 3072 9.3 against 10.2; f32 MFMA on the unsplit rows
// 15.4 and 8.5). More rows: 32 x 32, or 32 x 64 in place of more than one round of those (128 x 3000
// x 1520 13.1 us, 19.7 as 32 x 32; 64 x 4096 x 4096, one round, 24.3 against 28.9).
template <int FM, int FN, int PF>
static void launch_w8a32_ksplit(const W8P& p, const W8Ws& ws, hipStream_t st) {
  const int S = w8a32_slices(p, FM, FN);
  if (S == 1 || (ws.ptr && ws.bytes >= W8_WS_BYTES)) return launch_w8a32_blocks<FM, FN, PF>(p, S, ws, st);
  const int KT = (p.K + 63) / 64, per = (KT + S - 1) / S;
  if (FM == 1 && per % W8_WAVES == 0) launch_w8a32_blocks<1, 1, 1, true>(p, S, ws, st);
  else if (FM == 1) launch_w8a32_blocks<1, 1, 2, true>(p, S, ws, st);
  else if (((p.M + 31) / 32) * ((p.N + 31) / 32) > 256) launch_w8a32_blocks<2, 4, 2, true>(p, S, ws, st);
  else launch_w8a32_blocks<2, 2, 2, true>(p, S, ws, st);
}

template <int FM, int FN, int WAVES>
static void launch_w8a32_tile(const W8P& p, hipStream_t st) {
  constexpr int BM = 16 * FM * WAVES, BN = 16 * FN;
  const unsigned tiles = (unsigned)(((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN));
  w8a32_tile_kernel<FM, FN, WAVES><<<tiles, WAVES * 64, 0, st>>>(p);
}

static int w8a32_common(const char* what, const float* x, const int8_t* W, int64_t M, int64_t N, int64_t K,
                        const float* sW, const float* bias, const float* res, int act, float* out, int max_m,
                        const W8Ws& ws, bq_stream_t stream) {
  if (M < 0 || N < 0 || K < 0) return set_error(BQ_ERR_ARG, "%s: negative size", what);
  if (M == 0 || N == 0) return BQ_OK;
  if (M > max_m)
    return set_error(BQ_ERR_UNSUPPORTED, "%s: M=%lld > %d (bq_linear_w8a32 takes any M)", what, (long long)M, max_m);
  if (K % 16) return set_error(BQ_ERR_UNSUPPORTED, "%s: K=%lld is not a multiple of 16", what, (long long)K);
  if (M > 0x7fffffff || N > 0x7fffffff || M * K * 4 >= ((int64_t)1 << 31) || N * K >= ((int64_t)1 << 31) ||
      M * N >= ((int64_t)1 << 40))
    return set_error(BQ_ERR_ARG, "%s: size too large (x and W must each be < 2 GiB)", what);
  if (!x || !W || !sW || !out) return set_error(BQ_ERR_ARG, "%s: null pointer", what);
  if (((uintptr_t)x & 15) || ((uintptr_t)W & 15)) return set_error(BQ_ERR_ARG, "%s: x and W must be 16-byte aligned", what);
  if (act < BQ_ACT_NONE || act > BQ_ACT_GELU) return set_error(BQ_ERR_ARG, "%s: bad activation %d", what, act);
  hipStream_t st = (hipStream_t)stream;
  if (M <= WA_MPW && K <= 8192) {
    launch_gemv_w8a32(x, W, (int)M, (int)N, (int)K, sW, bias, res, act, out, st);
    return check_launch(what);
  }
  const W8P p{x, W, (int)M, (int)N, (int)K, sW, bias, res, act, out};
  // The K-split kernel up to 256 tiles of 32 x 128, its tile the largest that with its slices still
  // gives the chip's CUs a workgroup each: 16 x 64 for 16 rows of 4096 x 4096 (16 x 32 12.0 us
  // against 11.1) but 16 x 32 at 2048 x 2048 (16 x 64 8.1 us against 7.5); 32 x 128 from 160
  // workgroups on (256 x 3072 x 768, 192 workgroups: 12.2 us, 17.0 in 384 of 32 x 64), and 32 x 64
  // rather than 32 x 32 in more than one round of workgroups (1024 x 300 x 512: 7.0 us against
  // 10.1), as 32 x 128 rather than 32 x 64 (951 x 640 x 640: 11.2 against 16.3). Over a K of at most
  // five chunks 16 x 64 by four waves, whose exchange is half as long, in one round (three a CU):
  // 256 x 3072 x 208 6.4 us, 7.2 as 32 x 128; at 384 9.7 against 9.0, and 449 x 1784 x 256, 812
  // workgroups, 9.1 against 7.3.
  // 5 to 12 rows of up to 2048 values, and 13 to 16 in fewer than three slices, stay with the f32
  // MFMA, which needs no split of x and no exchange (12 x 3000 x 1520 5.8 us against 7.3, 16 x 4096 x
  // 1280 6.6 against 7.5; 16 x 300 x 1792, three slices, 7.5 against 6.4).
  // Tiled above 256: 64 x 64 workgroups up to 511 (1024 x 1400 x 1024 21.4 us, 27.5 K-split, 22.1 in 64
  // x 128; 4096 x 300 x 320 10.7, 14.5 and 12.0), up to 1023 under K = 512 (2000 x 1200 x 400 15.8
  // against 19.0; 4096 x 768 x 640 24.0 against 23.6), then 128 x 128 where they fill the chip evenly
  // (2048^3 55 us against 59 in 64 x 128), else 64 x 128 (6304 x 768 x 3072, 300 tiles of 128 x 128:
  // 108 us against 122).
  const auto tiles = [&](int bm, int bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  // workgroups a K-split tile shape can fill: its tiles times the slices of at least a chunk a wave
  const auto fill = [&](int fm, int fn) { return tiles(16 * fm, 16 * fn) * std::max<int64_t>(1, (K + 63) / 64 / W8_WAVES); };
  if (M <= WA_MMAX) {
    const int fn = fill(1, 4) >= 256 ? 4 : fill(1, 2) >= 256 ? 2 : 1;
    if (K <= 1024 || (K <= 2048 && (M <= 12 || w8a32_slices(p, 1, fn) < 3))) {
      const unsigned grid = (unsigned)((N + WM_ROWS - 1) / WM_ROWS);
      gemv_w8a32_mfma_kernel<4><<<grid, WA_WAVES * 64, 0, st>>>(x, W, (int)M, (int)N, (int)K, sW, bias, res, act, out);
      return check_launch(what);
    }
    if (fn == 4) launch_w8a32_ksplit<1, 4, 2>(p, ws, st);
    else if (fn == 2) launch_w8a32_ksplit<1, 2, 4>(p, ws, st);
    else launch_w8a32_ksplit<1, 1, 4>(p, ws, st);
  } else if (tiles(32, 128) <= 256) {
    if (K <= 320 && tiles(16, 64) <= 768) launch_w8a32_blocks<1, 4, 1, false, 4>(p, 1, ws, st);
    else if (M > 32 && (fill(2, 8) >= 160 || tiles(32, 64) > 256)) launch_w8a32_ksplit<2, 8, 1>(p, ws, st);
    else if (fill(2, 4) >= 256 || tiles(32, 32) > 256) launch_w8a32_ksplit<2, 4, 2>(p, ws, st);
    else launch_w8a32_ksplit<2, 2, 2>(p, ws, st);
  } else if (tiles(32, 128) < (K < 512 ? 1024 : 512)) {
    launch_w8a32_tile<1, 4, 4>(p, st);
  } else {
    const int64_t t = tiles(128, 128);
    if (t >= 512 || (t >= 192 && t <= 256)) launch_w8a32_tile<1, 8, 8>(p, st);
    else launch_w8a32_tile<1, 8, 4>(p, st);
  }
  return check_launch(what);
}

}  // namespace bq

using namespace bq;

extern "C" {

int bq_gemv_w8a32(const float* x, const int8_t* W, int64_t M, int64_t N, int64_t K, const float* sW,
                  const float* bias, int act, float* out, bq_stream_t stream) {
  if (K > 8192) return set_error(BQ_ERR_UNSUPPORTED, "bq_gemv_w8a32: K=%lld > 8192", (long long)K);
  return w8a32_common("bq_gemv_w8a32", x, W, M, N, K, sW, bias, nullptr, act, out, WA_MMAX, W8Ws{nullptr, 0},
                      stream);
}

int bq_linear_w8a32(const float* x, const int8_t* W, int64_t M, int64_t N, int64_t K, const float* sW,
                    const float* bias, const float* residual, int act, float* out, bq_stream_t stream) {
  return w8a32_common("bq_linear_w8a32", x, W, M, N, K, sW, bias, residual, act, out, 0x7fffffff,
                      W8Ws{nullptr, 0}, stream);
}

int bq_linear_w8a32_ws(const float* x, const int8_t* W, int64_t M, int64_t N, int64_t K, const float* sW,
                       const float* bias, const float* residual, int act, float* out, void* ws, size_t ws_bytes,
                       bq_stream_t stream) {
  return w8a32_common("bq_linear_w8a32_ws", x, W, M, N, K, sW, bias, residual, act, out, 0x7fffffff,
                      W8Ws{ws, ws_bytes}, stream);
}

int bq_dequant_i8(const int8_t* q, int64_t N, int64_t K, const float* s, float* w, bq_stream_t stream) {
  const char* what = "bq_dequant_i8";
  if (N < 0 || K < 0) return set_error(BQ_ERR_ARG, "%s: negative size", what);
  if (N == 0 || K == 0) return BQ_OK;
  if (!q || !s || !w) return set_error(BQ_ERR_ARG, "%s: null pointer", what);
  if (((uintptr_t)q & 3) || ((uintptr_t)w & 15)) return set_error(BQ_ERR_ARG, "%s: misaligned pointer", what);
  int64_t blocks = (N * K / 4 + 255) / 256;
  if (blocks > 16384) blocks = 16384;
  if (blocks < 1) blocks = 1;
  dequant_i8_kernel<<<(unsigned)blocks, 256, 0, (hipStream_t)stream>>>(q, N, K, s, w);
  return check_launch(what);
}

}  // extern "C"
