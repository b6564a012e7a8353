// Softmax attention in f32 for a transformer's heads of width 64 and sequences of at most
// 256 tokens (ViT-B/16's 197): out = softmax((q k^T) * (1 / sqrt(64))) v per (image, head),
// the computation of borch's scaled_dot_product_attention (borch/_nn.py:2143-2170; its
// softmax is softmaxRows, borch-ts/src/kernels.ts:2483-2532: exp(x - max) / sum). It reads
// q, k and v straight from the qkv projection's output [B, T, 3, H, 64] and writes the heads
// side by side, [B, T, H * 64], the layout the output projection reads (no permute or
// transpose pass on either side).
//
// One workgroup per (image, head, 128 queries), 8 waves of 16 queries. The products run on the
// bf16 MFMA (16 times the f32 MFMA's rate): every f32 operand is the exact sum of three bf16
// pieces (bq_bf16x3.h), and of the nine products of pieces the six of weight 2^-18 and above are
// added, the largest of each product into one f32 accumulator and the other five into a second.
// The three left out are below 2^-26 of the product, under the f32 rounding of the sum; measured
// against float64 on N(0, 1) inputs the output's relative error is 1.6e-7, where f32 MFMAs gave
// 3.3e-7 (9.4e-8 and 1.9e-7 on flat softmaxes, scores of 0.01).
//
// k's planes are staged in LDS once, split there by the whole workgroup, and v's take their
// place after the scores: 80 KB at 208 keys, so that two workgroups share a CU and one's loads
// and softmax run under the other's MFMAs (k and v together as f32 left one workgroup a CU).
// The scores are computed transposed, S^T = k q^T, so that each lane holds one query's scores
// (keys 16 j + 4 (lane / 16) + i in register i of key block j): the softmax of a query is a
// reduction over the lane's own registers and its 3 partner lanes, and the exponentials are,
// register for register, the second operand of O^T = v^T E^T (O divided by the row sum last).
// The contracted index of that product (keys) and its rows (head dims) are permuted to suit:
// a 32-key step takes keys 32 s + 16 (e / 4) + 4 g + e % 4 as group g's eight, and row n of block
// d is head dim 4 n + d, so that v is written to LDS and the output to memory in whole pieces.
//
// ViT-B/16 at 32 images (197 tokens, 12 heads): 70 -> 35 us; 256 tokens 86 -> 53 us (98 KB
// of LDS, one workgroup a CU).
#include <math.h>

#include "bq_bf16x3.h"
#include "bq_common.h"

namespace bq {

constexpr int ATT_DH = 64;    // head width
constexpr int ATT_WAVES = 8;  // 16 queries each

__device__ __forceinline__ float xor_max(float v, int m) { return fmaxf(v, __shfl_xor(v, m)); }
__device__ __forceinline__ float xor_add(float v, int m) { return __fadd_rn(v, __shfl_xor(v, m)); }

// Attention of query q of one head by one wave in plain f32: for queries whose outputs did not
// come out finite above (an infinity among the inputs, or a value a bf16 piece cannot hold) or
// came out smaller than the pieces of v reach.
// Lane l scores keys l, l + 64, ..., then sums head dim l.
__device__ __attribute__((noinline)) void attention_f32_query(const float* base, size_t tok, int T, int D, int q,
                                                              float* orow) {
  const int lane = threadIdx.x & 63;
  const float* qp = base + q * tok;
  float s[4], m = -INFINITY;
  for (int t = 0; t < 4; ++t) {
    const int key = lane + 64 * t;
    float v = 0.f;
    if (key < T)
      for (int d = 0; d < ATT_DH; ++d) v = __fmaf_rn(qp[d], base[key * tok + D + d], v);
    s[t] = key < T ? __fmul_rn(v, 0.125f) : -INFINITY;
    m = fmaxf(m, s[t]);
  }
  for (int d = 1; d < 64; d *= 2) m = xor_max(m, d);
  float sum = 0.f;
  for (int t = 0; t < 4; ++t) {
    s[t] = expf(__fsub_rn(s[t], m));  // exp(-inf) = 0 past T
    sum = __fadd_rn(sum, s[t]);
  }
  sum = wave_sum_fixed(sum);
  float o = 0.f;
  for (int key = 0; key < T; ++key) {
    const float e = __shfl(key < 64 ? s[0] : key < 128 ? s[1] : key < 192 ? s[2] : s[3], key & 63);
    o = __fmaf_rn(e, base[key * tok + 2 * D + lane], o);
  }
  orow[lane] = __fdiv_rn(o, sum);
}

// A fragment's products with another's: those of the first pieces into acc, the five smaller ones
// into low, a sum of its own that is added last, so that each of acc's roundings stands for a whole
// 32-deep product and not for a sixth of one (39 such roundings in one sum of 197 keys made the
// error of flat softmaxes larger than f32 MFMAs', 2.1e-7 against 1.9e-7).
__device__ __forceinline__ void mfma6(const Split8& a, const Split8& b, v4f& acc, v4f& low) {
  low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.p3, b.p1, low, 0, 0, 0);
  low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.p2, b.p2, low, 0, 0, 0);
  low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.p1, b.p3, low, 0, 0, 0);
  low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.p2, b.p1, low, 0, 0, 0);
  low = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.p1, b.p2, low, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.p1, b.p1, acc, 0, 0, 0);
}

template <int KB>  // key blocks of 16
__global__ __launch_bounds__(ATT_WAVES * 64, KB <= 13 ? 4 : 2) void attention_f32_kernel(const float* __restrict__ qkv,
                                                                                        int T, int H, int qblocks,
                                                                                        float* __restrict__ out) {
  constexpr int THREADS = ATT_WAVES * 64;
  constexpr int PLANE = KB * 16 * ATT_DH * 2;   // bytes of one bf16 plane of k or v
  constexpr int STEPS = KB / 2;                 // 32-key steps of the second product (then 16 keys if KB is odd)
  constexpr int TAIL = STEPS * ATT_DH * 64;     // where those 16 keys' rows start
  __shared__ __attribute__((aligned(16))) unsigned char kv[3 * PLANE];
  const int id = xcd_order(blockIdx.x, gridDim.x);  // a head's blocks run on one XCD
  const int bh = id / qblocks, qb = id - bh * qblocks;
  const int b = bh / H, h = bh - b * H;
  const int D = H * ATT_DH;
  const size_t tok = (size_t)3 * D;  // floats from one token's q to the next's
  const float* base = qkv + (size_t)b * T * tok + (size_t)h * ATT_DH;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n = lane & 15;  // this lane's query within the wave's 16
  const int g = lane >> 4;
  const int q0 = qb * (ATT_WAVES * 16) + wave * 16;
  const int q = q0 + n;

  // k's planes: rows of 128 bytes (64 head dims), 16-byte pieces XORed by row bits so that the 16
  // rows of a fragment read cover all 64 banks; keys past T as zeros (masked below)
  constexpr int PER = (KB * 256 + THREADS - 1) / THREADS;  // float4s of k a thread
  float4 kr[PER], q4[4];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int idx = tid + i * THREADS, key = idx >> 4;
    kr[i] = key < T ? *reinterpret_cast<const float4*>(base + key * tok + D + (idx & 15) * 4)
                    : make_float4(0.f, 0.f, 0.f, 0.f);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)  // head dims 32 (e / 2) + 8 g + 4 (e % 2) .. + 3 of this lane's query
    q4[e] = q < T ? *reinterpret_cast<const float4*>(base + q * tok + 32 * (e >> 1) + 8 * g + 4 * (e & 1))
                  : make_float4(0.f, 0.f, 0.f, 0.f);
  // v: a thread takes 4 keys x 4 head dims at a time, loaded under the softmax; up to 64 keys with
  // k, where a workgroup is one chain of round trips (64 tokens, 3 heads 6.2 -> 6.0 us)
  constexpr int VPER = ((KB + 1) / 2 * 128 + THREADS - 1) / THREADS;
  float4 vr[VPER][4];
  auto load_v = [&]() {
#pragma unroll
    for (int i = 0; i < VPER; ++i) {
      const int idx = tid + i * THREADS, kq = ((idx >> 3) & 7) + 8 * (idx >> 7), c4 = (idx & 7) + 8 * ((idx >> 6) & 1);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        vr[i][e] = 4 * kq + e < T ? *reinterpret_cast<const float4*>(base + (4 * kq + e) * tok + 2 * D + 4 * c4)
                                  : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  if constexpr (KB <= 4) load_v();
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int idx = tid + i * THREADS, key = idx >> 4, c = idx & 15;
    if (KB * 256 % THREADS == 0 || key < KB * 16) {
      uint2 p1, p2, p3;
      split3(kr[i].x, kr[i].y, p1.x, p2.x, p3.x);
      split3(kr[i].z, kr[i].w, p1.y, p2.y, p3.y);
      unsigned char* at = kv + key * 128 + (((c >> 1) ^ ((key >> 1) & 7)) << 4) + (c & 1) * 8;
      *reinterpret_cast<uint2*>(at) = p1;
      *reinterpret_cast<uint2*>(at + PLANE) = p2;
      *reinterpret_cast<uint2*>(at + 2 * PLANE) = p3;
    }
  }
  __syncthreads();

  const bool live = q0 < T;  // a wave past the last query only helps to stage
  v4f s[KB];
  float sum = 0.f;
  if (live) {
    // S^T = k q^T: key block j, lane (n, g), register i -> key 16 j + 4 g + i, query q
    const Split8 qf[2] = {split8(q4[0], q4[1]), split8(q4[2], q4[3])};
#pragma unroll
    for (int j = 0; j < KB; ++j) {
      s[j] = v4f{0.f, 0.f, 0.f, 0.f};
      v4f low = s[j];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const unsigned char* at = kv + (16 * j + n) * 128 + (((4 * t + g) ^ ((n >> 1) & 7)) << 4);
        const Split8 kf = {*reinterpret_cast<const v8bf*>(at), *reinterpret_cast<const v8bf*>(at + PLANE),
                           *reinterpret_cast<const v8bf*>(at + 2 * PLANE)};
        mfma6(kf, qf[t], s[j], low);
      }
      s[j] += low;
    }
  }
  if constexpr (KB > 4) load_v();
  if (live) {
    // softmax over the keys of query q: exp((score - max) / sqrt(64)), keys past T at -inf, in
    // powers of two. The maximum is subtracted first, so that its own exponential is 1 whatever
    // its size: folded into one FMA, fma(s, c, -fl(m c)), every exponential carried the factor
    // 2^(m c - fl(m c)), which cancels in the quotient only while it stays in range (scores
    // near 2^34 lost their lower pieces, 4e-3 of the output). 34.3 -> 34.5 us at 32 x 197 tokens.
    constexpr float c = 0.125f * 1.4426950408889634f;
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < KB; ++j) {
      if (16 * j + 16 > T)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (16 * j + 4 * g + i >= T) s[j][i] = -INFINITY;
      m = fmaxf(fmaxf(m, fmaxf(s[j][0], s[j][1])), fmaxf(s[j][2], s[j][3]));
    }
    m = xor_max(xor_max(m, 16), 32);
#pragma unroll
    for (int j = 0; j < KB; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float e = __builtin_amdgcn_exp2f(__fmul_rn(__fsub_rn(s[j][i], m), c));  // 0 for the masked keys
        s[j][i] = e;
        sum = __fadd_rn(sum, e);
      }
    sum = xor_add(xor_add(sum, 16), 32);
  }

  __syncthreads();  // every wave has read its k fragments
  // v's planes, transposed: each head dim's four keys as one 8-byte piece; row (d, n) = dim
  // 4 n + d holds a step's 32 keys in 64 bytes (32 bytes for the last 16 keys), pieces XORed by
  // row bits as k's are
#pragma unroll
  for (int i = 0; i < VPER; ++i) {
    const int idx = tid + i * THREADS, kq = ((idx >> 3) & 7) + 8 * (idx >> 7), c4 = (idx & 7) + 8 * ((idx >> 6) & 1);
    if (kq >= 4 * KB) continue;
    const int step = kq >> 3, half = (kq >> 2) & 1, vg = kq & 3;
    const float col[4][4] = {{vr[i][0].x, vr[i][1].x, vr[i][2].x, vr[i][3].x},
                             {vr[i][0].y, vr[i][1].y, vr[i][2].y, vr[i][3].y},
                             {vr[i][0].z, vr[i][1].z, vr[i][2].z, vr[i][3].z},
                             {vr[i][0].w, vr[i][1].w, vr[i][2].w, vr[i][3].w}};
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      uint2 p1, p2, p3;
      split3(col[d][0], col[d][1], p1.x, p2.x, p3.x);
      split3(col[d][2], col[d][3], p1.y, p2.y, p3.y);
      const int row = d * 16 + c4;
      unsigned char* at = kv + (step < STEPS ? step * ATT_DH * 64 + row * 64 + ((vg ^ ((c4 >> 2) & 3)) << 4) + half * 8
                                             : TAIL + row * 32 + vg * 8);
      *reinterpret_cast<uint2*>(at) = p1;
      *reinterpret_cast<uint2*>(at + PLANE) = p2;
      *reinterpret_cast<uint2*>(at + 2 * PLANE) = p3;
    }
  }
  __syncthreads();
  if (!live) return;  // no barrier follows

  // O^T = v^T E^T with the unnormalised exponentials E, then O / sum (the normalisation moves past
  // the f32 sums, within their bound): block d, lane (n, g), register r -> dim 16 g + 4 r + d, query q
  v4f o[4], low[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) o[d] = low[d] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < STEPS; ++t) {
    const v4f e0 = s[2 * t], e1 = s[2 * t + 1];
    const Split8 ef = split8(make_float4(e0[0], e0[1], e0[2], e0[3]), make_float4(e1[0], e1[1], e1[2], e1[3]));
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const unsigned char* at = kv + t * ATT_DH * 64 + (d * 16 + n) * 64 + ((g ^ ((n >> 2) & 3)) << 4);
      const Split8 vf = {*reinterpret_cast<const v8bf*>(at), *reinterpret_cast<const v8bf*>(at + PLANE),
                         *reinterpret_cast<const v8bf*>(at + 2 * PLANE)};
      mfma6(vf, ef, o[d], low[d]);
    }
  }
  if constexpr (KB % 2) {
    uint2 p1, p2, p3;
    split3(s[KB - 1][0], s[KB - 1][1], p1.x, p2.x, p3.x);
    split3(s[KB - 1][2], s[KB - 1][3], p1.y, p2.y, p3.y);
    const v4s e1 = __builtin_bit_cast(v4s, p1), e2 = __builtin_bit_cast(v4s, p2), e3 = __builtin_bit_cast(v4s, p3);
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const unsigned char* at = kv + TAIL + (d * 16 + n) * 32 + g * 8;
      const v4s v1 = *reinterpret_cast<const v4s*>(at), v2 = *reinterpret_cast<const v4s*>(at + PLANE),
                v3 = *reinterpret_cast<const v4s*>(at + 2 * PLANE);
      low[d] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(v3, e1, low[d], 0, 0, 0);
      low[d] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(v2, e2, low[d], 0, 0, 0);
      low[d] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(v1, e3, low[d], 0, 0, 0);
      low[d] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(v2, e1, low[d], 0, 0, 0);
      low[d] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(v1, e2, low[d], 0, 0, 0);
      o[d] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(v1, e1, o[d], 0, 0, 0);
    }
  }
#pragma unroll
  for (int d = 0; d < 4; ++d) o[d] += low[d];
  float* orow = out + ((size_t)b * T + q) * D + (size_t)h * ATT_DH;
  float4 y[4];
  // taken again: an output that is not finite, or (zero aside) below 2^-109, where the up to 2^-134
  // that the split takes from a smaller v is more than a rounding
  float zero = 0.f;  // NaN beside a value that is not finite
  uint32_t least = ~0u;  // |y| as an integer, 0 as the largest
  auto look = [&](float v) {
    zero = __fmaf_rn(v, 0.f, zero);
    least = min(least, (__float_as_uint(v) << 1) - 1u);
  };
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    y[r] = make_float4(__fdiv_rn(o[0][r], sum), __fdiv_rn(o[1][r], sum), __fdiv_rn(o[2][r], sum), __fdiv_rn(o[3][r], sum));
    look(y[r].x); look(y[r].y); look(y[r].z); look(y[r].w);
  }
  const bool good = zero == 0.f && least >= (__float_as_uint(0x1p-109f) << 1) - 1u;
  uint64_t again = __ballot(q < T && !good);  // bit n of each 16: query q0 + n
  again |= again >> 32;
  again |= again >> 16;
  if (q < T && !((again >> n) & 1))
#pragma unroll
    for (int r = 0; r < 4; ++r) *reinterpret_cast<float4*>(orow + 16 * g + 4 * r) = y[r];
  for (int i = 0; i < 16; ++i)
    if ((again >> i) & 1)
      attention_f32_query(base, tok, T, D, q0 + i, out + ((size_t)b * T + q0 + i) * D + (size_t)h * ATT_DH);
}

}  // namespace bq

using namespace bq;

int bq_attention_f32(const float* qkv, int64_t B, int64_t T, int64_t H, int64_t dh, float* out, bq_stream_t stream) {
  const char* what = "bq_attention_f32";
  if (B < 0 || T < 0 || H < 1) return set_error(BQ_ERR_ARG, "%s: bad sizes", what);
  if (dh != ATT_DH) return set_error(BQ_ERR_UNSUPPORTED, "%s: head width %lld (64 only)", what, (long long)dh);
  if (T > 256) return set_error(BQ_ERR_UNSUPPORTED, "%s: %lld tokens (at most 256)", what, (long long)T);
  if (B == 0 || T == 0) return BQ_OK;
  if (B * T * 3 * H * dh >= ((int64_t)1 << 31) || B * H > 0x7fffffff / 4)
    return set_error(BQ_ERR_ARG, "%s: size too large", what);
  if (!qkv || !out) return set_error(BQ_ERR_ARG, "%s: null pointer", what);
  if (((uintptr_t)qkv & 15) || ((uintptr_t)out & 15)) return set_error(BQ_ERR_ARG, "%s: misaligned pointer", what);
  const int qblocks = (int)((T + ATT_WAVES * 16 - 1) / (ATT_WAVES * 16));
  const unsigned grid = (unsigned)(B * H * qblocks);
  hipStream_t st = (hipStream_t)stream;
  const int kb = (int)((T + 15) / 16);
  if (kb <= 4) attention_f32_kernel<4><<<grid, ATT_WAVES * 64, 0, st>>>(qkv, (int)T, (int)H, qblocks, out);
  else if (kb <= 8) attention_f32_kernel<8><<<grid, ATT_WAVES * 64, 0, st>>>(qkv, (int)T, (int)H, qblocks, out);
  else if (kb <= 13) attention_f32_kernel<13><<<grid, ATT_WAVES * 64, 0, st>>>(qkv, (int)T, (int)H, qblocks, out);
  else attention_f32_kernel<16><<<grid, ATT_WAVES * 64, 0, st>>>(qkv, (int)T, (int)H, qblocks, out);
  return check_launch(what);
}
