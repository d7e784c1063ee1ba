// Exact attention of many query rows over fp16 K/V (attention.py:39-105) on
// the matrix cores: what rfsn_blockwise_attention runs for a chunk of a prompt,
// and for single queries of grouped heads.
//
// The B x G query rows that read one KV head (G query heads per KV head) are
// one row range; a wave takes 32 of them, WR waves share a block's K/V tiles of
// 64 tokens in LDS, and WT such groups of waves take the tiles in turn (merged
// through LDS at the end, which keeps small problems free of global partials).
// Per 32 tokens and wave:
//   S^T = K Q^T    MFMA 32x32x16, A = 32 tokens of K, B = the wave's rows: a
//                  lane holds 16 scores of ONE row, so the softmax stays in the
//                  lane;
//   O^T += V^T P^T with the score registers as the B operand as they are: k
//                  slot (half hf, j) of step st is token 16 st + 8 (j >> 2) +
//                  4 hf + (j & 3), and ds_read_b64_tr_b16 reads V^T in that
//                  order from row-major V, so neither P nor V changes lanes.
// P is kept to 2^-23 of itself (exp2's own error), p * 2^8 as fp16 hi + fp16 lo
// (two MFMAs; V is exact); everything accumulates in fp32, and the row sum adds
// the unsplit p.  Before its fp16 rounding a result is off by 2.5e-7 to 5.8e-7
// (2-norm against float64, 64 to 1,000 queries, 500 to 8,192 tokens, scores of
// deviation 1 to 16); attention.hip's fp32 products of fp32 weights are off by
// 3.2e-7 to 1.6e-6 on the same inputs.
// Infinities in V: hi * V and lo * V cancel or meet 0 where p * V is infinite, so
// a block that finds a sum that is not finite takes its rows again in fp32
// (careful_rows).
// The maximum is moved only when a lane's sum of p says that it must be, which
// takes the max scan and its cross-lane step out of most tiles.
//
// Bound: VALU issue of the softmax (5 per score: fma, exp2, add, half a cvt_pk
// twice, fma_mix) beside 24 MFMAs per 64 x 32 scores: 70 % of the issue cycles, the
// matrix cores 49 %, LDS 21 %, at 1,000 queries over 8,192 tokens.  1,000 queries x 32 heads
// over 8,192 tokens of 8 KV heads (D 64, causal): 1,815 us on the scalar kernel
// of attention.hip (one lane per token, K/V re-read per query), 116 us here, 543 TFLOP/s of
// S and P V together; 128 queries x 32 heads, D 128, 4,096 tokens: 685 -> 31 us.
#include "rfsn_common.h"
#include "rfsn_internal.h"

namespace rfsn {
namespace {

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef short short4v __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));

constexpr int kTile = 64;          // tokens per LDS tile
constexpr float kPBias = 8.f;      // P is kept as p * 2^8
constexpr float kPSum = 32768.f;   // a lane's tile sum below it: every p of the tile is finite in fp16

// 16-byte chunk c of row t of a [64][D] fp16 tile sits at chunk c ^ swz(t):
// K rows are read 16 at a time at one chunk, V rows four at a time over 64
// bytes; both then touch every bank once.
template <int D>
__device__ __forceinline__ int k_swz(int t) { return D == 64 ? (t >> 1) & 7 : t & 15; }
template <int D>
__device__ __forceinline__ int v_swz(int t) { return D == 64 ? ((t >> 1) & 1) * 4 : (t & 3) * 4; }

__device__ __forceinline__ float half_max(float x) {
  return fmaxf(x, __shfl_xor(x, 32, 64));
}

__device__ __forceinline__ half8 join(const half2v* p) {
  return half8{p[0][0], p[0][1], p[1][0], p[1][1], p[2][0], p[2][1], p[3][0], p[3][1]};
}

// Four rows over the tokens t0 .. lim[row] by one wave, as attention.hip's kernel
// takes them: lane = token for scores, lane = coordinate for P V, weights and
// products in fp32.  NaN and infinite values meet the weights of the tokens a row
// may read, and no others.  Four rows share each K and V load (one: 8.2 ms for 1,000
// queries x 32 heads over 8,192 tokens with an infinity in each block, four 3.7,
// attention.hip's kernel 1.8); eight spill registers in the first pass (118 -> 122 us).
constexpr int kCareful = 4;
template <int D>
__device__ __forceinline__ void careful_rows(const uint16_t* const (&q)[kCareful], const uint16_t* __restrict__ K,
                                             const uint16_t* __restrict__ V, int64_t stride_t, float scale_log2, int t0,
                                             const int (&lim)[kCareful], int lane, float (&m)[kCareful],
                                             float (&l)[kCareful], float (&acc)[kCareful][D / 64]) {
  int end = lim[0];
#pragma unroll
  for (int r = 0; r < kCareful; ++r) {
    end = max(end, lim[r]);
    m[r] = -__builtin_inff();
    l[r] = 0.f;
#pragma unroll
    for (int e = 0; e < D / 64; ++e) acc[r][e] = 0.f;
  }
#pragma unroll 1
  for (int base = t0; base <= end; base += 64) {
    const half8* k = reinterpret_cast<const half8*>(K + (int64_t)min(base + lane, end) * stride_t);
    float s[kCareful] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
    for (int c = 0; c < D / 8; ++c) {
      const half8 kv = k[c];
#pragma unroll
      for (int r = 0; r < kCareful; ++r) {
        const half8 qv = reinterpret_cast<const half8*>(q[r])[c];
#pragma unroll
        for (int e = 0; e < 8; ++e) s[r] = fmaf((float)qv[e] * scale_log2, (float)kv[e], s[r]);
      }
    }
    float p[kCareful];
#pragma unroll
    for (int r = 0; r < kCareful; ++r) {
      if (base + lane > lim[r]) s[r] = -__builtin_inff();
      const float mn = fmaxf(m[r], wave_max(s[r]));
      p[r] = mn > -__builtin_inff() ? exp2f(s[r] - mn) : s[r] != s[r] ? s[r] : 0.f;  // a NaN score is no maximum
      const float corr = m[r] > -__builtin_inff() ? exp2f(m[r] - mn) : (mn > -__builtin_inff() ? 0.f : 1.f);
      l[r] = l[r] * corr + wave_sum(p[r]);
      m[r] = mn;
#pragma unroll
      for (int e = 0; e < D / 64; ++e) acc[r][e] *= corr;
    }
    const int count = min(64, end - base + 1);
#pragma unroll 4
    for (int t = 0; t < count; ++t) {
      const uint16_t* v = V + (int64_t)(base + t) * stride_t + lane * (D / 64);
      float vv[D / 64];
#pragma unroll
      for (int e = 0; e < D / 64; ++e) vv[e] = h2f(v[e]);
#pragma unroll
      for (int r = 0; r < kCareful; ++r) {
        const float pt = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, p[r]), t));
        const bool read = base + t <= lim[r];
#pragma unroll
        for (int e = 0; e < D / 64; ++e) acc[r][e] = read ? fmaf(pt, vv[e], acc[r][e]) : acc[r][e];
      }
    }
  }
}

template <int D, int WR, int WT, int MW>
__global__ void __launch_bounds__(WR * WT * 64, MW)
prompt_attn_kernel(const uint16_t* __restrict__ q, int B, int Hq, int G, const uint16_t* __restrict__ K,
                   const uint16_t* __restrict__ V, int T, int64_t stride_t, int64_t stride_h, float scale_log2,
                   int causal, const int32_t* __restrict__ qpos, int row_tiles, int tokens_per_split, int splits,
                   float bad, uint16_t* __restrict__ out, float* __restrict__ part_ml,
                   float* __restrict__ part_acc) {
  constexpr int kThreads = WR * 64;                         // threads of a token group
  constexpr int kChunks = D / 8;                            // 16-byte chunks of a row
  constexpr int kLoads = kTile * kChunks / kThreads;        // chunks a thread stages per tile and tensor
  constexpr int kKS = D / 16;                               // MFMA k steps of a score
  constexpr int kDT = D / 32;                               // 32-coordinate tiles of O^T
  constexpr int kTileVecs = kTile * kChunks;
  __shared__ uint4v smem[WT * 4 * kTileVecs];               // per group: K, V of two tiles
  __shared__ int s_hi[WR * WT];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wave % WR, grp = wave / WR, tid = threadIdx.x - grp * kThreads;
  const int col = lane & 31, hf = lane >> 5;
  // KV heads vary fastest over the blocks: with 8 of them each XCD's L2 keeps one
  // head's K/V.  The last row tiles (of a causal prompt the longest) start first.
  const int h = blockIdx.x, rt = row_tiles - 1 - (int)blockIdx.y, split = blockIdx.z;
  const int rows = B * G;
  const int row = rt * (WR * 32) + wr * 32 + col;
  const int rc = row < rows ? row : rows - 1;
  const int64_t qi = (int64_t)(rc / G) * Hq + (int64_t)h * G + rc % G;  // (query, query head) of the lane's row

  const int t0 = split * tokens_per_split;
  const int t1 = min(T, t0 + tokens_per_split);
  int lim = T - 1;  // last token the lane's row may read
  if (causal && qpos) lim = min(lim, qpos[qi]);
  lim = min(lim, t1 - 1);
  int w_hi = lim, w_lo = lim;
#pragma unroll
  for (int o = 16; o > 0; o >>= 1) {
    w_hi = max(w_hi, __shfl_xor(w_hi, o, 64));
    w_lo = min(w_lo, __shfl_xor(w_lo, o, 64));
  }
  w_hi = __builtin_amdgcn_readfirstlane(w_hi);
  w_lo = __builtin_amdgcn_readfirstlane(w_lo);
  if (lane == 0) s_hi[wave] = w_hi;
  __syncthreads();
  int b_hi = s_hi[0];
#pragma unroll
  for (int w = 1; w < WR; ++w) b_hi = max(b_hi, s_hi[w]);
  const int tiles = b_hi < t0 ? 0 : (b_hi - t0) / kTile + 1;
  const int iters = (tiles + WT - 1) / WT;  // group g takes tiles g, g + WT, ...

  half8 qf[kKS];
  {
    const uint4v* qr = reinterpret_cast<const uint4v*>(q + qi * D);
#pragma unroll
    for (int s = 0; s < kKS; ++s) qf[s] = __builtin_bit_cast(half8, qr[2 * s + hf]);
  }
  float16v o[kDT];
#pragma unroll
  for (int d = 0; d < kDT; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[d][i] = 0.f;
  // reference exponent of the row's p (its running maximum in base-2 units less
  // kPBias, one rounded value that every rescale and merge uses) and the sum of p
  float m_run = -__builtin_inff(), l_run = 0.f;

  const uint16_t* Kh = K + (int64_t)h * stride_h;
  const uint16_t* Vh = V + (int64_t)h * stride_h;
  uint4v* const sg = smem + grp * 4 * kTileVecs;
  uint4v kr[kLoads], vr[kLoads];
  // tokens past the split's end re-read its last one: their scores are masked
  // (t > lim), and its V is a value the row range reads anyway
  auto fetch = [&](int it) {
    const int tb = t0 + (it * WT + grp) * kTile;
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const int i = u * kThreads + tid, t = i / kChunks, c = i % kChunks;
      const int64_t off = (int64_t)min(tb + t, t1 - 1) * stride_t + c * 8;
      kr[u] = *reinterpret_cast<const uint4v*>(Kh + off);
      vr[u] = *reinterpret_cast<const uint4v*>(Vh + off);
    }
  };
  auto store = [&](int buf) {
    uint4v* const sk = sg + buf * 2 * kTileVecs;
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const int i = u * kThreads + tid, t = i / kChunks, c = i % kChunks;
      sk[t * kChunks + (c ^ k_swz<D>(t))] = kr[u];
      sk[kTileVecs + t * kChunks + (c ^ v_swz<D>(t))] = vr[u];
    }
  };
  if (iters > 0) {
    fetch(0);
    store(0);
  }
  __syncthreads();
  // lane parts of the V^T reads: 16 lanes read 4 tokens x 16 coordinates
  const int vt = ((lane >> 5) << 2) + ((lane & 15) >> 2);                 // token within 8
  const int vc = ((lane >> 4) & 1) * 16 + (lane & 3) * 4;                 // coordinate within 32
  // constants the compiler may not see through: v_med3 and v_fma_mix stay one instruction each
  float inf = __builtin_inff(), minus1 = -1.f;
  asm("" : "+s"(inf), "+s"(minus1));

  for (int it = 0; it < iters; ++it) {
    const int buf = it & 1;
    const int tb = t0 + (it * WT + grp) * kTile;
    if (it + 1 < iters) fetch(it + 1);
    if (tb <= w_hi) {
      const uint4v* const sk = sg + buf * 2 * kTileVecs;
      const uint4v* const sv = sk + kTileVecs;
#pragma unroll
      for (int u = 0; u < 2; ++u) {  // 32 tokens at a time: few live registers, so four waves fit a SIMD
        float16v s;
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = 0.f;
        const int t = 32 * u + col;
#pragma unroll
        for (int k = 0; k < kKS; ++k) {
          const half8 kf = __builtin_bit_cast(half8, sk[t * kChunks + ((2 * k + hf) ^ k_swz<D>(t))]);
          s = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[k], s, 0, 0, 0);
        }
        if (tb + 32 * u + 31 > w_lo) {
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (tb + 32 * u + 8 * (i >> 2) + 4 * hf + (i & 3) > lim) s[i] = -__builtin_inff();
        }
        half2v ph[8], pl[8];
        float ls;
        auto weights = [&]() {
          const float mb = m_run > -__builtin_inff() ? m_run : 0.f;
          ls = 0.f;
#pragma unroll
          for (int i = 0; i < 16; i += 2) {
            const float2v p = {__builtin_amdgcn_exp2f(fmaf(s[i], scale_log2, -mb)),
                               __builtin_amdgcn_exp2f(fmaf(s[i + 1], scale_log2, -mb))};
            ls += p[0];
            ls += p[1];
            const half2v hi = __builtin_convertvector(p, half2v);
            const float2v r = {fmaf(minus1, (float)hi[0], p[0]), fmaf(minus1, (float)hi[1], p[1])};
            ph[i / 2] = hi;
            pl[i / 2] = __builtin_convertvector(r, half2v);
          }
        };
        weights();
        // The running max is moved only when a lane's sum says that some p may leave
        // fp16's range (or nothing was seen yet): p >= 0, so no p exceeds the sum.
        if (__any(!(ls < kPSum) || m_run == -__builtin_inff())) {
          float mx = -__builtin_inff();
#pragma unroll
          for (int i = 0; i < 16; i += 2) mx = fmaxf(mx, __builtin_amdgcn_fmed3f(s[i], s[i + 1], inf));
          mx = half_max(mx);
          const float m_new = fmaxf(m_run, fmaf(mx, scale_log2, -kPBias));
          const float corr = m_run > -__builtin_inff() ? __builtin_amdgcn_exp2f(m_run - m_new) : 0.f;
          l_run *= corr;
#pragma unroll
          for (int d = 0; d < kDT; ++d)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[d][i] *= corr;
          m_run = m_new;
          weights();
        }
        l_run += ls;
#pragma unroll
        for (int st = 0; st < 2; ++st) {
          const half8 bh = join(ph + 4 * st), bl = join(pl + 4 * st);
#pragma unroll
          for (int d = 0; d < kDT; ++d) {
            typedef __attribute__((address_space(3))) short4v lds4;
            short4v a[2];
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              const int tv = 32 * u + 16 * st + 8 * e + vt, c = d * 32 + vc;
              const int off = (tv * kChunks + ((c >> 3) ^ v_swz<D>(tv))) * 16 + (c & 7) * 2;
              a[e] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)((__attribute__((address_space(3))) char*)sv + off));
            }
            const half4 a0 = __builtin_bit_cast(half4, a[0]), a1 = __builtin_bit_cast(half4, a[1]);
            const half8 vf = {a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
            o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, bh, o[d], 0, 0, 0);
            o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, bl, o[d], 0, 0, 0);
          }
        }
      }
    }
    if (it + 1 < iters) store(buf ^ 1);
    __syncthreads();
  }

  float zero[4] = {0.f, 0.f, 0.f, 0.f};  // NaN where a sum is infinite or NaN
#pragma unroll
  for (int d = 0; d < kDT; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) zero[i & 3] = fmaf(o[d][i], 0.f, zero[i & 3]);
  const int odd = __any((zero[0] + zero[1]) + (zero[2] + zero[3]) != 0.f);
  if (lane == 0) s_hi[wave] = odd;  // its bounds were read before the barriers above
  __syncthreads();
  int any = s_hi[0];
#pragma unroll
  for (int w = 1; w < WR * WT; ++w) any |= s_hi[w];
  if (any) {  // block-uniform: the block's rows again, four at a time a wave
#pragma unroll 1
    for (int r0 = wave * kCareful; r0 < WR * 32; r0 += WR * WT * kCareful) {
      const int row0 = rt * (WR * 32) + r0;
      if (row0 >= rows) break;
      const uint16_t* qp[kCareful];
      int64_t qr[kCareful];
      int last[kCareful];
      float m[kCareful], lr[kCareful], acc[kCareful][D / 64];
#pragma unroll
      for (int u = 0; u < kCareful; ++u) {
        const int rw = min(row0 + u, rows - 1);
        qr[u] = (int64_t)(rw / G) * Hq + (int64_t)h * G + rw % G;
        qp[u] = q + qr[u] * D;
        last[u] = min(T, t1) - 1;
        if (causal && qpos) last[u] = min(last[u], __builtin_amdgcn_readfirstlane(qpos[qr[u]]));
      }
      careful_rows<D>(qp, Kh, Vh, stride_t, scale_log2, t0, last, lane, m, lr, acc);
#pragma unroll
      for (int u = 0; u < kCareful; ++u) {
        if (row0 + u >= rows) break;
        if (splits > 1) {
          const int64_t slot = qr[u] * splits + split;
          if (lane == 0) part_ml[2 * slot] = m[u], part_ml[2 * slot + 1] = lr[u];
#pragma unroll
          for (int e = 0; e < D / 64; ++e) part_acc[slot * D + lane * (D / 64) + e] = acc[u][e];
        } else {
#pragma unroll
          for (int e = 0; e < D / 64; ++e)
            out[qr[u] * D + lane * (D / 64) + e] = f2h(lr[u] > 0.f ? acc[u][e] / lr[u] : lr[u] == 0.f ? 0.f : bad);
        }
      }
    }
    return;
  }

  float l = l_run + __shfl_xor(l_run, 32, 64);
  if constexpr (WT > 1) {
    // groups 1.. hand their (m, l, O) to group 0 through LDS, one at a time
    float* const sf = reinterpret_cast<float*>(smem);
    constexpr int kWave = (kDT * 16 + 2) * 64;
    for (int g = 1; g < WT; ++g) {
      if (grp == g) {
        float* w = sf + wr * kWave + lane;
        w[0] = m_run;
        w[64] = l;
#pragma unroll
        for (int d = 0; d < kDT; ++d)
#pragma unroll
          for (int i = 0; i < 16; ++i) w[(2 + d * 16 + i) * 64] = o[d][i];
      }
      __syncthreads();
      if (grp == 0) {
        const float* w = sf + wr * kWave + lane;
        const float m2 = w[0], mn = fmaxf(m_run, m2);
        const float f1 = m_run > -__builtin_inff() ? __builtin_amdgcn_exp2f(m_run - mn) : 0.f;
        const float f2 = m2 > -__builtin_inff() ? __builtin_amdgcn_exp2f(m2 - mn) : 0.f;
        l = l * f1 + w[64] * f2;
#pragma unroll
        for (int d = 0; d < kDT; ++d)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[d][i] = o[d][i] * f1 + w[(2 + d * 16 + i) * 64] * f2;
        m_run = mn;
      }
      __syncthreads();
    }
    if (grp != 0) return;
  }
  if (row >= rows) return;
  if (splits == 1) {
    const float inv = l > 0.f ? 1.f / l : 0.f;  // nothing allowed: zeros (a NaN sum has NaN products, handled above)
#pragma unroll
    for (int d = 0; d < kDT; ++d)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        half4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = (f16)(o[d][4 * g + e] * inv);
        *reinterpret_cast<half4*>(out + qi * D + d * 32 + 8 * g + 4 * hf) = w;
      }
    return;
  }
  const int64_t slot = qi * splits + split;
  if (hf == 0) {
    part_ml[2 * slot] = m_run;
    part_ml[2 * slot + 1] = l;
  }
#pragma unroll
  for (int d = 0; d < kDT; ++d)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float4 w = make_float4(o[d][4 * g], o[d][4 * g + 1], o[d][4 * g + 2], o[d][4 * g + 3]);
      *reinterpret_cast<float4*>(part_acc + slot * D + d * 32 + 8 * g + 4 * hf) = w;
    }
}

// out = sum_s w_s acc_s / sum_s w_s l_s, w_s = exp2(m_s - max m): D/4 threads
// per row, each four coordinates.
template <int D>
__global__ void __launch_bounds__(256)
prompt_merge_kernel(const float* __restrict__ ml, const float* __restrict__ acc, int64_t rows, int splits,
                    float bad, uint16_t* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t r = i / (D / 4);
  const int c = (int)(i % (D / 4)) * 4;
  if (r >= rows) return;
  float mx = -__builtin_inff();
#pragma unroll 8
  for (int s = 0; s < splits; ++s) mx = fmaxf(mx, ml[2 * (r * splits + s)]);
  float l = 0.f;
  float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 8
  for (int s = 0; s < splits; ++s) {
    const float m = ml[2 * (r * splits + s)];
    const float w = m > -__builtin_inff() ? exp2f(m - mx) : 0.f;
    l += ml[2 * (r * splits + s) + 1] * w;
    const float4 v = *reinterpret_cast<const float4*>(acc + (r * splits + s) * D + c);
    a.x += w * v.x, a.y += w * v.y, a.z += w * v.z, a.w += w * v.w;
  }
  const float inv = 1.f / l;
  half4 o = {(f16)(a.x * inv), (f16)(a.y * inv), (f16)(a.z * inv), (f16)(a.w * inv)};
  if (!(l > 0.f)) {  // nothing allowed: zeros; a sum that is no number: bad
    const f16 none = (f16)(l == 0.f ? 0.f : bad);
    o = half4{none, none, none, none};
  }
  *reinterpret_cast<half4*>(out + r * D + c) = o;
}

template <int D, int WR, int WT, int MW>
int launch(const void* q, int B, int Hq, int G, const void* k, const void* v, int T, int Hkv, int64_t stride_t,
           int64_t stride_h, float sl2, int causal, const int32_t* qpos, float bad, void* out, void* ws, int splits,
           hipStream_t s) {
  const int row_tiles = (int)ceil_div((int64_t)B * G, WR * 32);
  const int tps = (int)(ceil_div(ceil_div(T, splits), kTile) * kTile);
  const int64_t slots = (int64_t)B * Hq * splits;
  // partials: acc [slots][D], then (m, l) pairs, which is what the workspace query sizes
  float* acc = (float*)ws;
  hipLaunchKernelGGL((prompt_attn_kernel<D, WR, WT, MW>), dim3((unsigned)Hkv, (unsigned)row_tiles, (unsigned)splits),
                     dim3(WR * WT * 64), 0, s, (const uint16_t*)q, B, Hq, G, (const uint16_t*)k, (const uint16_t*)v, T,
                     stride_t, stride_h, sl2, causal, qpos, row_tiles, tps, splits, bad, (uint16_t*)out,
                     acc + slots * D, acc);
  if (splits > 1) {
    const int64_t rows = (int64_t)B * Hq;
    hipLaunchKernelGGL(prompt_merge_kernel<D>, dim3((unsigned)ceil_div(rows * (D / 4), 256)), dim3(256), 0, s,
                       acc + slots * D, acc, rows, splits, bad, (uint16_t*)out);
  }
  return check_launch("prompt_attention");
}

}  // namespace

bool prompt_attention_ok(const void* q, int64_t B, int Hq, int Hkv, int D, const void* k, const void* v, int64_t T,
                         float sl2, const void* out, const void* ws) {
  auto aligned = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
  // From 4 rows per KV head the tiles win although most of their 64 rows are empty
  // (4 rows, 8 KV heads, 8,192 tokens: 11.7 us against 13.4; 32 rows: 12.9 against
  // 27); one row is faster on the scalar kernel (9.8 against 11.6).  The row maximum
  // is taken before the scale, which therefore has to be positive.
  return (D == 64 || D == 128) && B * (Hq / Hkv) >= 4 && T > 0 && T < (1 << 30) && sl2 > 0.f &&
         sl2 < __builtin_inff() && aligned(q) && aligned(k) && aligned(v) && aligned(out) && aligned(ws);
}

int launch_prompt_attention(const void* q, int B, int Hq, int Hkv, int D, const void* k, const void* v, int64_t T,
                            int64_t stride_t, int64_t stride_h, float sl2, int causal, const int32_t* qpos, float bad,
                            void* out, void* ws, size_t ws_bytes, hipStream_t s) {
  const int G = Hq / Hkv;
  const int64_t rows = (int64_t)B * G;
  // Rows per block: 64 (two token groups share them) fill the chip soonest and waste
  // least on few rows or a short triangle (4,096 rows x 1,024 tokens: 17.3 us against
  // 19.6 with 128 rows); 128 halve the K/V staging of longer windows (4,000 x 3,000:
  // 32.5 us against 33.0 with 256 rows); 256 in 8 waves, four per SIMD, stage it once
  // more seldom where the windows are longest (4,000 x 8,192: 116 us against 123).
  const int wr = D == 64 && rows > 1024 && T > 6144 ? 8 : rows > (D == 64 ? 256 : 64) && T > 1536 ? 4 : 2;
  // Token splits until the blocks fill the 256 CUs (two per CU, one of the 128-row
  // blocks), of at least 256 tokens (512 where the merge has many rows to write).
  const int64_t blocks = ceil_div(rows, 32 * wr) * Hkv, min_tokens = rows <= 64 ? 256 : 512;
  int64_t splits = ceil_div(wr == 4 ? 256 : 512, blocks);
  if (splits > ceil_div(T, min_tokens)) splits = ceil_div(T, min_tokens);
  const int64_t fit = (int64_t)(ws_bytes / ((size_t)B * Hq * (D + 2) * sizeof(float)));
  if (splits > fit) splits = fit;
  if (splits > 64) splits = 64;
  if (splits < 1) splits = 1;
#define RFSN_PROMPT(DD, WR, WT, MW)                                                                                    \
  return launch<DD, WR, WT, MW>(q, B, Hq, G, k, v, (int)T, Hkv, stride_t, stride_h, sl2, causal, qpos, bad, out, ws,   \
                                (int)splits, s)
  if (D == 64) {
    if (wr == 8) RFSN_PROMPT(64, 8, 1, 4);
    if (wr == 4) RFSN_PROMPT(64, 4, 2, 2);
    RFSN_PROMPT(64, 2, 2, 2);
  }
  if (wr == 4) RFSN_PROMPT(128, 4, 2, 2);
  RFSN_PROMPT(128, 2, 2, 2);
#undef RFSN_PROMPT
}

}  // namespace rfsn
