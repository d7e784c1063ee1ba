// The decoder layer's projections (llama32_adapter.py:555-587) for gfx950:
// y = x W^T with fp16 activations and fp32 weights, RMSNorm in front and
// rotary embedding, SwiGLU or the residual add behind, each result rounded to
// fp16 at the reference's cast points.
//
//  - one row (a decode step): linear_row_kernel, fp32 FMAs, one pass over the
//    weights;
//  - more rows: the weights are split on their way to the matrix cores, w =
//    (hi + lo) / scale with hi, lo fp16, and x is exact, so x W^T = MFMA(x, hi)
//    + MFMA(x, lo) in one fp32 accumulator.  At the scale of 2^12 a weight keeps
//    its value to 2^-23 of itself or 2^-37, whichever is more.  A block that
//    holds a row whose largest weight is past fp16's range there, or below
//    2^-12, where 2^-37 is no longer little, repeats its work with each row at a
//    scale of its own: 2^-23 of the weight or 2^-39 of the row's largest.
//    Measured against float64 as the share of fp16 results that are not the
//    nearest: 0.12 to 0.35 % (8 to 1,024 rows, k 2,048 and 8,192), torch's fp32
//    products 0.33 to 0.69 % on the same inputs.
//    An infinite x times lo would cancel or meet 0, so a block that finds a sum
//    that is not finite repeats its work too, with infinities kept from the lo product and
//    hi kept from 0: x W^T is then infinite or NaN as fp32 sums of x w are.
//
// The Llama-3.2-1B layer's seven matrices (243 MB of fp32), torch's fp32 products
// against this file, without the elementwise kernels around the former:
//   1 row      88 -> 50 us (4.8 TB/s; passes in a row find half of the weights in
//              the 256 MB last-level cache: 120 MB come from HBM)
//   1,024 rows 865 -> 298 us (418 TFLOP/s of fp32 products) on their own in a row,
//              345 us in the layer's pass under a kernel trace
#include "rfsn_common.h"
#include "rfsn_internal.h"

#include <type_traits>

namespace rfsn {
namespace {

typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef _Float16 half4 __attribute__((ext_vector_type(4)));
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float2v __attribute__((ext_vector_type(2)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef uint16_t ushort8 __attribute__((ext_vector_type(8)));
typedef uint32_t uint4v __attribute__((ext_vector_type(4)));

constexpr int kModePlain = 0, kModeSwiglu = 1, kModeResidual = 2;

// Output row r of the weights stacked as [w0; w1; w2].
struct Row {
  const float* w;
  uint16_t* out;
  int n, i;
};
__device__ __forceinline__ Row weight_row(const rfsn_linear_params& p, int r) {
  if (r < p.n[0]) return {p.w[0] + (int64_t)r * p.k, (uint16_t*)p.out[0], p.n[0], r};
  r -= p.n[0];
  if (r < p.n[1]) return {p.w[1] + (int64_t)r * p.k, (uint16_t*)p.out[1], p.n[1], r};
  r -= p.n[1];
  return {p.w[2] + (int64_t)r * p.k, (uint16_t*)p.out[2], p.n[2], r};
}

__device__ __forceinline__ uint16_t swiglu(float g, float u) {
  const float gate = h2f(f2h(g));
  const float act = h2f(f2h(gate * (1.f / (1.f + expf(-gate)))));
  return f2h(act * h2f(f2h(u)));
}

// cos, sin of coordinate i < D/2 at row s
__device__ __forceinline__ void rope_angle(const rfsn_linear_params& p, int s, int i, float& c0, float& s0, float& c1,
                                           float& s1) {
  if (p.inv_freq) {
    const double a = (double)(p.pos0 + s) * p.inv_freq[i];
    c0 = c1 = (float)cos(a);
    s0 = s1 = (float)sin(a);
  } else {
    const int D = p.head_dim;
    const int64_t o = (int64_t)s * D + i;
    c0 = p.cos[o], s0 = p.sin[o], c1 = p.cos[o + D / 2], s1 = p.sin[o + D / 2];
  }
}

// ---------------------------------------------------------------- one row
// A wave takes a pair of output rows over a slice of k: 2048 / 64 lanes = 32
// floats of each row per lane and round, 16 loads of 16 bytes in flight.  KS
// waves of the block share a pair (slices of k, summed in LDS).  The pair is
// (j, j + 1), (gate j, up j) under SwiGLU, or the two halves (i, i + D/2) of a
// head where rotary embedding needs both.  The loads carry no branch: with one
// per load they were waited for in turn (gate and up 63 -> 25 us).  Bound: the
// weights' HBM read.
constexpr int kRowSlice = 2048;

template <int MODE, int KS>
__global__ void __launch_bounds__(256, 4) linear_row_kernel(const rfsn_linear_params p, int pairs) {
  extern __shared__ uint16_t xs[];  // x (normed) [k]
  __shared__ float red[4][2];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int pair = blockIdx.x * (4 / KS) + wave / KS, slice = wave % KS;
  const int k = p.k;
  int ra, rb;  // output rows of the pair
  const int rot = MODE == kModePlain ? p.head_dim : 0;
  if (MODE == kModeSwiglu) {
    ra = pair, rb = p.n[0] + pair;
  } else if (rot) {
    ra = pair / (rot / 2) * rot + pair % (rot / 2), rb = ra + rot / 2;
  } else {
    ra = 2 * pair, rb = 2 * pair + 1;
  }
  const bool live = pair < pairs;
  const int total = p.n[0] + p.n[1] + p.n[2];
  Row A = weight_row(p, live ? ra : 0), B = weight_row(p, live && rb < total ? rb : 0);
  const int ks = (k + KS - 1) / KS;              // a slice's share of k (a multiple of 4)
  const int k0 = slice * ks, k1 = min(k, k0 + ks);
  constexpr int U = kRowSlice / 256;
  float4v wa[U], wb[U];
  auto fetch = [&](int base) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = min(base + u * 256 + lane * 4, k - 4);  // no branch: every load is issued at once
      wa[u] = *reinterpret_cast<const float4v*>(A.w + c);
      wb[u] = *reinterpret_cast<const float4v*>(B.w + c);
    }
  };
  fetch(k0);  // in flight while x is normed
  const uint16_t* x = (const uint16_t*)p.x;
  if (p.norm_w) {
    float ss = 0.f;
    for (int c = tid * 4; c < k; c += 1024) {
      const half4 v = *reinterpret_cast<const half4*>(x + c);
#pragma unroll
      for (int e = 0; e < 4; ++e) ss = fmaf((float)v[e], (float)v[e], ss);
    }
    ss = wave_sum(ss);
    if (lane == 0) red[wave][0] = ss;
    __syncthreads();
    const float r = 1.f / sqrtf((red[0][0] + red[1][0] + red[2][0] + red[3][0]) / (float)k + p.norm_eps);
    for (int c = tid * 4; c < k; c += 1024) {
      const half4 v = *reinterpret_cast<const half4*>(x + c);
      const float4v g = *reinterpret_cast<const float4v*>(p.norm_w + c);
      half4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (f16)((float)v[e] * r * g[e]);
      *reinterpret_cast<half4*>(xs + c) = o;
    }
  } else {
    for (int c = tid * 4; c < k; c += 1024) *reinterpret_cast<half4*>(xs + c) = *reinterpret_cast<const half4*>(x + c);
  }
  __syncthreads();
  float a = 0.f, b = 0.f;
  for (int base = k0; base < k1; base += kRowSlice) {
    if (base != k0) fetch(base);
    if (base + kRowSlice > k1) {  // past the slice's end: weights that are not its own, infinite perhaps
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (base + u * 256 + lane * 4 >= k1) wa[u] = wb[u] = (float4v)0.f;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int c = base + u * 256 + lane * 4;
      const half4 v = c < k1 ? *reinterpret_cast<const half4*>(xs + c) : (half4)(f16)0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        a = fmaf(wa[u][e], (float)v[e], a);
        b = fmaf(wb[u][e], (float)v[e], b);
      }
    }
  }
  a = wave_sum(a);
  b = wave_sum(b);
  if constexpr (KS > 1) {
    __syncthreads();  // red was read by the norm
    if (lane == 0) red[wave][0] = a, red[wave][1] = b;
    __syncthreads();
    if (slice != 0) return;
    a = b = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s) a += red[wave + s][0], b += red[wave + s][1];
  }
  if (lane != 0 || !live) return;
  if (MODE == kModeSwiglu) {
    A.out[A.i] = swiglu(a, b);
  } else if (MODE == kModeResidual) {
    const uint16_t* res = (const uint16_t*)p.residual;
    A.out[A.i] = hadd_bits(res[A.i], f2h(a));
    if (rb < total) B.out[B.i] = hadd_bits(res[B.i], f2h(b));
  } else if (rot && ra < p.n[0] + p.n[1]) {
    float c0, s0, c1, s1;
    rope_angle(p, 0, A.i % rot, c0, s0, c1, s1);
    const float va = h2f(f2h(a)), vb = h2f(f2h(b));
    A.out[A.i] = f2h(va * c0 - vb * s0);
    B.out[B.i] = f2h(vb * c1 + va * s1);
  } else {
    A.out[A.i] = f2h(a);
    if (rb < total) B.out[B.i] = f2h(b);
  }
}

// ---------------------------------------------------------------- more rows
__global__ void __launch_bounds__(256)
rms_rows_kernel(const uint16_t* __restrict__ x, int k, const float* __restrict__ w, float eps,
                uint16_t* __restrict__ out) {
  __shared__ float red[4];
  const uint16_t* xr = x + (int64_t)blockIdx.x * k;
  uint16_t* o = out + (int64_t)blockIdx.x * k;
  const int tid = threadIdx.x;
  float ss = 0.f;
  for (int c = tid * 4; c < k; c += 1024) {
    const half4 v = *reinterpret_cast<const half4*>(xr + c);
#pragma unroll
    for (int e = 0; e < 4; ++e) ss = fmaf((float)v[e], (float)v[e], ss);
  }
  ss = wave_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  const float r = 1.f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)k + eps);
  for (int c = tid * 4; c < k; c += 1024) {
    const half4 v = *reinterpret_cast<const half4*>(xr + c);
    const float4v g = *reinterpret_cast<const float4v*>(w + c);
    half4 y;
#pragma unroll
    for (int e = 0; e < 4; ++e) y[e] = (f16)((float)v[e] * r * g[e]);
    *reinterpret_cast<half4*>(o + c) = y;
  }
}

// Rotary embedding in place on q and k: a thread takes one coordinate pair of
// kRopeHeads heads of a row, all loaded before the first is stored.
constexpr int kRopeHeads = 4;
__global__ void __launch_bounds__(256) rope_rows_kernel(const rfsn_linear_params p, int rows, int groups) {
  const int half = p.head_dim / 2, D = p.head_dim, hq = p.n[0] / D, heads = hq + p.n[1] / D;
  const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int i = (int)(id % half), g = (int)(id / half % groups), s = (int)(id / half / groups);
  if (s >= rows) return;
  uint16_t* o[kRopeHeads];
  float a[kRopeHeads], b[kRopeHeads];
#pragma unroll
  for (int u = 0; u < kRopeHeads; ++u) {
    const int h = min(g * kRopeHeads + u, heads - 1);
    o[u] = h < hq ? (uint16_t*)p.out[0] + (int64_t)s * p.n[0] + h * D + i
                  : (uint16_t*)p.out[1] + (int64_t)s * p.n[1] + (h - hq) * D + i;
    a[u] = h2f(o[u][0]);
    b[u] = h2f(o[u][half]);
  }
  float c0, s0, c1, s1;
  rope_angle(p, s, i, c0, s0, c1, s1);
#pragma unroll
  for (int u = 0; u < kRopeHeads; ++u) {
    if (g * kRopeHeads + u >= heads) return;
    o[u][0] = f2h(a[u] * c0 - b[u] * s0);
    o[u][half] = f2h(b[u] * c1 + a[u] * s1);
  }
}

// Scale of the weights: 2^12 for every row at first; where a row's largest weight
// does not suit that (scale_ok), the largest power of two that keeps it below 2^15
// (an infinite weight counts as the largest float, and stays infinite).
constexpr float kScale = 4096.f;
__device__ __forceinline__ bool scale_ok(float wmax) {
  return wmax == 0.f || (wmax >= 0x1p-12f && wmax * kScale < 65504.f);
}
__device__ __forceinline__ float scale_for(float wmax) {
  if (scale_ok(wmax)) return kScale;
  int e = 128;
  if (wmax < __builtin_inff()) frexpf(wmax, &e);  // wmax < 2^e
  return ldexpf(1.f, min(15 - e, 100));
}

// eight consecutive weights as hi and lo halves of w * scale; their maximum folded into wmax
template <bool CAREFUL>
__device__ __forceinline__ void split8(const float4v& a, const float4v& b, float scale, half8& hi, half8& lo,
                                       float& wmax, float minus1) {
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    const float w0 = e < 4 ? a[e] : b[e - 4], w1 = e < 4 ? a[e + 1] : b[e - 3];
    if (!CAREFUL) wmax = fmaxf(fmaxf(wmax, fabsf(w0)), fabsf(w1));
    const float2v s = {w0 * scale, w1 * scale};
    half2v h = __builtin_convertvector(s, half2v);
    if (CAREFUL) {  // hi is 0 for a weight of 0 alone: an infinite x has to meet the others' sign
      if (h[0] == (f16)0.f && w0 != 0.f) h[0] = (f16)copysignf(0x1p-24f, w0);
      if (h[1] == (f16)0.f && w1 != 0.f) h[1] = (f16)copysignf(0x1p-24f, w1);
    }
    float2v r = {fmaf(minus1, (float)h[0], s[0]), fmaf(minus1, (float)h[1], s[1])};
    if (CAREFUL) {  // an infinite weight stays infinite
      if (!(fabsf(s[0]) < __builtin_inff())) r[0] = 0.f;
      if (!(fabsf(s[1]) < __builtin_inff())) r[1] = 0.f;
    }
    const half2v l = __builtin_convertvector(r, half2v);
    hi[e] = h[0], hi[e + 1] = h[1];
    lo[e] = l[0], lo[e + 1] = l[1];
  }
}

// x with 0 for its infinities and NaN: what lo is multiplied by where some may be
__device__ __forceinline__ half8 finite8(half8 x) {
  const ushort8 b = __builtin_bit_cast(ushort8, x);
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = (b[e] & 0x7C00) == 0x7C00 ? (f16)0.f : x[e];
  return x;
}

// Output rows r .. r + 3 (of one matrix: sizes are multiples of 4) at row s of x,
// from sums at the scales 1 / ia (and 1 / iu of the up rows).
template <int MODE>
__device__ __forceinline__ void write4(const rfsn_linear_params& p, float4v acc, float4v up, const float* ia,
                                       const float* iu, int r, int limit, int s, int rows) {
  if (s >= rows || r >= limit) return;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    acc[e] *= ia[e];
    if (MODE == kModeSwiglu) up[e] *= iu[e];
  }
  uint16_t v[4];
  int i = r, t = 0;
  if (MODE == kModeSwiglu) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = swiglu(acc[e], up[e]);
  } else {
    while (t < 2 && i >= p.n[t]) i -= p.n[t++];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = f2h(acc[e]);
  }
  const int64_t o = (int64_t)s * p.n[t] + i;
  if (MODE == kModeResidual) {
    const uint2 w = *reinterpret_cast<const uint2*>((const uint16_t*)p.residual + o);
    v[0] = hadd_bits((uint16_t)w.x, v[0]), v[1] = hadd_bits((uint16_t)(w.x >> 16), v[1]);
    v[2] = hadd_bits((uint16_t)w.y, v[2]), v[3] = hadd_bits((uint16_t)(w.y >> 16), v[3]);
  }
  *reinterpret_cast<uint2*>((uint16_t*)p.out[t] + o) =
      make_uint2(v[0] | (uint32_t)v[1] << 16, v[2] | (uint32_t)v[3] << 16);
}

// The same for a 32x32 accumulator: output rows r0 + 8 g + 4 hf + e, column s.
template <int MODE>
__device__ __forceinline__ void write_tile(const rfsn_linear_params& p, const float16v& acc, const float16v& up,
                                           const float* ia, const float* iu, int r0, int limit, int s, int rows,
                                           int hf) {
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const float4v a = {acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
    const float4v b = {up[4 * g], up[4 * g + 1], up[4 * g + 2], up[4 * g + 3]};
    const int r = 8 * g + 4 * hf;
    write4<MODE>(p, a, b, ia + r, iu + r, r0 + r, limit, s, rows);
  }
}

// Few rows (at most 16 CT): the weights stream once from HBM straight into
// MFMA operands, without LDS.  A block takes 16 output rows (16 gate and 16 up
// rows under SwiGLU), its W waves every W-th run of 128 k: lane (row, quarter
// q) loads k 32 q .. 32 q + 31 of its row, 128 contiguous bytes, and k step j
// of both operands is the lane's values 8 j .. 8 j + 7.  The next run's weights
// are requested before this one's are used; the waves' sums meet in LDS.
// Bound: HBM; 8 KB per wave, matrix and run in flight.  16 rows: 90 us for the
// layer's matrices; 32x32 tiles without the early request took 180 us.
template <int MODE, int CT, int W>
__global__ void __launch_bounds__(W * 64)
linear_skinny_kernel(const rfsn_linear_params p, const uint16_t* __restrict__ x, int rows) {
  constexpr int AN = MODE == kModeSwiglu ? 2 : 1;
  __shared__ float4v sums[W][AN * CT][64];
  __shared__ int again;
  __shared__ int row_max[AN * 16];
  __shared__ float row_inv[AN * 16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, q = lane >> 4;
  const int limit = MODE == kModeSwiglu ? p.n[0] : p.n[0] + p.n[1] + p.n[2];
  const int r0 = blockIdx.x * 16;
  const float* wp[AN];
  wp[0] = weight_row(p, min(r0 + col, limit - 1)).w + 32 * q;
  if (AN == 2) wp[AN - 1] = p.w[1] + (int64_t)min(r0 + col, limit - 1) * p.k + 32 * q;
  const uint16_t* xp[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) xp[c] = x + (int64_t)min(c * 16 + col, rows - 1) * p.k + 32 * q;
  float minus1 = -1.f;
  asm("" : "+s"(minus1));
  float scale[AN];
  scale[0] = scale[AN - 1] = kScale;
  if (threadIdx.x == 0) again = 0;
  if (threadIdx.x < AN * 16) {
    row_max[threadIdx.x] = 0;
    row_inv[threadIdx.x] = 1.f / kScale;
  }
  float wmax[AN];
  wmax[0] = wmax[AN - 1] = 0.f;
  float4v acc[AN][CT];
  auto run = [&](auto careful) {
    constexpr bool kCareful = decltype(careful)::value;
#pragma unroll
    for (int a = 0; a < AN; ++a)
#pragma unroll
      for (int c = 0; c < CT; ++c) acc[a][c] = (float4v)0.f;
    float4v wv[AN][8];
    auto fetch = [&](int kb) {
#pragma unroll
      for (int a = 0; a < AN; ++a)
#pragma unroll
        for (int u = 0; u < 8; ++u) wv[a][u] = *reinterpret_cast<const float4v*>(wp[a] + kb + 4 * u);
    };
    int kb = wave * 128;
    if (kb < p.k) fetch(kb);
    while (kb < p.k) {
      uint4v xv[CT][4];
#pragma unroll
      for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int u = 0; u < 4; ++u) xv[c][u] = *reinterpret_cast<const uint4v*>(xp[c] + kb + 8 * u);
      half8 hi[AN][4], lo[AN][4];
#pragma unroll
      for (int a = 0; a < AN; ++a)
#pragma unroll
        for (int u = 0; u < 4; ++u)
          split8<kCareful>(wv[a][2 * u], wv[a][2 * u + 1], scale[a], hi[a][u], lo[a][u], wmax[a], minus1);
      kb += W * 128;
      if (kb < p.k) fetch(kb);
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int c = 0; c < CT; ++c) {
          const half8 xf = __builtin_bit_cast(half8, xv[c][u]), xl = kCareful ? finite8(xf) : xf;
#pragma unroll
          for (int a = 0; a < AN; ++a) {
            acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi[a][u], xf, acc[a][c], 0, 0, 0);
            acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo[a][u], xl, acc[a][c], 0, 0, 0);
          }
        }
    }
  };
  run(std::false_type{});
  float zero[4] = {0.f, 0.f, 0.f, 0.f};  // NaN where a sum is infinite or NaN
#pragma unroll
  for (int a = 0; a < AN; ++a)
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) zero[i] = fmaf(acc[a][c][i], 0.f, zero[i]);
  __syncthreads();  // row_max and again hold their first values
#pragma unroll
  for (int a = 0; a < AN; ++a)
    atomicMax(&row_max[a * 16 + col], __builtin_bit_cast(int, wmax[a]));  // wmax >= 0: ordered as its bits
  if ((zero[0] + zero[1]) + (zero[2] + zero[3]) != 0.f) again = 1;
  __syncthreads();
  if (threadIdx.x < AN * 16 && !scale_ok(__builtin_bit_cast(float, row_max[threadIdx.x]))) again = 1;
  __syncthreads();
  if (again) {  // block-uniform
#pragma unroll
    for (int a = 0; a < AN; ++a) {
      scale[a] = scale_for(__builtin_bit_cast(float, row_max[a * 16 + col]));
      if (q == 0) row_inv[a * 16 + col] = 1.f / scale[a];
    }
    run(std::true_type{});
  }
#pragma unroll
  for (int a = 0; a < AN; ++a)
#pragma unroll
    for (int c = 0; c < CT; ++c) sums[wave][a * CT + c][lane] = acc[a][c];
  __syncthreads();
  if (wave >= CT) return;
  // wave c finishes column tile c
  float4v t[AN];
#pragma unroll
  for (int a = 0; a < AN; ++a) {
    t[a] = sums[0][a * CT + wave][lane];
#pragma unroll
    for (int w = 1; w < W; ++w) t[a] += sums[w][a * CT + wave][lane];
  }
  write4<MODE>(p, t[0], t[AN - 1], row_inv + 4 * q, row_inv + (AN - 1) * 16 + 4 * q, r0 + 4 * q, limit,
               wave * 16 + col, rows);
}

// Many rows: 64 CT rows of x by AN * 64 output rows per block (64 gate and 64 up
// rows under SwiGLU), two groups of 4 waves that take k runs of 32 in turn (an
// in-block split of k: with one block or two per CU every SIMD then has two
// waves or more), W split into its hi and lo planes on its way to LDS.
// No unit is full: at 1,024 rows the matrix cores are busy 39, 42 and 50 % of the
// cycles (q, k and v; down; gate and up), VALU issue 30 %, LDS 32, 43 and 28 %, and
// a SIMD's two waves wait 27 to 36 % of theirs between the barriers.  Gate and up
// run at 830 to 950 TFLOP/s of issued MFMAs (145 to 166 us by box and clock; 228 us
// before the loads ran two stages ahead and the row tiles of a panel shared an XCD).
template <int MODE, int AN, int CT, int kBK>
__global__ void __launch_bounds__(512, AN == 1 && kBK == 32 ? 4 : 2)
linear_tiles_kernel(const rfsn_linear_params p, const uint16_t* __restrict__ x, int rows, int row_tiles, int panels) {
  constexpr int kG = 2, TN = AN * 64, TS = CT * 64, kRow = kBK / 8;
  constexpr int kWv = TN * kRow, kXv = TS * kRow;                    // 16-byte units of a plane of W, of X
  constexpr int kStage = 2 * kWv + kXv;
  // X comes from L2: where its two register sets would spill, one stage ahead is enough
  constexpr int kXS = CT == 4 ? 1 : 2;
  constexpr int kWL = TN * kBK / 8 / 256, kXL = TS * kBK / 8 / 256;  // 8-element units a thread stages
  __shared__ uint4v smem[kG * 2 * kStage];
  __shared__ int again;
  __shared__ int row_max[TN];
  __shared__ float row_inv[TN];
  static_assert(sizeof(smem) >= 256 * 16 * AN * CT * 4, "the groups' sums fit the staging buffers");
  const int grp = threadIdx.x >> 8, tid = threadIdx.x & 255, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wn = wave & 1, ws = wave >> 1;
  const int col = lane & 31, hf = lane >> 5;
  const int limit = MODE == kModeSwiglu ? p.n[0] : p.n[0] + p.n[1] + p.n[2];
  // The row tiles that share a weight panel run together on one XCD (block ids go
  // round the 8 XCDs), so a panel passes from HBM into one L2, once.
  const int xcd = blockIdx.x & 7, seq = blockIdx.x >> 3;
  const int st = seq % row_tiles, nt = seq / row_tiles * 8 + xcd;
  if (nt >= panels) return;
  const int s0 = st * TS, n0 = nt * (MODE == kModeSwiglu ? TN / 2 : TN);
  uint4v* const sg = smem + grp * 2 * kStage;
  // 16-byte unit c of row r sits at r kRow + (c ^ swz(r)): 16 rows of one unit touch every bank once
  auto at = [](int r, int c) { return r * kRow + (c ^ (kBK == 32 ? (r >> 2) & 3 : (r >> 1) & 7)); };
  // staged rows of the thread: unit i = u * 256 + tid is row i / kRow, k 8 (i % kRow)
  const float* wrow[kWL];
#pragma unroll
  for (int u = 0; u < kWL; ++u) {
    const int r = (u * 256 + tid) / kRow;
    if (MODE == kModeSwiglu) {  // rows 64 wn' + 32 a + j: a = 0 gate, a = 1 up
      const int half = (r >> 5) & 1, j = (r >> 6) * 32 + (r & 31);
      wrow[u] = p.w[half] + (int64_t)min(n0 + j, limit - 1) * p.k;
    } else {
      wrow[u] = weight_row(p, min(n0 + r, limit - 1)).w;
    }
  }
  const uint16_t* xrow[kXL];
#pragma unroll
  for (int u = 0; u < kXL; ++u) xrow[u] = x + (int64_t)min(s0 + ((u * 256 + tid) / kRow), rows - 1) * p.k;
  const int kc = tid % kRow * 8;
  float minus1 = -1.f;
  asm("" : "+s"(minus1));
  float scale[kWL];
#pragma unroll
  for (int u = 0; u < kWL; ++u) scale[u] = kScale;
  if (threadIdx.x == 0) again = 0;
  if (threadIdx.x < TN) {
    row_max[threadIdx.x] = 0;
    row_inv[threadIdx.x] = 1.f / kScale;
  }
  float wmax[kWL];
#pragma unroll
  for (int u = 0; u < kWL; ++u) wmax[u] = 0.f;
  float16v acc[AN][CT];
  const int iters = p.k / (kBK * kG);  // the launch takes a kBK that divides k evenly

  auto run = [&](auto careful) {
    constexpr bool kCareful = decltype(careful)::value;
#pragma unroll
    for (int a = 0; a < AN; ++a)
#pragma unroll
      for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[a][c][i] = 0.f;
    // two register sets in front of the two LDS buffers: stage it + 3 is requested when
    // stage it + 1 goes to LDS.  No branch inside: past the end the last stage is loaded
    // and stored again, unread, which keeps the vmcnt waits exact and lets the
    // conversions of one stage overlap the products of another.
    float4v wv[2][kWL][2];
    uint4v xv[kXS][kXL];
    auto fetch_x = [&](int it, auto set) {
      constexpr int R = decltype(set)::value % kXS;
      const int kb = (min(it, iters - 1) * kG + grp) * kBK + kc;
#pragma unroll
      for (int u = 0; u < kXL; ++u) xv[R][u] = *reinterpret_cast<const uint4v*>(xrow[u] + kb);
    };
    auto fetch_w = [&](int it, auto set) {
      constexpr int R = decltype(set)::value;
      const int kb = (min(it, iters - 1) * kG + grp) * kBK + kc;
#pragma unroll
      for (int u = 0; u < kWL; ++u) {
        wv[R][u][0] = *reinterpret_cast<const float4v*>(wrow[u] + kb);
        wv[R][u][1] = *reinterpret_cast<const float4v*>(wrow[u] + kb + 4);
      }
    };
    auto fetch = [&](int it, auto set) {  // it >= 1 with one X set
      fetch_w(it, set);
      fetch_x(kXS == 2 ? it : it - 1, set);
    };
    auto store = [&](auto set) {
      constexpr int R = decltype(set)::value;
      uint4v* const s = sg + R * kStage;
#pragma unroll
      for (int u = 0; u < kWL; ++u) {
        const int i = at((u * 256 + tid) / kRow, tid % kRow);
        half8 hi, lo;
        split8<kCareful>(wv[R][u][0], wv[R][u][1], scale[u], hi, lo, wmax[u], minus1);
        // the units in turn: left to interleave their maxima, the compiler waits for LDS more
        // often (gate and up, 1,024 rows: 151 -> 145 us; 128 rows: 37.4 -> 34.3)
        if (!kCareful && u + 1 < kWL) asm("" : "+v"(wmax[u + 1]), "+v"(wv[R][u + 1][0]) : "v"(wmax[u]));
        s[i] = __builtin_bit_cast(uint4v, hi);
        s[kWv + i] = __builtin_bit_cast(uint4v, lo);
      }
#pragma unroll
      for (int u = 0; u < kXL; ++u) s[2 * kWv + at((u * 256 + tid) / kRow, tid % kRow)] = xv[R % kXS][u];
    };
    auto products = [&](auto set) {
      const uint4v* const s = sg + decltype(set)::value * kStage;
#pragma unroll
      for (int ks = 0; ks < kBK / 16; ++ks) {
        half8 xf[CT];
#pragma unroll
        for (int c = 0; c < CT; ++c) {
          xf[c] = __builtin_bit_cast(half8, s[2 * kWv + at(ws * (CT * 32) + c * 32 + col, 2 * ks + hf)]);
        }
#pragma unroll
        for (int a = 0; a < AN; ++a) {
          const int i = at(wn * AN * 32 + a * 32 + col, 2 * ks + hf);
          const half8 hi = __builtin_bit_cast(half8, s[i]), lo = __builtin_bit_cast(half8, s[kWv + i]);
#pragma unroll
          for (int c = 0; c < CT; ++c) acc[a][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(hi, xf[c], acc[a][c], 0, 0, 0);
#pragma unroll
          for (int c = 0; c < CT; ++c)
            acc[a][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo, kCareful ? finite8(xf[c]) : xf[c], acc[a][c], 0, 0, 0);
        }
      }
    };
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    fetch_w(0, even);
    fetch_x(0, even);
    fetch_w(1, odd);
    if (kXS == 2) fetch_x(1, odd);
    store(even);
    fetch(2, even);
    __syncthreads();
    int it = 0;
    for (; it + 1 < iters; it += 2) {
      products(even);
      store(odd);
      fetch(it + 3, odd);
      __syncthreads();
      products(odd);
      store(even);
      fetch(it + 4, even);
      __syncthreads();
    }
    if (it < iters) products(even);
  };
  run(std::false_type{});
  float zero[4] = {0.f, 0.f, 0.f, 0.f};  // NaN where a sum is infinite or NaN
#pragma unroll
  for (int a = 0; a < AN; ++a)
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int i = 0; i < 16; ++i) zero[i & 3] = fmaf(acc[a][c][i], 0.f, zero[i & 3]);
#pragma unroll
  for (int u = 0; u < kWL; ++u)  // wmax >= 0: ordered as its bits
    atomicMax(&row_max[(u * 256 + tid) / kRow], __builtin_bit_cast(int, wmax[u]));
  if ((zero[0] + zero[1]) + (zero[2] + zero[3]) != 0.f) again = 1;
  __syncthreads();
  if (threadIdx.x < TN && !scale_ok(__builtin_bit_cast(float, row_max[threadIdx.x]))) again = 1;
  __syncthreads();
  if (again) {  // block-uniform
#pragma unroll
    for (int u = 0; u < kWL; ++u) {
      const int r = (u * 256 + tid) / kRow;
      scale[u] = scale_for(__builtin_bit_cast(float, row_max[r]));
      row_inv[r] = 1.f / scale[u];  // the row's threads agree
    }
    run(std::true_type{});
    __syncthreads();
  }
  float* m = reinterpret_cast<float*>(smem) + wave * AN * CT * 16 * 64 + lane;
  if (grp == 1) {
#pragma unroll
    for (int a = 0; a < AN; ++a)
#pragma unroll
      for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int i = 0; i < 16; ++i) m[((a * CT + c) * 16 + i) * 64] = acc[a][c][i];
  }
  __syncthreads();
  if (grp == 1) return;
  const float* ri = row_inv + wn * AN * 32;  // the wave's staged rows (32 gate, then 32 up, under SwiGLU)
#pragma unroll
  for (int c = 0; c < CT; ++c) {
#pragma unroll
    for (int a = 0; a < AN; ++a)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][c][i] += m[((a * CT + c) * 16 + i) * 64];
    const int s = s0 + ws * (CT * 32) + c * 32 + col;
    if (MODE == kModeSwiglu) {
      write_tile<MODE>(p, acc[0][c], acc[AN - 1][c], ri, ri + 32, n0 + wn * 32, limit, s, rows, hf);
    } else {
#pragma unroll
      for (int a = 0; a < AN; ++a)
        write_tile<MODE>(p, acc[a][c], acc[a][c], ri + a * 32, ri, n0 + wn * AN * 32 + a * 32, limit, s, rows, hf);
    }
  }
}

template <int MODE>
int launch_linear(const rfsn_linear_params& p, hipStream_t s) {
  const int rows = (int)p.rows, k = p.k;
  const int limit = MODE == kModeSwiglu ? p.n[0] : p.n[0] + p.n[1] + p.n[2];
  if (rows == 1) {
    const int pairs = MODE == kModeSwiglu ? p.n[0] : (limit + 1) / 2;
    const size_t lds = (size_t)k * 2;
    if (k >= 8192 && k % 16 == 0)
      hipLaunchKernelGGL((linear_row_kernel<MODE, 4>), dim3((unsigned)pairs), dim3(256), lds, s, p, pairs);
    else
      hipLaunchKernelGGL((linear_row_kernel<MODE, 1>), dim3((unsigned)ceil_div(pairs, 4)), dim3(256), lds, s, p, pairs);
    return check_launch("layer_linear");
  }
  const uint16_t* x = (const uint16_t*)p.x;
  if (p.norm_w) {
    hipLaunchKernelGGL(rms_rows_kernel, dim3((unsigned)rows), dim3(256), 0, s, x, k, p.norm_w, p.norm_eps,
                       (uint16_t*)p.xn);
    x = (const uint16_t*)p.xn;
  }
  constexpr int AN = MODE == kModeSwiglu ? 2 : 1;
  // Up to 64 rows the weights' one read is the cost: stream them through registers
  // (64 rows: 134 us against 166 us for the tiles' fixed 128 rows).  Past that the
  // tiles' reuse of W in LDS pays.
  if (rows <= 64 && k % 128 == 0) {
    const unsigned grid = (unsigned)ceil_div(limit, 16);
#define RFSN_SKINNY(CT, W)                                                                                           \
  hipLaunchKernelGGL((linear_skinny_kernel<MODE, CT, W>), dim3(grid), dim3(W * 64), 0, s, p, x, rows)
    if (rows <= 16)
      RFSN_SKINNY(1, 16 / AN);
    else if (rows <= 32)
      RFSN_SKINNY(2, 16 / AN);
    else
      RFSN_SKINNY(4, 8);
#undef RFSN_SKINNY
  } else {
    // Blocks run 256 at a time (LDS leaves one per CU).  Twice the tile costs 1.7 to
    // 1.8 times the round, as its waves read less LDS per MFMA, and pays where it
    // halves the rounds: gate and up at 1,024 rows 170 -> 156 us (768 rows, two
    // rounds against three: 133 -> 143), qkv at 1,024 rows 56 -> 50 us.
    auto blocks = [&](int out_rows, int x_rows) {
      return ceil_div(ceil_div(limit, out_rows), 8) * 8 * ceil_div(rows, x_rows);
    };
#define RFSN_TILES(A, CT, BK)                                                                                          \
  do {                                                                                                                 \
    const int panels = (int)ceil_div(limit, MODE == kModeSwiglu ? 32 * A : 64 * A);                                    \
    const int row_tiles = (int)ceil_div(rows, CT * 64);                                                                \
    hipLaunchKernelGGL((linear_tiles_kernel<MODE, A, CT, BK>), dim3((unsigned)(row_tiles * ceil_div(panels, 8) * 8)),  \
                       dim3(512), 0, s, p, x, rows, row_tiles, panels);                                                \
  } while (0)
    if constexpr (MODE == kModeSwiglu) {
      if (16 * ceil_div(blocks(64, 256), 256) < 9 * ceil_div(blocks(64, 128), 256))
        RFSN_TILES(2, 4, 32);
      else
        RFSN_TILES(2, 2, 32);
    } else {
      if (17 * ceil_div(blocks(128, 128), 256) < 10 * ceil_div(blocks(64, 128), 256))
        RFSN_TILES(2, 2, 32);
      else if (k % 128 == 0)
        RFSN_TILES(1, 2, 64);
      else
        RFSN_TILES(1, 2, 32);
    }
#undef RFSN_TILES
  }
  if (MODE == kModePlain && p.head_dim) {
    const int groups = (int)ceil_div((p.n[0] + p.n[1]) / p.head_dim, kRopeHeads);
    hipLaunchKernelGGL(rope_rows_kernel, dim3((unsigned)ceil_div((int64_t)rows * groups * (p.head_dim / 2), 256)),
                       dim3(256), 0, s, p, rows, groups);
  }
  return check_launch("layer_linear");
}

}  // namespace
}  // namespace rfsn

using namespace rfsn;

extern "C" int rfsn_layer_linear(const rfsn_linear_params* p, void* stream) {
  RFSN_REQUIRE(p && p->x && p->w[0] && p->out[0], "layer_linear: null pointer");
  RFSN_REQUIRE(p->rows >= 0 && p->rows < (1 << 24) && p->k >= 64 && p->k % 64 == 0 && p->k <= 32768,
               "layer_linear: k must be a multiple of 64 in [64, 32768]");
  int64_t total = 0;
  for (int t = 0; t < 3; ++t) {
    RFSN_REQUIRE(p->n[t] >= 0 && p->n[t] % 4 == 0 && (p->n[t] == 0 || (p->w[t] && (p->out[t] || p->mode == kModeSwiglu))),
                 "layer_linear: output sizes must be multiples of 4 with weights and outputs");
    total += p->n[t];
  }
  RFSN_REQUIRE(p->n[0] > 0 && total < (1 << 28) && (p->n[2] == 0 || p->n[1] > 0), "layer_linear: bad output sizes");
  auto aligned = [](const void* q, uintptr_t a) { return ((uintptr_t)q & (a - 1)) == 0; };
  bool ok = aligned(p->x, 16) && aligned(p->norm_w, 16) && aligned(p->residual, 8) && aligned(p->xn, 16);
  for (int t = 0; t < 3; ++t) ok = ok && aligned(p->w[t], 16) && aligned(p->out[t], 8);
  RFSN_REQUIRE(ok, "layer_linear: buffers must be 16-byte aligned (outputs and residual 8)");
  RFSN_REQUIRE(!p->norm_w || p->rows <= 1 || p->xn, "layer_linear: a norm of several rows needs the xn buffer");
  if (p->mode == kModePlain) {
    if (p->head_dim) {
      RFSN_REQUIRE(p->head_dim % 8 == 0 && p->n[0] % p->head_dim == 0 && p->n[1] % p->head_dim == 0 &&
                       p->n[2] % p->head_dim == 0,
                   "layer_linear: rotary embedding needs whole heads");
      RFSN_REQUIRE(p->inv_freq || (p->cos && p->sin), "layer_linear: rotary embedding needs frequencies or tables");
    }
  } else if (p->mode == kModeSwiglu) {
    RFSN_REQUIRE(p->n[1] == p->n[0] && p->n[2] == 0 && p->head_dim == 0, "layer_linear: SwiGLU takes two equal matrices");
  } else {
    RFSN_REQUIRE(p->mode == kModeResidual && p->residual && p->n[1] == 0 && p->n[2] == 0 && p->head_dim == 0,
                 "layer_linear: the residual add takes one matrix");
  }
  if (p->rows == 0) return RFSN_OK;
  hipStream_t s = (hipStream_t)stream;
  if (p->mode == kModeSwiglu) return launch_linear<kModeSwiglu>(*p, s);
  if (p->mode == kModeResidual) return launch_linear<kModeResidual>(*p, s);
  return launch_linear<kModePlain>(*p, s);
}
