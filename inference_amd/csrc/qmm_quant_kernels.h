// Quantizers, layout conversion and dequantization kernels (gfx950).
//
// Activation quantizers follow the vec-dot types of Candle's CPU quantized
// matmul (candle-core quantized/k_quants.rs @1e6aa85e, Cargo.toml:54):
//   BlockQ8K::from_float  -- activations of Q4_K / Q6_K weights
//   BlockQ8_0::from_float -- activations (and weights) of Q8_0
// Weight quantizers restate BlockQ4K::from_float / BlockQ6K::from_float with
// their helpers make_qkx1_quants / make_qx_quants (quantized/utils.rs) step by
// step, because their output bytes depend on the exact f32 operation order.
// Every f32 operation in those functions is a single IEEE-rounded operation
// (contraction off, correctly rounded division), so the bytes match the CPU's.
// Byte layouts: crates/media/candle-gen/vendor/candle-kernels/src/quantized.cu:329-433.
#pragma once

#include "qmm_common.h"

namespace qmm {

// ---------------------------------------------------------------------------
// Q8_K activation quantizer: one wave per 256-element block.
//   max   = the element of largest |x| (the first one on ties)
//   iscale = -128 / max, q = min(127, round(iscale * x)) (ties away from zero)
//   bsums[j] = sum of q[16j .. 16j+16), d = 1 / iscale; an all-zero block is all zeros.
// ---------------------------------------------------------------------------
// Lane-local result of quantizing one 256-element block (lane owns elements
// 4*lane .. 4*lane+3).
// silu(g) * u as LlamaMlp::forward computes it (crates/llm/candle-llm/src/models/llama.rs:1386-1391):
// g / (1 + exp(-g)) * u, each operation rounded on its own.
__device__ __forceinline__ float silu_mul(float g, float u) {
#pragma clang fp contract(off)
  return g / (1.0f + expf(-g)) * u;
}

struct Q8KLane {
  uint32_t packed;  // its four int8 quants
  int sum16;        // sum of the 16-element group it belongs to
  float d;
};

__device__ __forceinline__ Q8KLane q8k_lane_vals(float e0, float e1, float e2, float e3, int lane) {
#pragma clang fp contract(off)
  const float amax = wave_max(fmaxf(fmaxf(fabsf(e0), fabsf(e1)), fmaxf(fabsf(e2), fabsf(e3))));
  Q8KLane r;
  if (amax == 0.0f) {
    r.packed = 0u;
    r.sum16 = 0;
    r.d = 0.0f;
    return r;
  }
  const int mine = fabsf(e0) == amax ? 0 : fabsf(e1) == amax ? 1 : fabsf(e2) == amax ? 2 : fabsf(e3) == amax ? 3 : 4;
  const int idx = wave_min(mine < 4 ? 4 * lane + mine : 256);
  const float cand = (idx & 3) == 0 ? e0 : (idx & 3) == 1 ? e1 : (idx & 3) == 2 ? e2 : e3;
  const float mx = readlane_f(cand, idx >> 2);
  const float iscale = -128.0f / mx;
  const float e[4] = {e0, e1, e2, e3};
  uint32_t packed = 0;
  int sum = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float v = roundf(iscale * e[j]);
    v = fminf(v, 127.0f);
    int q = (int)v;
    q = q < -128 ? -128 : q;
    sum += q;
    packed |= (uint32_t)(q & 0xff) << (8 * j);
  }
  r.packed = packed;
  r.sum16 = quad_sum(sum);
  r.d = 1.0f / iscale;
  return r;
}

__device__ __forceinline__ Q8KLane q8k_lane(const float* __restrict__ xs, int lane) {
  return q8k_lane_vals(xs[4 * lane], xs[4 * lane + 1], xs[4 * lane + 2], xs[4 * lane + 3], lane);
}

// Standalone form: one wave writes one GGML Q8_K block.
__device__ __forceinline__ void q8k_block(const float* __restrict__ xs, uint8_t* __restrict__ blk, int lane) {
  const Q8KLane q = q8k_lane(xs, lane);
  reinterpret_cast<uint32_t*>(blk + 4)[lane] = q.packed;
  const int next = __shfl_down(q.sum16, 4);
  if ((lane & 7) == 0)
    reinterpret_cast<uint32_t*>(blk + 4 + 256)[lane >> 3] = ((uint32_t)q.sum16 & 0xffffu) | ((uint32_t)next << 16);
  if (lane == 0) *reinterpret_cast<float*>(blk) = q.d;
}

// ---------------------------------------------------------------------------
// Q8_0 quantizer (activations and weights): 8 lanes per 32-element block.
//   d = amax / 127, q = round(x * (1/d)) (0 when d == 0), d stored as f16.
// Writes GGML 34-byte blocks.
// ---------------------------------------------------------------------------
// Lane l (of the block's 8): its four quants; *dh the block's f16 scale.
__device__ __forceinline__ uint32_t q80_lane(const float (&e)[4], uint16_t* dh) {
#pragma clang fp contract(off)
  float amax = 0.0f;
#pragma unroll
  for (int j = 0; j < 4; ++j) amax = fmaxf(amax, fabsf(e[j]));
  amax = fmaxf(amax, dpp_f<0xb1>(amax));   // max over the 8 lanes of the block
  amax = fmaxf(amax, dpp_f<0x4e>(amax));
  amax = fmaxf(amax, dpp_f<0x141>(amax));
  const float d = amax / 127.0f;
  const float id = d != 0.0f ? 1.0f / d : 0.0f;
  *dh = f2h(d);
  uint32_t q4 = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float r = roundf(e[j] * id);
    r = fminf(fmaxf(r, -128.0f), 127.0f);
    q4 |= (uint32_t)((int)r & 0xff) << (8 * j);
  }
  return q4;
}

__device__ __forceinline__ void q80_block(const float* __restrict__ xs, uint8_t* __restrict__ blk,
                                          int l, bool valid) {
  float e[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) e[j] = valid ? xs[4 * l + j] : 0.0f;
  uint16_t d;
  const uint32_t q4 = q80_lane(e, &d);
  if (!valid) return;
  uint16_t* p = reinterpret_cast<uint16_t*>(blk);
  if (l == 0) p[0] = d;
  p[1 + 2 * l] = (uint16_t)(q4 & 0xffff);
  p[2 + 2 * l] = (uint16_t)(q4 >> 16);
}

// ---------------------------------------------------------------------------
// Weight quantizers: one lane per sub-block (32 values of a Q4_K block, 16 of a
// Q6_K block), its values and codes in registers, every loop over them unrolled.
// The fits are sequential f32 sums that have to keep their order, so a lane is
// the smallest unit; the lanes of a block then agree on the block's scales with
// DPP exchanges and write its bytes 16 at a time.
//
// What bounds them: VALU issue (Q4_K: five passes of ~12 instructions a value).
// A wave stages its 64 sub-blocks through LDS, because a lane's own values are
// contiguous and reading them directly would touch 64 lines per load.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int round_i(float v) {
  // f32::round (ties away from zero) then a saturating cast to i32.
  const float r = roundf(v);
  if (!(r == r)) return 0;
  if (r >= 2147483647.0f) return 2147483647;
  if (r <= -2147483648.0f) return (int)0x80000000;
  return (int)r;
}

// round(v) clamped to [0, hi] as an integer-valued float: f32::round (ties away
// from zero) and a saturating cast, of which NaN gives 0. For v >= 0 that is
// floor(v + 0.5 - 2^-25): the sum rounds up to the next integer exactly from
// .5 on (with 0.5 itself 0.5 - 2^-25 would round to 1).
__device__ __forceinline__ float round_to(float v, float hi) {
  return fminf(floorf(fmaxf(v, 0.0f) + 0.49999997f), hi);
}

// The same for a signed range.
__device__ __forceinline__ float round_between(float v, float lo, float hi) {
  const float r = fminf(fmaxf(truncf(v + copysignf(0.49999997f, v)), lo), hi);
  return v == v ? r : 0.0f;
}

// Asymmetric fit of 32 values to [0, 15] codes, five tries (make_qkx1_quants);
// returns the scale and the (positive) offset `-min`.
__device__ __forceinline__ float fit_q4(const float (&x)[32], float* neg_min) {
#pragma clang fp contract(off)
  float c[32];
  float lo = x[0], hi = x[0];
#pragma unroll
  for (int i = 1; i < 32; ++i) {
    if (x[i] < lo) lo = x[i];
    if (x[i] > hi) hi = x[i];
  }
#pragma unroll
  for (int i = 0; i < 32; ++i) c[i] = 0.0f;
  *neg_min = 0.0f;
  if (hi == lo) return 0.0f;
  float mn = fminf(lo, 0.0f);
  float iscale = 15.0f / (hi - mn);
  float scale = 1.0f / iscale;
#pragma unroll 1
  for (int it = 0; it < 5; ++it) {
    float sumlx = 0.0f, suml2 = 0.0f;  // suml2 counts exactly: at most 32 * 225
    bool changed = false;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      const float d = x[i] - mn, n = round_to(iscale * d, 15.0f);
      changed |= n != c[i];
      c[i] = n;
      sumlx += d * n;
      suml2 += n * n;
    }
    scale = sumlx / suml2;
    float acc = 0.0f;
#pragma unroll
    for (int i = 0; i < 32; ++i) acc += x[i] - scale * c[i];
    mn = acc / 32.0f;
    if (mn > 0.0f) mn = 0.0f;
    iscale = 1.0f / scale;
    if (!changed) break;
  }
  *neg_min = -mn;
  return scale;
}

__device__ __forceinline__ void q4k_scale_min(int j, const uint8_t* s, int* sc, int* m) {
  if (j < 4) {
    *sc = s[j] & 63;
    *m = s[j + 4] & 63;
  } else {
    *sc = (s[j + 4] & 0x0f) | ((s[j - 4] >> 6) << 4);
    *m = (s[j + 4] >> 4) | ((s[j] >> 6) << 4);
  }
}

// v of the lane whose index differs in the low bits of MASK (1, 2 or 4)
template <int MASK>
__device__ __forceinline__ uint32_t lane_xor(uint32_t v) {
  static_assert(MASK == 1 || MASK == 2 || MASK == 4, "");
  if constexpr (MASK == 4) return (uint32_t)__shfl_xor((int)v, 4);
  return (uint32_t)dpp_i<MASK == 1 ? 0xb1 : 0x4e>((int)v);
}
__device__ __forceinline__ float fmax8(float v) {  // over the 8 lanes of a block, from 0
  v = fmaxf(fmaxf(v, 0.0f), dpp_f<0xb1>(v));
  v = fmaxf(v, dpp_f<0x4e>(v));
  return fmaxf(v, dpp_f<0x141>(v));
}

// The wave's 64 sub-blocks of N values: `first` is the first one's index, `total`
// their number. Coalesced 16-byte loads into LDS (chunk c of sub-block r in slot
// c ^ r % (N / 4)), then each lane's own values. Lanes past the end repeat the
// last sub-block.
template <int N>
__device__ __forceinline__ void load_sub_block(const float* __restrict__ w, long long first, long long total,
                                               float* lds, int lane, float (&x)[N]) {
  constexpr int C = N / 4;
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  f32x4* l4 = reinterpret_cast<f32x4*>(lds);
#pragma unroll
  for (int i = 0; i < C; ++i) {
    const int s = 64 * i + lane, r = s / C, c = s % C;
    const float* p = w + (first + r < total ? first + r : total - 1) * N + 4 * c;
    l4[r * C + (c ^ (r % C))] = (f32x4){p[0], p[1], p[2], p[3]};
  }
  // (a wave reads only what it wrote itself: LDS keeps a wave's order)
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const f32x4 v = l4[lane * C + (c ^ (lane % C))];
#pragma unroll
    for (int e = 0; e < 4; ++e) x[4 * c + e] = v[e];
  }
}

// Q4_K blocks: 8 lanes each.
__device__ __forceinline__ void quantize_q4k_lanes(const float* __restrict__ w, uint8_t* __restrict__ out,
                                                   long long nblocks, float* lds) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63, j = lane & 7;
  const long long first = ((long long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * 64;
  if (first >= 8 * nblocks) return;
  float x[32];
  load_sub_block<32>(w, first, 8 * nblocks, lds, lane, x);
  float sub_min;
  const float sub_scale = fit_q4(x, &sub_min);
  const float max_scale = fmax8(sub_scale), max_min = fmax8(sub_min);
  const float inv_scale = max_scale > 0.0f ? 63.0f / max_scale : 0.0f;
  const float inv_min = max_min > 0.0f ? 63.0f / max_min : 0.0f;
  int ls = round_i(inv_scale * sub_scale);
  int lm = round_i(inv_min * sub_min);
  ls = ls < 63 ? ls : 63;
  lm = lm < 63 ? lm : 63;
  // the scale bytes: lanes 0-3 hold bytes j and j + 4 (own low bits, lane j + 4's
  // top two), lanes 4-7 byte j + 4 (own low nibbles)
  const int pls = (int)lane_xor<4>((uint32_t)ls), plm = (int)lane_xor<4>((uint32_t)lm);
  const uint32_t a = (uint32_t)((ls & 0xff) | (((pls >> 4) << 6) & 0xff));
  const uint32_t b = (uint32_t)((lm & 0xff) | (((plm >> 4) << 6) & 0xff));
  const uint32_t c = (uint32_t)((ls & 0x0f) | ((lm & 0x0f) << 4));
  const uint32_t pa = lane_xor<4>(a), pb = lane_xor<4>(b);
  const int s = j < 4 ? (int)(a & 63) : (int)((c & 0x0f) | ((pa >> 6) << 4));
  const int m = j < 4 ? (int)(b & 63) : (int)((c >> 4) | ((pb >> 6) << 4));
  const uint16_t dh = f2h(max_scale / 63.0f), mh = f2h(max_min / 63.0f);
  const float d = h2f(dh) * (float)s, dm = h2f(mh) * (float)m;
  uint32_t q[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    q[i] = 0;
    if (d != 0.0f) {
#pragma unroll
      for (int e = 0; e < 4; ++e) q[i] |= (uint32_t)round_to((x[4 * i + e] + dm) / d, 15.0f) << (8 * e);
    }
  }
  // quad-wide OR: dword of bytes 0-3 / 4-7 in lanes 0-3, of bytes 8-11 in lanes 4-7
  auto gather = [&](uint32_t v) {
    v <<= 8 * (j & 3);
    v |= lane_xor<1>(v);
    return v | lane_xor<2>(v);
  };
  const uint32_t ga = gather(a), gb = gather(b), gc = lane_xor<4>(gather(c));
  // lanes 2i, 2i + 1 share 32 bytes of quants (low and high nibbles): each writes 16
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t give = (j & 1) ? q[i] : q[4 + i], keep = (j & 1) ? q[4 + i] : q[i];
    const uint32_t got = lane_xor<1>(give);
    o[i] = (j & 1) ? got | keep << 4 : keep | got << 4;
  }
  if (first + lane >= 8 * nblocks) return;
  uint4* blk = reinterpret_cast<uint4*>(out + kQ4KBytes * ((first + lane) >> 3));
  if (j == 0) blk[0] = make_uint4((uint32_t)dh | (uint32_t)mh << 16, ga, gb, gc);
  blk[1 + j] = make_uint4(o[0], o[1], o[2], o[3]);
}

// Symmetric fit of 16 values to [-32, 31] with the squared-value weighting
// (make_qx_quants with rmse_type 1); codes are integer-valued floats.
__device__ __forceinline__ float fit_q6(const float (&x)[16], float (&codes)[16]) {
#pragma clang fp contract(off)
  float amax = 0.0f, vmax = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float a = fabsf(x[i]);
    if (a > amax) {
      amax = a;
      vmax = x[i];
    }
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) codes[i] = -32.0f;  // stored as 0 where every value is 0
  if (amax == 0.0f) return 0.0f;
  const float iscale = -32.0f / vmax;
  float sumlx = 0.0f, suml2 = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float l = round_between(iscale * x[i], -32.0f, 31.0f);
    codes[i] = l;
    const float w = x[i] * x[i];
    sumlx += w * x[i] * l;
    suml2 += w * l * l;
  }
  float scale = sumlx / suml2;
  float best = scale * sumlx;
#pragma unroll 1
  for (int t = 0; t < 3; ++t) {
    const float is = 1.0f / scale;
    float slx = 0.0f, sl2 = 0.0f, n[16];
    bool changed = false;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      n[i] = round_between(is * x[i], -32.0f, 31.0f);
      changed |= n[i] != codes[i];
      const float w = x[i] * x[i];
      slx += w * x[i] * n[i];
      sl2 += w * n[i] * n[i];
    }
    if (!changed || sl2 == 0.0f || slx * slx <= best * sl2) break;
#pragma unroll
    for (int i = 0; i < 16; ++i) codes[i] = n[i];
    sumlx = slx;
    suml2 = sl2;
    scale = sumlx / suml2;
    best = scale * sumlx;
  }
#pragma unroll 1
  for (int t = 0; t < 5; ++t) {
    bool any = false;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float w = x[i] * x[i], l = codes[i];
      float slx = sumlx - w * x[i] * l;
      if (slx > 0.0f) {
        float sl2 = suml2 - w * l * l;
        const float nl = round_between(x[i] * sl2 / slx, -32.0f, 31.0f);
        if (nl != l) {
          slx += w * x[i] * nl;
          sl2 += w * nl * nl;
          if (sl2 > 0.0f && slx * slx * suml2 > sumlx * sumlx * sl2) {
            codes[i] = nl;
            sumlx = slx;
            suml2 = sl2;
            scale = sumlx / suml2;
            any = true;
          }
        }
      }
    }
    if (!any) break;
  }
  return scale;
}

// Q6_K blocks in the device layout (bodies, then the f16 scales): 16 lanes each.
__device__ __forceinline__ void quantize_q6k_lanes(const float* __restrict__ w, uint8_t* __restrict__ out,
                                                   long long nblocks, float* lds) {
#pragma clang fp contract(off)
  const int lane = threadIdx.x & 63, j = lane & 15;
  const long long first = ((long long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * 64;
  if (first >= 16 * nblocks) return;
  float x[16], codes[16];
  load_sub_block<16>(w, first, 16 * nblocks, lds, lane, x);
  const float scale = fit_q6(x, codes);
  // the first sub-block scale of the largest magnitude (0 if none is above 0)
  const float a = fabsf(scale) > 0.0f ? fabsf(scale) : 0.0f;
  float amax = fmaxf(a, dpp_f<0xb1>(a));
  amax = fmaxf(amax, dpp_f<0x4e>(amax));
  amax = fmaxf(amax, dpp_f<0x141>(amax));
  amax = fmaxf(amax, dpp_f<0x140>(amax));
  int at = a == amax && amax > 0.0f ? j : 16;
  at = min(at, dpp_i<0xb1>(at));
  at = min(at, dpp_i<0x4e>(at));
  at = min(at, dpp_i<0x141>(at));
  at = min(at, dpp_i<0x140>(at));
  const float first_max = __shfl(scale, (lane & 48) + (at & 15));
  const float max_scale = at < 16 ? first_max : 0.0f;
  const float iscale = -128.0f / max_scale;
  const uint16_t dh = f2h(1.0f / iscale);
  const int v = round_i(iscale * scale);
  const int8_t sc = (int8_t)(v < 127 ? v : 127);
  const float d = h2f(dh) * (float)sc;
  if (!(d == 0.0f)) {
#pragma unroll
    for (int i = 0; i < 16; ++i) codes[i] = round_between(x[i] / d, -32.0f, 31.0f);
  }
  // lane j = 8 h + 2 g + p: values 128 h + 32 g + 16 p ...; quants of g and g + 2
  // share bytes (low and high nibbles), the top two bits of the four g share one
  const int h = j >> 3, g = (j >> 1) & 3, p = j & 1;
  uint32_t lo[4], hi[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    lo[i] = hi[i] = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t c = (uint32_t)((int)codes[4 * i + e] + 32);
      lo[i] |= (c & 15) << (8 * e);
      hi[i] |= ((c >> 4) & 3) << (8 * e + 2 * g);
    }
    lo[i] |= lane_xor<4>(lo[i]) << 4;  // of use in lanes g < 2
    hi[i] |= lane_xor<2>(hi[i]);
    hi[i] |= lane_xor<4>(hi[i]);
  }
  const long long blk = (first + lane) >> 4;
  if (blk >= nblocks) return;
  uint8_t* body = out + kQ6KBody * blk;
  if (g < 2) *reinterpret_cast<uint4*>(body + 64 * h + 32 * g + 16 * p) = make_uint4(lo[0], lo[1], lo[2], lo[3]);
  if (g == 2) *reinterpret_cast<uint4*>(body + 128 + 32 * h + 16 * p) = make_uint4(hi[0], hi[1], hi[2], hi[3]);
  body[192 + j] = (uint8_t)sc;
  if (j == 0) reinterpret_cast<uint16_t*>(out + kQ6KBody * nblocks)[blk] = dh;
}

}  // namespace qmm

// ===========================================================================
// kernels
// ===========================================================================

// x: f32 [m, k] row stride ldx; y: m*k/256 Q8_K blocks. One wave per block.
extern "C" __global__ void __launch_bounds__(256) qmm_quantize_q8k(const float* __restrict__ x,
                                                                   long long ldx, uint8_t* __restrict__ y,
                                                                   int k, int m) {
  const int nb = k / 256;
  const long long w = (long long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (w >= (long long)m * nb) return;
  const int row = (int)(w / nb), b = (int)(w % nb);
  qmm::q8k_block(x + row * ldx + 256LL * b, y + w * qmm::kQ8KBytes, threadIdx.x & 63);
}

// x: f32 [m, k] row stride ldx; y: m*k/32 GGML Q8_0 blocks. 8 lanes per block.
extern "C" __global__ void __launch_bounds__(256) qmm_quantize_q8_0(const float* __restrict__ x,
                                                                    long long ldx, uint8_t* __restrict__ y,
                                                                    int k, int m) {
  const int nb = k / 32;
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long blk = t >> 3;
  const bool valid = blk < (long long)m * nb;
  const long long bc = valid ? blk : 0;
  const int row = (int)(bc / nb), b = (int)(bc % nb);
  qmm::q80_block(x + row * ldx + 32LL * b, y + bc * qmm::kQ80Bytes, (int)(t & 7), valid);
}

// Weight quantizers to the device layout, four waves of 64 sub-blocks. One
// qmm_qtensor_quantize call on 4096 x 4096 values (allocation and a
// synchronisation included): Q4_K 65 us, Q6_K 103 us; with one thread per
// super-block and its codes in byte arrays (scratch memory) 983 us and 402 us.
extern "C" __global__ void __launch_bounds__(256) qmm_quantize_q4k_w(const float* __restrict__ w,
                                                                     uint8_t* __restrict__ out, long long nblocks) {
  __shared__ __attribute__((aligned(16))) float lds[4][64 * 32];
  qmm::quantize_q4k_lanes(w, out, nblocks, lds[threadIdx.x >> 6]);
}

extern "C" __global__ void __launch_bounds__(256) qmm_quantize_q6k_w(const float* __restrict__ w,
                                                                     uint8_t* __restrict__ out, long long nblocks) {
  __shared__ __attribute__((aligned(16))) float lds[4][64 * 16];
  qmm::quantize_q6k_lanes(w, out, nblocks, lds[threadIdx.x >> 6]);
}

// Q8_0 weights straight to the device layout (quants, then the f16 scales): the
// call takes 40 us on 4096 x 4096 values, 82 us by way of GGML blocks in a
// buffer of their own.
extern "C" __global__ void __launch_bounds__(256) qmm_quantize_q8_0_w(const float* __restrict__ w,
                                                                      uint8_t* __restrict__ out, long long nblocks) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long blk = t >> 3;
  const bool valid = blk < nblocks;
  const float* x = w + (valid ? 4 * t : 0);
  const float e[4] = {x[0], x[1], x[2], x[3]};
  uint16_t d;
  const uint32_t q = qmm::q80_lane(e, &d);
  if (!valid) return;
  reinterpret_cast<uint32_t*>(out)[t] = q;
  if ((t & 7) == 0) reinterpret_cast<uint16_t*>(out + qmm::kQ80Body * nblocks)[blk] = d;
}

// GGML bytes <-> device layout for the formats whose blocks are not 16-byte
// multiples (Q6_K: body | d at the end; Q8_0: d | qs at the front).
// One thread per block, 16-bit copies (GGML blocks are 2-byte aligned).
extern "C" __global__ void qmm_ggml_to_dev(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst,
                                           long long nblocks, int fmt) {
  const long long b = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nblocks) return;
  if (fmt == qmm::kFmtQ6K) {
    const uint16_t* s = reinterpret_cast<const uint16_t*>(src + qmm::kQ6KBytes * b);
    uint16_t* body = reinterpret_cast<uint16_t*>(dst + qmm::kQ6KBody * b);
    for (int i = 0; i < qmm::kQ6KBody / 2; ++i) body[i] = s[i];
    reinterpret_cast<uint16_t*>(dst + qmm::kQ6KBody * nblocks)[b] = s[qmm::kQ6KBody / 2];
  } else {
    const uint16_t* s = reinterpret_cast<const uint16_t*>(src + qmm::kQ80Bytes * b);
    uint16_t* body = reinterpret_cast<uint16_t*>(dst + qmm::kQ80Body * b);
    for (int i = 0; i < qmm::kQ80Body / 2; ++i) body[i] = s[1 + i];
    reinterpret_cast<uint16_t*>(dst + qmm::kQ80Body * nblocks)[b] = s[0];
  }
}

extern "C" __global__ void qmm_dev_to_ggml(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst,
                                           long long nblocks, int fmt) {
  const long long b = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nblocks) return;
  if (fmt == qmm::kFmtQ6K) {
    const uint16_t* body = reinterpret_cast<const uint16_t*>(src + qmm::kQ6KBody * b);
    uint16_t* d = reinterpret_cast<uint16_t*>(dst + qmm::kQ6KBytes * b);
    for (int i = 0; i < qmm::kQ6KBody / 2; ++i) d[i] = body[i];
    d[qmm::kQ6KBody / 2] = reinterpret_cast<const uint16_t*>(src + qmm::kQ6KBody * nblocks)[b];
  } else {
    const uint16_t* body = reinterpret_cast<const uint16_t*>(src + qmm::kQ80Body * b);
    uint16_t* d = reinterpret_cast<uint16_t*>(dst + qmm::kQ80Bytes * b);
    d[0] = reinterpret_cast<const uint16_t*>(src + qmm::kQ80Body * nblocks)[b];
    for (int i = 0; i < qmm::kQ80Body / 2; ++i) d[1 + i] = body[i];
  }
}

// Dequantize a device-layout tensor (QTensor::dequantize); formulas of
// crates/llm/mlx-llm/src/gguf/dequant.rs:284-290 (Q8_0), :391-416 (Q4_K),
// :452-474 (Q6_K), one rounding per f32 operation; the f16 / bf16 outputs round
// the f32 value once more, to nearest even (the f32 dequantize followed by
// to_dtype; a NaN stays one).
//
// Bound by memory: a thread forms 16 bytes of consecutive outputs (4 f32 or 8
// 16-bit values, always inside one sub-block), so that a wave's loads and stores
// are whole lines, and in large tensors kDqUnits of them 256 threads apart, so
// that their loads are in flight together. 14336 x 4096 Q8_0 to f32 (295 MB) took
// 93 us with one thread per 32 consecutive values, 128 bytes from its neighbour's,
// and its conversion to bf16 63 us; to bf16 at once (180 MB) it takes 29 us.
namespace qmm {
constexpr int kDqUnits = 4;

__device__ __forceinline__ uint32_t bf16_bits(float v) {  // round to nearest even
  const uint32_t b = __builtin_bit_cast(uint32_t, v);
  return v == v ? (b + 0x7fffu + ((b >> 16) & 1u)) >> 16 : 0x7fc0u;
}
__device__ __forceinline__ void put_vals(float* y, const float (&v)[4]) {
  *reinterpret_cast<float4*>(y) = make_float4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ void put_vals(_Float16* y, const float (&v)[8]) {
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = v[2 * i], b = v[2 * i + 1];
    // the f32 product first: folded into its conversion as v_fma_mixlo_f16 x, y, 0
    // a -0 would come out as +0
    asm("" : "+v"(a), "+v"(b));
    w[i] = (uint32_t)f2h(a) | (uint32_t)f2h(b) << 16;
  }
  *reinterpret_cast<uint4*>(y) = make_uint4(w[0], w[1], w[2], w[3]);
}
__device__ __forceinline__ void put_vals(uint16_t* y, const float (&v)[8]) {  // bf16
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = bf16_bits(v[2 * i]) | bf16_bits(v[2 * i + 1]) << 16;
  *reinterpret_cast<uint4*>(y) = make_uint4(w[0], w[1], w[2], w[3]);
}

__device__ __forceinline__ void put_val(float* y, float v) { *y = v; }
__device__ __forceinline__ void put_val(_Float16* y, float v) {
  asm("" : "+v"(v));
  *y = (_Float16)v;
}
__device__ __forceinline__ void put_val(uint16_t* y, float v) { *y = (uint16_t)bf16_bits(v); }

// N consecutive bytes (4 or 8, aligned) as dwords
template <int N>
struct Bytes {
  uint32_t w[N / 4];
  __device__ __forceinline__ uint32_t operator[](int i) const { return (w[i / 4] >> (8 * (i % 4))) & 0xffu; }
};
template <int N>
__device__ __forceinline__ Bytes<N> load_bytes(const uint8_t* p) {
  Bytes<N> b;
  if constexpr (N == 4) {
    b.w[0] = *reinterpret_cast<const uint32_t*>(p);
  } else {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    b.w[0] = v.x;
    b.w[1] = v.y;
  }
  return b;
}

// What a unit (outputs N u .. N u + N - 1) needs from memory, and its values.
template <int FMT, int N>
struct DqUnit {
  Bytes<N> q, h;     // quants; Q6_K: their top bits
  uint4 head;        // Q4_K: d, dmin and the scale bytes
  uint16_t d;        // Q6_K, Q8_0
  int8_t sc;         // Q6_K
  __device__ __forceinline__ void load(const uint8_t* __restrict__ src, long long u, long long nblocks) {
    if constexpr (FMT == kFmtQ80) {
      q = load_bytes<N>(src + N * u);
      d = reinterpret_cast<const uint16_t*>(src + kQ80Body * nblocks)[u / (32 / N)];
    } else {
      const long long b = u / (256 / N);
      const int e = (int)(u % (256 / N)) * N, part = e / 32, l = e % 32;
      if constexpr (FMT == kFmtQ4K) {
        const uint8_t* blk = src + kQ4KBytes * b;
        head = *reinterpret_cast<const uint4*>(blk);
        q = load_bytes<N>(blk + 16 + 32 * (part >> 1) + l);
      } else {
        // outputs 128 h + 32 s + [0, 32): low / high nibbles of ql, 2 bits of qh
        const uint8_t* body = src + kQ6KBody * b;
        const int hf = part >> 2, s = part & 3;
        q = load_bytes<N>(body + 64 * hf + 32 * (s & 1) + l);
        h = load_bytes<N>(body + 128 + 32 * hf + l);
        sc = (int8_t)body[192 + 8 * hf + 2 * s + l / 16];
        d = reinterpret_cast<const uint16_t*>(src + kQ6KBody * nblocks)[b];
      }
    }
  }
  __device__ __forceinline__ void values(long long u, float (&v)[N]) const {
#pragma clang fp contract(off)
    if constexpr (FMT == kFmtQ80) {
      const float df = h2f(d);
#pragma unroll
      for (int i = 0; i < N; ++i) v[i] = (float)(int8_t)q[i] * df;
      return;
    }
    const int part = (int)(u % (256 / N)) * N / 32;
    if constexpr (FMT == kFmtQ4K) {
      const uint32_t hw[4] = {head.x, head.y, head.z, head.w};
      // q4k_scale_min on the header's dwords: bytes 0-3, 4-7 and 8-11 are hw[1..3]
      const int j = part & 3, o = 8 * j;
      const uint32_t a = (hw[1] >> o) & 0xff, b = (hw[2] >> o) & 0xff, c = (hw[3] >> o) & 0xff;
      const uint32_t sc4 = part < 4 ? a & 63 : (c & 0x0f) | (a >> 6) << 4;
      const uint32_t mn4 = part < 4 ? b & 63 : (c >> 4) | (b >> 6) << 4;
      const float d1 = h2f(hw[0]) * (float)(int)sc4, m1 = h2f(hw[0] >> 16) * (float)(int)mn4;
      const int sh = (part & 1) * 4;
#pragma unroll
      for (int i = 0; i < N; ++i) v[i] = d1 * (float)(int)((q[i] >> sh) & 0xf) - m1;
    } else {
      const int s = part & 3, nsh = (s >> 1) * 4, hsh = 2 * s;
      const float ds = h2f(d) * (float)sc;
#pragma unroll
      for (int i = 0; i < N; ++i)
        v[i] = ds * (float)((int)(((q[i] >> nsh) & 0xf) | (((h[i] >> hsh) & 3) << 4)) - 32);
    }
  }
};

// U units a thread, 256 threads apart.
template <int FMT, int U, class T>
__device__ __forceinline__ void dequantize_units(const uint8_t* __restrict__ src, T* __restrict__ y, long long nblocks) {
  constexpr int N = 16 / (int)sizeof(T);
  const long long units = nblocks * ((FMT == kFmtQ80 ? 32 : 256) / N);
  const long long u0 = (long long)blockIdx.x * (256 * U) + threadIdx.x;
  const bool aligned = (reinterpret_cast<uintptr_t>(y) & 15) == 0;
  DqUnit<FMT, N> unit[U];
#pragma unroll
  for (int i = 0; i < U; ++i) unit[i].load(src, min(u0 + 256 * i, units - 1), nblocks);
#pragma unroll
  for (int i = 0; i < U; ++i) {
    const long long u = u0 + 256 * i;
    if (u >= units) return;
    float v[N];
    unit[i].values(u, v);
    if (aligned) {
      put_vals(y + N * u, v);
    } else {  // a destination off the 16-byte grid: value by value
#pragma unroll
      for (int j = 0; j < N; ++j) put_val(y + N * u + j, v[j]);
    }
  }
}

template <int U, class T>
__device__ __forceinline__ void dequantize_blocks(const uint8_t* __restrict__ src, T* __restrict__ y,
                                                  long long nblocks, int fmt) {
  if (fmt == kFmtQ80) return dequantize_units<kFmtQ80, U>(src, y, nblocks);
  if (fmt == kFmtQ4K) return dequantize_units<kFmtQ4K, U>(src, y, nblocks);
  dequantize_units<kFmtQ6K, U>(src, y, nblocks);
}
}  // namespace qmm

#define QMM_DEQUANTIZE(SUFFIX, T, U)                                                                              \
  extern "C" __global__ void __launch_bounds__(256) qmm_dequantize##SUFFIX(                                       \
      const uint8_t* __restrict__ src, T* __restrict__ y, long long nblocks, int fmt) {                           \
    qmm::dequantize_blocks<U>(src, y, nblocks, fmt);                                                              \
  }
QMM_DEQUANTIZE(, float, qmm::kDqUnits)
QMM_DEQUANTIZE(_f16, _Float16, qmm::kDqUnits)
QMM_DEQUANTIZE(_bf16, uint16_t, qmm::kDqUnits)
QMM_DEQUANTIZE(_u1, float, 1)
QMM_DEQUANTIZE(_f16_u1, _Float16, 1)
QMM_DEQUANTIZE(_bf16_u1, uint16_t, 1)
