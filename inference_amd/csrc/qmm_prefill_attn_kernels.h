// Causal attention of a prompt's rows on the f32 matrix cores.
//
// Per kv head, the G = heads / kv_heads query heads of P = 32 / G consecutive
// prompt rows form one 32-column tile (column = row * G + head). A workgroup
// is four waves over one tile; wave w takes key tiles w, w + 4, ... of 32
// positions and keeps its own online-softmax state, and the four states are
// merged through LDS at the end. No wave waits for another before that.
//
// One key tile of a wave (head_dim 128: 128 MFMAs of 64 cycles):
//   S^T = K Q^T      v_mfma_f32_32x32x2_f32, A = the 32 keys, B = the 32
//                    columns. D column = lane & 31, so a column's 32 scores
//                    sit in 16 registers of two lanes: the row maximum is 15
//                    in-lane maxima and one exchange of wave halves.
//   O^T += V^T P^T   A = V^T, B = P^T. P^T stays where S^T left it: register r
//                    of lane half h is key 8(r/4) + 4h + r%4, and the MFMA's two
//                    k slots are the two lane halves, so step r takes V rows of
//                    exactly those two keys. No shuffle and no LDS for P.
// The k index of both products may be permuted freely: lane half h takes
// elements [h dim/2, (h+1) dim/2) of q and k, and A row m of V^T tile j is
// element DT m + j (DT = dim / 32), which makes every load, LDS read and store
// of a lane DT contiguous floats.
//
// K goes straight to LDS (buffer_load ... lds, 16 bytes a lane) with its 16-byte
// chunks XORed by the key, so that the 32 keys' reads of one chunk hit distinct
// banks; the queries sit in LDS in the same layout, shared by the four waves;
// V goes to registers (a half-wave reads one key's row). V of this tile is in
// flight during the S product, K of the next during the softmax and P V.
//
// What bounds it: the f32 matrix cores (256 FLOP per cycle and CU; a large f32
// library product reaches 151 TFLOP/s). All arithmetic stays f32, and the sums
// are kept in short chains (eight per score, 16 keys per addition to the
// running output), so the error against 64 bits stays that of the row kernel
// (1999 rows: 1.6e-7 against 1.7e-7 of the output's norm; with one chain of
// each it was 2.7e-7, at 296 us). 1999 rows from position 0, 32 / 8 heads of
// 128: 304 us = 108 TFLOP/s of the causal half (309 with the mask in every tile),
// against 1642 us with one workgroup per row (each of which read every K and V
// row for G heads and ran on the VALU); 700 rows 59 us against 245. The rest of the time is the
// softmax's VALU work where a SIMD's two waves meet in it, and the ramp of each
// workgroup (~3 us of merge and first loads for ~16 tiles of ~5 us a wave).
#pragma once

#include "qmm_common.h"
#include "qmm_quant_kernels.h"

namespace qmm {

typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kPaWaves = 4;   // waves of a workgroup (key splits)
constexpr int kPaKeys = 32;   // positions of a key tile
constexpr int kPaCols = 32;   // query columns of a workgroup

template <int N>
struct __attribute__((aligned(N >= 4 ? 16 : 4 * N))) FloatN {
  float v[N];
};

// max over the two lanes (halves) of a column
__device__ __forceinline__ float half_max(float v) { return fmaxf(v, __shfl_xor(v, 32)); }

template <int DT, bool PLANES>
__device__ __forceinline__ void prefill_attention_tile(const float* __restrict__ q, long long ldq,
                                                       const float* __restrict__ kcache,
                                                       const float* __restrict__ vcache, int first, int count,
                                                       float* __restrict__ out, long long ldo,
                                                       int8_t* __restrict__ pq8, float* __restrict__ pd,
                                                       int16_t* __restrict__ ps, int kq, int heads, int kv_heads,
                                                       int max_seq, float scale) {
  constexpr int dim = 32 * DT;
  constexpr int CH = dim / 4;  // 16-byte chunks of a key row
  constexpr int HC = CH / 2;   // those of one lane half
  __shared__ __attribute__((aligned(16))) float buf[kPaWaves][kPaKeys * dim];  // a wave's K tile, then its O^T
  __shared__ __attribute__((aligned(16))) float qb[kPaCols * dim];             // the columns' queries
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int half = lane >> 5, col = lane & 31;
  const int g = blockIdx.x, G = heads / kv_heads, P = kPaCols / G;
  // the tiles with the most keys first, so that the short ones fill the end
  const int i0 = (int)(gridDim.y - 1 - blockIdx.y) * P;
  const int nrow = min(P, count - i0);  // prompt rows of this tile (>= 1)
  const int pi = min(col / G, nrow - 1);  // columns past the rows repeat the last row; they are not stored
  const int p = first + i0 + pi;       // the column's last visible position
  const int pmin = first + i0;         // the tile's first row's
  const int n = first + i0 + nrow;     // positions any column sees
  const int ntiles = (n + kPaKeys - 1) / kPaKeys;
  const float* kc = kcache + (size_t)g * max_seq * dim;
  const float* vc = vcache + (size_t)g * max_seq * dim;

  // q in K's layout: chunk c of column r in slot c ^ (r % CH)
#pragma unroll
  for (int i = 0; i < kPaCols * CH / (64 * kPaWaves); ++i) {
    const int s = 64 * kPaWaves * i + t, r = s / CH, c = s % CH;
    const int ri = min(r / G, nrow - 1);
    const float* qp = q + (long long)(i0 + ri) * ldq + (long long)(g * G + r % G) * dim + 4 * c;
    FloatN<4> v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v.v[e] = qp[e];
    *reinterpret_cast<FloatN<4>*>(qb + r * dim + 4 * (c ^ (r & (CH - 1)))) = v;
  }
  float* kb = buf[wave];
  // Key tile kt of K or V as a buffer that ends at the last visible position:
  // the hardware's bounds check returns 0 for the rows past it, so nothing
  // unwritten is read (their scores are masked) and no lane clamps an address.
  auto tile = [&](const float* c, int kt) {
    kt = __builtin_amdgcn_readfirstlane(kt);  // (it is uniform: the descriptor lives in SGPRs)
    const int rows = __builtin_amdgcn_readfirstlane(min(max(n - kPaKeys * kt, 0), kPaKeys));
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(c + (size_t)kPaKeys * min(kt, ntiles) * dim), 0,
                                             rows * dim * 4, 0x00020000);
  };
  // Rows of a K tile to LDS, 64 chunks at a time: 64 / CH rows per load, chunk c
  // of row r in slot c ^ (r % CH). Lane offsets are one XOR away from each other;
  // the asm keeps them from being hoisted into a register each.
  constexpr int RPL = 64 / CH;  // rows per load
  unsigned klane = (unsigned)(lane / CH * dim * 4) + 16u * ((unsigned)(lane % CH) ^ (unsigned)(lane / CH));
  auto load_k = [&](int kt) {
    asm volatile("" : "+v"(klane));
    const auto r = tile(kc, kt);
#pragma unroll
    for (int i = 0; i < kPaKeys / RPL; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          r, (__attribute__((address_space(3))) void*)(kb + 256 * i), 16,
          (klane ^ (16u * ((RPL * i) & (CH - 1)))) + 1024 * i, 0, 0, 0);
  };
  // V rows of steps 8 b .. 8 b + 7
  unsigned vlane = 4u * (unsigned)(4 * half * dim + DT * col);
  auto load_v = [&](FloatN<DT>(&v)[8], int kt, int b) {
    asm volatile("" : "+v"(vlane));
    const auto rs = tile(vc, kt);
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const unsigned o = vlane + 4u * (unsigned)((16 * b + 8 * (r >> 2) + (r & 3)) * dim);
      if constexpr (DT == 4)
        v[r] = __builtin_bit_cast(FloatN<DT>, __builtin_amdgcn_raw_buffer_load_b128(rs, o, 0, 0));
      else
        v[r] = __builtin_bit_cast(FloatN<DT>, __builtin_amdgcn_raw_buffer_load_b64(rs, o, 0, 0));
    }
  };

  f32x16 acc[DT];
#pragma unroll
  for (int j = 0; j < DT; ++j) acc[j] = (f32x16)(0.0f);
  bool bad = false;
  float m = -INFINITY, ml = 0.0f, l = 0.0f;  // maximum, maximum * log2 e (0 while it is -inf), this half's sum

  // byte offset of this lane's first K chunk; chunk c is 16 c XORed in
  unsigned kread = (unsigned)(col * dim * 4) + 16u * ((unsigned)(half * HC) ^ (unsigned)(col & (CH - 1)));
  load_k(wave);
  __syncthreads();
#pragma unroll 1
  for (int kt = wave; kt < ntiles; kt += kPaWaves) {
    const bool diag = kPaKeys * kt + kPaKeys - 1 > pmin;
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the K tile is in LDS
    FloatN<DT> va[8], vb[8];  // V rows of the first and the last eight steps
    load_v(va, kt, 0);
    __builtin_amdgcn_sched_barrier(0);  // they are in flight during the S product, not after it
    asm volatile("" : "+v"(kread));
    auto chunk = [&](const float* base, int c) {
      return *reinterpret_cast<const FloatN<4>*>(reinterpret_cast<const char*>(base) + (kread ^ (16u * c)));
    };
    FloatN<4> ka = chunk(kb, 0), qa = chunk(qb, 0);
    // eight chains of roundings, each an eighth of the sum
    f32x16 s0;
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      f32x16 c4[4] = {(f32x16)(0.0f), (f32x16)(0.0f), (f32x16)(0.0f), (f32x16)(0.0f)};
#pragma unroll
      for (int c = x * HC / 2; c < (x + 1) * HC / 2; ++c) {  // the next chunks' reads fly under this one's products
        const FloatN<4> kn = chunk(kb, c + 1 < HC ? c + 1 : c), qn = chunk(qb, c + 1 < HC ? c + 1 : c);
#pragma unroll
        for (int e = 0; e < 4; ++e) c4[e] = __builtin_amdgcn_mfma_f32_32x32x2f32(ka.v[e], qa.v[e], c4[e], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        ka = kn;
        qa = qn;
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float v = (c4[0][r] + c4[1][r]) + (c4[2][r] + c4[3][r]);
        s0[r] = x == 0 ? v : s0[r] + v;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // every lane's reads of the K tile are consumed: the next may overwrite it.
    // Unconditional (past the end the keys are clamped and nothing reads them):
    // under a condition the waits below would have to assume it was not issued.
    load_v(vb, kt, 1);
    load_k(kt + kPaWaves);
    __builtin_amdgcn_sched_barrier(0);

    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) s0[r] *= scale;
    if (diag) {
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (kPaKeys * kt + 8 * (r >> 2) + 4 * half + (r & 3) > p) s0[r] = -INFINITY;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s0[r]);
    mx = fmaxf(m, half_max(mx));
    const float nml = mx == -INFINITY ? 0.0f : mx * kLog2e;
    float a;
    if (__builtin_expect(__any(!(fabsf(nml) < kBigRef)), 0)) {  // (see kBigRef)
      const AttnRef ref = attn_ref(mx);
      a = state_weight(m, ref);
#pragma unroll
      for (int r = 0; r < 16; ++r) s0[r] = score_weight(s0[r], ref);
    } else {
      // e^(s - m) as 2^(s log2 e - m log2 e) with one rounding; the rounding of
      // m log2 e is the same for every term of a column and cancels in o / l
      a = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ml - nml);
#pragma unroll
      for (int r = 0; r < 16; ++r) s0[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s0[r], kLog2e, -nml));
    }
    l *= a;
    m = mx;
    ml = nml;
#pragma unroll
    for (int r = 0; r < 16; ++r) l += s0[r];
    if (diag) {
      // 0 * v is not 0 for an infinity or a NaN in a masked position's value
      // row: such a tile is computed again below, position by position
      float z = 0.0f;
#pragma unroll
      for (int r = 0; r < 8; ++r)
#pragma unroll
        for (int j = 0; j < DT; ++j) z = __builtin_fmaf(vb[r].v[j], 0.0f, __builtin_fmaf(va[r].v[j], 0.0f, z));
      bad |= !__all(z == 0.0f);
    }
    // 16 keys' products are summed on their own and added to the running sum
    // once: its chain of roundings is then n / 64 long, as short as the sums of
    // the row kernel it replaces
    f32x16 o[2];
#pragma unroll
    for (int j = 0; j <= 2 * DT; ++j) {
      if (j < 2 * DT) {
        o[j & 1] = (f32x16)(0.0f);
#pragma unroll
        for (int r = 0; r < 8; ++r)
          o[j & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(j < DT ? va[r].v[j % DT] : vb[r].v[j % DT],
                                                          s0[(j < DT ? 0 : 8) + r], o[j & 1], 0, 0, 0);
      }
      if (j > 0) {  // added while the next 16 keys' products run
        const int i = (j - 1) % DT;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] = __builtin_fmaf(acc[i][r], j <= DT ? a : 1.0f, o[(j - 1) & 1][r]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  __syncthreads();  // the queries are read no more: their place takes the waves' maxima, sums and marks
  float(*st)[2][kPaCols] = reinterpret_cast<float(*)[2][kPaCols]>(qb);
  int* sbad = reinterpret_cast<int*>(qb + kPaWaves * 2 * kPaCols);

  // O^T of the wave to LDS: slot (column c, m ^ c) of DT floats holds elements
  // DT m ... of column c (the XOR spreads the 32 columns over the banks)
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): no K load may land on it
  l += __shfl_xor(l, 32);
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    FloatN<DT> o;
#pragma unroll
    for (int j = 0; j < DT; ++j) o.v[j] = acc[j][r];
    *reinterpret_cast<FloatN<DT>*>(kb + col * dim + DT * ((8 * (r >> 2) + 4 * half + (r & 3)) ^ col)) = o;
  }
  if (half == 0) {
    // -inf marks a wave without weights (a wave whose scores are all NaN has the
    // maximum -inf too, and a sum that must not be left out)
    st[wave][0][col] = l != 0.0f && m == -INFINITY ? 0.0f : m;
    st[wave][1][col] = l;
  }
  if (lane == 0) sbad[wave] = bad;
  __syncthreads();
  if (sbad[0] | sbad[1] | sbad[2] | sbad[3]) {
    // one column per wave, position by position, only what the column sees
    constexpr int R = dim / 64;
#pragma unroll 1
    for (int c = wave; c < G * nrow; c += kPaWaves) {
      const float* qp = q + (long long)(i0 + c / G) * ldq + (long long)(g * G + c % G) * dim;
      float cm = -INFINITY, cl = 0.0f, o[R];
#pragma unroll
      for (int e = 0; e < R; ++e) o[e] = 0.0f;
#pragma unroll 1
      for (int key = 0; key <= first + i0 + c / G; ++key) {
        float d = 0.0f;
#pragma unroll
        for (int e = 0; e < R; ++e) d += qp[R * lane + e] * kc[(unsigned)(key * dim + R * lane + e)];
        d = wave_sum(d) * scale;
        const float mx = fmaxf(cm, d);
        const float a = mx == -INFINITY ? 0.0f : expf(cm - mx), w = d == -INFINITY ? 0.0f : expf(d - mx);
        cm = mx;
        cl = cl * a + w;
#pragma unroll
        for (int e = 0; e < R; ++e) o[e] = o[e] * a + w * vc[(unsigned)(key * dim + R * lane + e)];
      }
#pragma unroll
      for (int e = 0; e < R; ++e) {
        const int d = R * lane + e;
        if constexpr (PLANES) {
          buf[0][c * dim + DT * ((d / DT) ^ c) + d % DT] = o[e] / cl;
        } else {
          out[(long long)(i0 + c / G) * ldo + (long long)(g * G + c % G) * dim + d] = o[e] / cl;
        }
      }
    }
  } else
#pragma unroll
  for (int i = 0; i < 32 * kPaCols / (64 * kPaWaves); ++i) {
    const int s = 64 * kPaWaves * i + t, c = s >> 5, e = s & 31;
    float M = -INFINITY, lsum = 0.0f;
#pragma unroll
    for (int w = 0; w < kPaWaves; ++w) M = fmaxf(M, st[w][0][c]);
    const AttnRef ref = attn_ref(M);
    FloatN<DT> o;
#pragma unroll
    for (int j = 0; j < DT; ++j) o.v[j] = 0.0f;
#pragma unroll
    for (int w = 0; w < kPaWaves; ++w) {
      if (st[w][0][c] != -INFINITY) {
        const float a = state_weight(st[w][0][c], ref);
        const FloatN<DT> x = *reinterpret_cast<const FloatN<DT>*>(buf[w] + c * dim + DT * (e ^ c));
        lsum += st[w][1][c] * a;
#pragma unroll
        for (int j = 0; j < DT; ++j) o.v[j] += x.v[j] * a;
      }
    }
#pragma unroll
    for (int j = 0; j < DT; ++j) o.v[j] /= lsum;
    const int ci = c / G;
    if constexpr (PLANES) {
      *reinterpret_cast<FloatN<DT>*>(buf[0] + c * dim + DT * (e ^ c)) = o;  // only this thread reads the slot
    } else if (ci < nrow) {
      float* op = out + (long long)(i0 + ci) * ldo + (long long)(g * G + c % G) * dim + DT * e;
#pragma unroll
      for (int j = 0; j < DT; ++j) op[j] = o.v[j];
    }
  }
  if constexpr (PLANES) {
    __syncthreads();
    // one wave per 256-element block of a row's G * dim outputs
    const int nb = kq / 256, nblk = G * dim / 256, b0 = g * G * dim / 256;
    for (int w = wave; w < nrow * nblk; w += kPaWaves) {
      const int ri = w / nblk, b = w % nblk;
      float e[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int x = 256 * b + 4 * lane + j, c = ri * G + x / dim, d = x % dim;
        e[j] = buf[0][c * dim + DT * ((d / DT) ^ c) + d % DT];
      }
      put_q8k_plane(q8k_lane_vals(e[0], e[1], e[2], e[3], lane), (long long)(i0 + ri) * nb + b0 + b, nb, kq, pq8, pd,
                    ps, lane);
    }
  }
}
}  // namespace qmm

// Grid kv_heads x ceil(count / (32 / G)), 256 threads. head_dim = 32 DT. A
// kv head's workgroups share an XCD (and its L2) where kv_heads is a multiple
// of 8: a dispatch deals workgroups to the XCDs by linear index.
#define QMM_PREFILL_ATTN_TILE(DT, WPS)                                                                            \
  extern "C" __global__ void __launch_bounds__(256, WPS) qmm_prefill_attn_tile_d##DT(                             \
      const float* __restrict__ q, long long ldq, const float* __restrict__ kcache,                               \
      const float* __restrict__ vcache, int first, int count, float* __restrict__ out, long long ldo, int heads,  \
      int kv_heads, int max_seq, float scale) {                                                                   \
    qmm::prefill_attention_tile<DT, false>(q, ldq, kcache, vcache, first, count, out, ldo, nullptr, nullptr,      \
                                           nullptr, 0, heads, kv_heads, max_seq, scale);                          \
  }                                                                                                               \
  extern "C" __global__ void __launch_bounds__(256, WPS) qmm_prefill_attn_tile_planes_d##DT(                      \
      const float* __restrict__ q, long long ldq, const float* __restrict__ kcache,                               \
      const float* __restrict__ vcache, int first, int count, int8_t* __restrict__ q8, float* __restrict__ d,     \
      int16_t* __restrict__ s, int kq, int heads, int kv_heads, int max_seq, float scale) {                       \
    qmm::prefill_attention_tile<DT, true>(q, ldq, kcache, vcache, first, count, nullptr, 0, q8, d, s, kq, heads,  \
                                          kv_heads, max_seq, scale);                                              \
  }
QMM_PREFILL_ATTN_TILE(2, 2)
QMM_PREFILL_ATTN_TILE(4, 2)
