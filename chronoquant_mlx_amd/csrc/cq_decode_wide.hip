// cq_decode_wide.hip — gfx950 MFMA split-K decode over the ChronoQuant cache for
// the shapes the head_dim-128 kernels do not take: any head_dim that is a
// multiple of 8, dense 2- and 3-bit rows, fp16 or bf16 queries, strides >= 4,
// any GQA ratio in chunks of 16 q heads.
//
// Reference semantics: the fused Metal kernel (kernels.py:79-228), in the
// factoring of the 16-head kernel (cq_decode_mfma.hip):
//   score_t = q'.a_g(t) + s_t * (q'.c_t)
//   out     = sum_g P_g a_g + sum_t (p_t s_t) c_t,   P_g = sum_{t in g} p_t
// These shapes ran on the portable kernel, whose weights and products are fp32,
// and keep that here:
// * scores: v_mfma_f32_16x16x32_f16 of operands that are exact in fp16 (q'; anchors;
//   codes -8 .. 7), summed in fp32.  bf16 q' rows are scaled by a power of two first,
//   and what a row holds below fp16's last place there, if anything, goes through
//   products of its own (kLow; the loops they make of the score products cost 1 to 3
//   us of these times);
// * P, p*s and the sums P_g stay fp32 numbers of any magnitude: the weighted sums
//   are fp32 matrix products of them with the codes and anchors as fp32.  (fp16
//   pairs hi + lo, whose products run 16 times as fast, hold 23 bits down to a
//   fixed step: behind a dominant token whose V is 0 the other tokens' weights were
//   off by 5e-4 at a gap of 10 nats.)
//
// Layout (NS K-steps of 32 dims, 32 NS >= D; W = D / 8 words of a row): lane (c,
// kg) of a score operand holds words NS kg .. NS kg + NS - 1 of token c (one or
// two wide loads), K-step j taking word NS kg + j; lane c of a V operand words
// NU c .. NU c + NU - 1 (NU = 2 beyond 128 dims) of 16 tokens.  Work: the balanced
// partition of cq_plan.h, 512-token units over one resident generation.
//
// Bound: the chain of a chunk (loads, two products, softmax) with two waves per SIMD
// in flight: on the first shape below the VALU is busy for 33 % of the time, the
// matrix cores for 12 (their fp32 products: 2600 clocks of a 256-dim chunk by 4x4x1,
// 10000 by 16x16x4), LDS for 6, and the waves wait for 39.  4 sequences of 16001
// tokens, 16/4 heads x 256 dims (82 MB): 45 us, 1.8 TB/s, against 370 on the
// portable kernel (fp32 VALU products, 8 head slots for 4 heads), 35 with the pairs
// and 57 with 16x16x4 products for 4 heads; 8 heads per kv head, 16/2: 41 and 28.5
// with the pairs; 16 ragged sequences of up to 4096, 32/8 x 64: 41 against 177; one
// of 1000, 16/4 x 256: 27 against 304.
// Error of the fp32 output against binary64, mean of 8 seeds of 4000 tokens by head
// dim: 8.0 to 9.3e-8 relative, the portable kernel 7.4 to 9.1e-8.
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>

#include "cq_mfma_common.h"

namespace cq {

namespace {

constexpr float kLow = 274877906944.f;  // 2^38: scale of the low parts of bf16 q'

template <int NS>
struct WideDims {
  static constexpr int kDP = 32 * NS;
  static constexpr int kNU = NS > 4 ? 2 : 1;  // V words per lane
  static constexpr int kTiles = 8 * kNU;      // 16-column V tiles
};

struct alignas(16) WideWave {
  int slot_k[kChunk], slot_v[kChunk];  // P-frame slot (-1: I-frame / padding)
  int gkl[kChunk], gvl[kChunk];        // anchor index relative to the chunk's first
  uint32_t s16[kChunk];                // fp16 K scale | fp16 V scale << 16 (0: none)
  float qa[16][kHeads];                // q'.anchor_k by (local anchor, head)
};

template <int NS>
struct alignas(16) WideMerge {
  static constexpr int kO = 16 * 8 * WideDims<NS>::kNU;  // dims the V tiles cover
  float t[kWaves][kMergeHeads][kO];
  float m[kWaves][kHeads], l[kWaves][kHeads];
  float wm[kHeads], wl[kHeads];
  float o[kHeads][kO];
};

template <int NS>
struct WideLds {
  // q' of K-step j, lane (head, kg): natural order, field order; [1]: the low parts
  h8_t qn[2][NS][64], qc[2][NS][64];
  float cs[kHeads];
  int low[kWaves];  // whether the wave's heads have low parts
  union {
    WideWave w[kWaves];
    WideMerge<NS> mg;
  };
};

// n consecutive dwords at a dword-aligned offset
template <int N>
__device__ __forceinline__ void bload_words(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t (&w)[N]) {
  int i = 0;
#pragma unroll
  for (; i + 4 <= N; i += 4) {
    const uint4 v = bload128(r, off + 4u * i);
    w[i] = v.x, w[i + 1] = v.y, w[i + 2] = v.z, w[i + 3] = v.w;
  }
#pragma unroll
  for (; i + 2 <= N; i += 2) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, (int)(off + 4u * i), 0, kPolicyStream);
    w[i] = (uint32_t)v[0], w[i + 1] = (uint32_t)v[1];
  }
  if (i < N) w[i] = bload32(r, off + 4u * i);
}

// Dense rows: the fields of dims 8 word .. 8 word + 7 (8 fb stream bits at bit 8 fb word),
// as the nibbles code + 8 of an INT4 word.
__device__ __forceinline__ uint32_t bload_dense(__amdgpu_buffer_rsrc_t r, uint32_t row, int word, int fb) {
  const uint32_t bit = 8u * fb * word;
  const uint32_t a = bload32(r, row + 4u * (bit >> 5)), b = bload32(r, row + 4u * (bit >> 5) + 4u);
  const uint32_t f = __builtin_amdgcn_alignbit(b, a, bit & 31u);
  const uint32_t m = (1u << fb) - 1u;
  uint32_t w = 0;
#pragma unroll
  for (int k = 0; k < 8; ++k) w |= ((f >> (fb * k)) & m) << (4 * k);
  return w + (8u - (1u << (fb - 1))) * 0x11111111u;  // (at most 15 each: no carry)
}

// K word (8 nibbles code + 8) -> A operand: the codes in unpack_k's order of dims.
__device__ __forceinline__ h8_t codes_k(uint32_t w) {
  const uint32_t m = 0x000F000Fu, magic = 0x64006400u;  // fp16 1024 in both halves
  const h2_t bias = {(_Float16)-1032.f, (_Float16)-1032.f};
  const h2_t a = as_h2(and_or(w, m, magic)) + bias, b = as_h2(and_or(w >> 4, m, magic)) + bias;
  const h2_t c = as_h2(and_or(w >> 8, m, magic)) + bias, d = as_h2(and_or(w >> 12, m, magic)) + bias;
  return h8_t{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
}
// Code e of a word of two's complement nibbles (an INT4 word ^ 0x88888888).
__device__ __forceinline__ float code_f32(uint32_t w, int e) {
  return (float)((int)(w << (28 - 4 * e)) >> 28);
}
// v_mfma_f32_16x16x4_f32: lane (c, kg) holds A[row c][kg], B[kg][col c], and C as
// mfma32's.
__device__ __forceinline__ f4_t mfma_f32(float a, float b, f4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// A weighted sum's step, weights a and values b by lane (c, kg).  16 heads: the
// product above (row = head c, summed over the 4 kg).  Up to 4 heads (Few): the 16
// blocks of v_mfma_f32_4x4x1_f32, block = 4 adjacent lanes, whose lane c holds head c %
// 4's weight and its own column's value and receives its column's sum for heads 0 .. 3
// over the tokens of its kg alone: 8 clocks in place of 32 for a product whose rows
// 4 .. 15 nobody needs.
template <bool Few>
__device__ __forceinline__ f4_t weigh(float a, float b, f4_t c) {
  if constexpr (Few) return __builtin_amdgcn_mfma_f32_4x4x1f32(a, b, c, 0, 0, 0);
  else return mfma_f32(a, b, c);
}

// Few: at most 4 q heads per kv head.  Score column c then belongs to head c % 4, so
// that every lane holds the weights weigh<true> wants from it.
template <int NS, bool Dense, bool Few>
__global__ __launch_bounds__(kThreadsMfma) __attribute__((amdgpu_waves_per_eu(2, 2)))
void decode_wide_kernel(DecodeArgs a) {
  using Dm = WideDims<NS>;
  constexpr int NU = Dm::kNU, NT = Dm::kTiles;
  __shared__ WideLds<NS> lds;
  __shared__ int32_t s_units[kMaxTableSeqs + 1];
  __shared__ int32_t s_loop[8];  // cursor unit [2], cursor sequence [2], end unit, P, n
  prefetch_args();
  const int h = blockIdx.y / a.n_chunks;
  const int chunk = blockIdx.y - h * a.n_chunks;
  const bool table = a.seq_lens && a.B > 1 && a.B <= kMaxTableSeqs;
  {
    if (table) build_unit_table(a, s_units);
    UnitSpace us;
    us.start = table ? s_units : nullptr;
    us.n = units_of(a.max_T);
    us.B = a.B;
    const int64_t U = us.total();
    const int64_t P = min((int64_t)gridDim.x, U);  // every workgroup below P has units
    if ((int64_t)blockIdx.x >= P) return;
    if (threadIdx.x == 0) {
      const int64_t u0 = unit_begin(blockIdx.x, U, P);
      s_loop[0] = (int32_t)u0;
      s_loop[2] = us.seq_of(u0);
      s_loop[4] = (int32_t)unit_begin(blockIdx.x + 1, U, P);
      s_loop[5] = (int32_t)P;
      s_loop[6] = (int32_t)us.n;
    }
    __syncthreads();
  }
  const int D = a.D, W = a.W;
  const int j0 = chunk * kHeads;
  const int gn = min(kHeads, a.G - j0);
  const int sk = a.stride[0], sv = a.stride[1];
  const float isk = a.inv_stride[0], isv = a.inv_stride[1];
  const int fbk = Dense ? a.fbits[0] : 4, fbv = Dense ? a.fbits[1] : 4;
  const uint32_t krow = 4u * row_words_of(D, fbk), vrow = 4u * row_words_of(D, fbv);
  uint32_t magic;  // fp16 1024 in both halves

  for (int it = 0;; ++it) {
    const int tid = thread_id();
    __builtin_assume(tid >= 0 && tid < kThreadsMfma);
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, kg = lane >> 4;
    const volatile int32_t *sl = s_loop;
    const int32_t u = __builtin_amdgcn_readfirstlane(sl[it & 1]);
    if (u >= __builtin_amdgcn_readfirstlane(sl[4])) break;
    const int b = __builtin_amdgcn_readfirstlane(sl[2 + (it & 1)]);
    Segment sg;
    {
      UnitSpace us;
      us.start = table ? s_units : nullptr;
      us.n = __builtin_amdgcn_readfirstlane(sl[6]);
      us.B = a.B;
      const int64_t u_next = segment_at(us, blockIdx.x, __builtin_amdgcn_readfirstlane(sl[5]), u, b,
                                        seq_len_of(a, b), sg);
      if (tid == 0) {
        s_loop[(it + 1) & 1] = (int32_t)u_next;
        s_loop[2 + ((it + 1) & 1)] = b + 1;
      }
    }
    if (sg.live == 0) {  // past the sequence's end
      __syncthreads();
      continue;
    }
    const int64_t t0 = sg.t0, t1 = sg.t1;
    const int64_t bh = (int64_t)b * a.H + h;
    const __amdgpu_buffer_rsrc_t r_kfk =
        make_rsrc(a.kf[0] + bh * a.cap_kf[0] * D, (uint32_t)(a.cap_kf[0] * D * 2));
    const __amdgpu_buffer_rsrc_t r_kfv =
        make_rsrc(a.kf[1] + bh * a.cap_kf[1] * D, (uint32_t)(a.cap_kf[1] * D * 2));
    const __amdgpu_buffer_rsrc_t r_pkk =
        make_rsrc((const char *)a.pk[0] + bh * a.cap_pf[0] * krow, (uint32_t)(a.cap_pf[0] * krow));
    const __amdgpu_buffer_rsrc_t r_pkv =
        make_rsrc((const char *)a.pk[1] + bh * a.cap_pf[1] * vrow, (uint32_t)(a.cap_pf[1] * vrow));
    const __amdgpu_buffer_rsrc_t r_sck = make_rsrc(a.sc[0] + bh * a.cap_pf[0], (uint32_t)(a.cap_pf[0] * 2));
    const __amdgpu_buffer_rsrc_t r_scv = make_rsrc(a.sc[1] + bh * a.cap_pf[1], (uint32_t)(a.cap_pf[1] * 2));

    // ---- q' tables: half-wave tid / 32 = head, its lane = word ----------------------
    {
      const int hh = tid >> 5, w = tid & 31;
      const int hq = Few ? hh & 3 : hh;  // head of column hh
      float v[8];
      float top = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = 0.f;
      if (hq < gn && w < W) {
        const uint4 raw = *(const uint4 *)((const uint16_t *)a.q +
                                           ((int64_t)b * a.nq + h * a.G + j0 + hq) * D + 8 * w);
        const uint32_t x[4] = {raw.x, raw.y, raw.z, raw.w};
        if (a.q_dtype == CQ_BF16) {
          const float scb = bf2f(f2bf(a.scale));
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            v[2 * i] = bf2f(f2bf(__uint_as_float(x[i] << 16) * scb));
            v[2 * i + 1] = bf2f(f2bf(__uint_as_float(x[i] & 0xffff0000u) * scb));
          }
        } else {
          const float sch = h2f(f2h(a.scale));
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            v[2 * i] = h2f(f2h(h2f((uint16_t)(x[i] & 0xffffu)) * sch));
            v[2 * i + 1] = h2f(f2h(h2f((uint16_t)(x[i] >> 16)) * sch));
          }
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) top = fmaxf(top, fabsf(v[e]));
#pragma unroll
      for (int x = 1; x < 32; x *= 2) top = fmaxf(top, __shfl_xor(top, x, 64));
      // bf16: a power of two brings the row's top to [2^13, 2^14), so that the fp16
      // form is exact down to 2^-31 of it (0, infinities, NaN: as they are); what it
      // leaves is below 2^-24, scaled by kLow exact down to 2^-69 of the top
      const int ex = (int)(__float_as_uint(top) >> 23);
      const int up = (a.q_dtype != CQ_BF16 || ex == 0 || ex == 255) ? 0 : min(127 + 13 - ex, 100);
      const float f = __uint_as_float((uint32_t)(127 + up) << 23);
      if (w == 0) lds.cs[hh] = kLog2e * __uint_as_float((uint32_t)(127 - up) << 23);
      bool some = false;
      if (w < 4 * NS) {
        const int qkg = w / NS, qj = w - qkg * NS;
        h8_t q, l;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float x = v[e] * f;
          q[e] = (_Float16)x;
          const float rest = ex == 255 ? 0.f : x - (float)q[e];
          l[e] = (_Float16)(rest * kLow);
          some |= rest != 0.f;
        }
        auto put = [&](int i, h8_t y) {
          lds.qn[i][qj][16 * qkg + hh] = y;
          lds.qc[i][qj][16 * qkg + hh] = h8_t{y[0], y[4], y[1], y[5], y[2], y[6], y[3], y[7]};
        };
        put(0, q);
        put(1, l);
      }
      const bool any = __any(some);
      if (lane == 0) lds.low[wave] = any;
    }
    __syncthreads();
    int low = 0;
#pragma unroll
    for (int i = 0; i < kWaves; ++i) low |= lds.low[i];
    low = __builtin_amdgcn_readfirstlane(low);
    const float cs = lds.cs[col];

    float m_run = -INFINITY;  // per column's head, log2 units
    float l_run = 0.f;        // sum of p over this lane's tokens
    f4_t acc[NT];             // tile 8x + e: heads 4kg + r (Few: r), dim 8 (NU col + x) + e
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[n] = f4_t{0.f, 0.f, 0.f, 0.f};
    WideWave &Ws = lds.w[wave];

    for (int64_t c0l = t0 + (int64_t)wave * kChunk; c0l < t1; c0l += kWaves * kChunk) {
      const int c0 = (int)c0l;
      const int nt = (int)min((int64_t)kChunk, t1 - c0l);
      const int gk_base = div_stride(c0, sk, isk), gk_last = div_stride(c0 + nt - 1, sk, isk);
      const int gv_base = div_stride(c0, sv, isv), gv_last = div_stride(c0 + nt - 1, sv, isv);
      // ---- token phase: one token per lane ------------------------------------------
      uint32_t s16;
      {
        const bool valid = lane < nt;
        const int t = c0 + (valid ? lane : nt - 1);
        const int gk = div_stride(t, sk, isk), gv = div_stride(t, sv, isv);
        const int slk = (valid && t != gk * sk) ? t - gk - 1 : -1;
        const int slv = (valid && t != gv * sv) ? t - gv - 1 : -1;
        const uint32_t sk16 = bload16(r_sck, (uint32_t)slk * 2u);  // slot -1: past the buffer, 0
        const uint32_t sv16 = bload16(r_scv, (uint32_t)slv * 2u);
        Ws.slot_k[lane] = slk;
        Ws.slot_v[lane] = slv;
        Ws.gkl[lane] = gk - gk_base;
        Ws.gvl[lane] = gv - gv_base;
        s16 = sk16 | (sv16 << 16);
      }
      wave_lds_sync();
      // ---- the chunk's loads ------------------------------------------------------------
      // (slot -1 wraps past the buffer, or to bytes of row 0: the token's scale is 0)
      uint32_t kw[4][NS];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t row = (uint32_t)Ws.slot_k[16 * i + col] * krow;
        if constexpr (Dense) {
#pragma unroll
          for (int j = 0; j < NS; ++j)
            kw[i][j] = fbk == 4 ? bload32(r_pkk, row + 4u * (NS * kg + j))
                                : bload_dense(r_pkk, row, NS * kg + j, fbk);
        } else {
          bload_words<NS>(r_pkk, row + 4u * NS * kg, kw[i]);
        }
      }
      uint4 ka[NS];
      {
        const uint32_t row = (uint32_t)min(gk_base + col, gk_last) * (uint32_t)(2 * D);
#pragma unroll
        for (int j = 0; j < NS; ++j)  // dims past D: zeros
          ka[j] = bload128(r_kfk, NS * kg + j < W ? row + 16u * (NS * kg + j) : 0x80000000u);
      }
      uint32_t vw[4][4][NU];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int4 s4 = *(const int4 *)&Ws.slot_v[16 * i + 4 * kg];
        const int ss[4] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const uint32_t row = (uint32_t)ss[r] * vrow;
          if constexpr (Dense) {
#pragma unroll
            for (int x = 0; x < NU; ++x)
              vw[i][r][x] = fbv == 4 ? bload32(r_pkv, row + 4u * (NU * col + x))
                                     : bload_dense(r_pkv, row, NU * col + x, fbv);
          } else {
            bload_words<NU>(r_pkv, row + 4u * NU * col, vw[i][r]);
          }
        }
      }
      uint4 va[4][NU];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        // groups past the chunk's last: zeros (their P_g is 0, and 0 * inf is not)
        const int g = gv_base + 4 * kg + r;
        const uint32_t row = g <= gv_last ? (uint32_t)g * (uint32_t)(2 * D) : 0x80000000u;
#pragma unroll
        for (int x = 0; x < NU; ++x) va[r][x] = bload128(r_kfv, row + 16u * (NU * col + x));
      }
      Ws.s16[lane] = s16;

      // ---- q'.anchor table -----------------------------------------------------------------
      {
        f4_t d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int i = low; i >= 0; --i) {  // (low parts first, brought back to q's scale)
#pragma unroll
          for (int j = 0; j < NS; ++j) d = mfma32(__builtin_bit_cast(h8_t, ka[j]), lds.qn[i][j][lane], d);
          if (i) d *= 1.f / kLow;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) Ws.qa[4 * kg + r][col] = d[r];
      }
      wave_lds_sync();
      // ---- scores of tokens 16i + 4kg + r, head col ------------------------------------------
      f4_t d[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) d[i] = f4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
      for (int i1 = low; i1 >= 0; --i1) {
#pragma unroll
        for (int j = 0; j < NS; ++j) {
          const h8_t q = lds.qc[i1][j][lane];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            asm volatile("" : "+v"(kw[i][j]));  // (keeps the unpacked words out of registers)
            d[i] = mfma32(codes_k(kw[i][j]), q, d[i]);
          }
        }
        if (i1) {
#pragma unroll
          for (int i = 0; i < 4; ++i) d[i] *= 1.f / kLow;
        }
      }
      float sc[4][4];
      float mx = -INFINITY;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int tb = 16 * i + 4 * kg;
        const int4 g4 = *(const int4 *)&Ws.gkl[tb];
        const uint4 s4 = *(const uint4 *)&Ws.s16[tb];
        const int gr[4] = {g4.x, g4.y, g4.z, g4.w};
        const uint32_t sr[4] = {s4.x, s4.y, s4.z, s4.w};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float x = __builtin_fmaf((float)as_h2(sr[r]).x, d[i][r], Ws.qa[gr[r]][col]) * cs;
          sc[i][r] = tb + r < nt ? x : -INFINITY;
          mx = fmaxf(mx, sc[i][r]);
        }
      }
      // ---- lazy running max ----------------------------------------------------------------------
      mx = shfl_max_kg(mx);
      if (__any(mx > m_run + kTau)) {
        const float m_new = fmaxf(m_run, mx);
        const float f = (m_run == -INFINITY) ? 0.f : fast_exp2(m_run - m_new);
        l_run *= f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float fr = __shfl(f, Few ? r : 4 * kg + r, 64);  // factor of acc's head r
#pragma unroll
          for (int n = 0; n < NT; ++n) acc[n][r] *= fr;
        }
        m_run = m_new;
      }
      const float mref = (m_run == -INFINITY) ? 0.f : m_run;

      // ---- weights, P_g and the code product: K index kg of step (i, r) is token
      // 16i + 4kg + r, whose weight for head col this lane holds -----------------------
      f4_t pg = {0.f, 0.f, 0.f, 0.f};  // groups 4kg + r, head col
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int tb = 16 * i + 4 * kg;
        const uint4 s4 = *(const uint4 *)&Ws.s16[tb];
        const int4 g4 = *(const int4 *)&Ws.gvl[tb];
        const uint32_t sr[4] = {s4.x, s4.y, s4.z, s4.w};
        const int gr[4] = {g4.x, g4.y, g4.z, g4.w};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float p = fast_exp2(sc[i][r] - mref);
          l_run += p;
          pg = mfma_f32(gr[r] == col ? 1.f : 0.f, p, pg);
          const float w = p * (float)as_h2(sr[r]).y;
#pragma unroll
          for (int x = 0; x < NU; ++x) {
            const uint32_t c = vw[i][r][x] ^ 0x88888888u;
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[8 * x + e] = weigh<Few>(w, code_f32(c, e), acc[8 * x + e]);
          }
        }
      }
      // ---- anchors: K index kg of step r is group 4kg + r ------------------------------
#pragma unroll
      for (int r = 0; r < 4; ++r) {
#pragma unroll
        for (int x = 0; x < NU; ++x) {
          const uint32_t a4[4] = {va[r][x].x, va[r][x].y, va[r][x].z, va[r][x].w};
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const h2_t a2 = as_h2(a4[e >> 1]);
            acc[8 * x + e] = weigh<Few>(pg[r], (float)(e & 1 ? a2.y : a2.x), acc[8 * x + e]);
          }
        }
      }
    }

    // ---- totals, workgroup merge, split epilogue -------------------------------------------------
    l_run = shfl_sum_kg(l_run);
    if constexpr (Few) {  // the four kg's tokens
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[n][r] = shfl_sum_kg(acc[n][r]);
    }
    WideMerge<NS> &M = lds.mg;
    constexpr int kO = WideMerge<NS>::kO;
    __syncthreads();  // wave scratch becomes the merge area
    if (kg == 0) {
      M.m[wave][col] = m_run;
      M.l[wave][col] = l_run;
    }
    for (int p0 = 0; p0 < gn; p0 += kMergeHeads) {
      const int pn = min(kMergeHeads, gn - p0);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int hp = (Few ? r : 4 * kg + r) - p0;
        if (hp >= 0 && hp < pn && (!Few || r == kg)) {
          float4 *dst = (float4 *)&M.t[wave][hp][8 * NU * col];
#pragma unroll
          for (int n = 0; n < NT; n += 4)
            dst[n / 4] = make_float4(acc[n][r], acc[n + 1][r], acc[n + 2][r], acc[n + 3][r]);
        }
      }
      __syncthreads();
      for (int e = tid; e < pn * (kO / 4); e += kThreadsMfma) {
        const int hp = e / (kO / 4), d0 = 4 * (e - hp * (kO / 4));
        const int hh = p0 + hp;
        float mw[kWaves], mm = -INFINITY;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
          mw[w] = M.m[w][hh];
          mm = fmaxf(mm, mw[w]);
        }
        float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
        float L = 0.f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
          const float f = (mw[w] == -INFINITY) ? 0.f : fast_exp2(mw[w] - mm);
          const float4 t = *(const float4 *)&M.t[w][hp][d0];
          o.x += f * t.x;
          o.y += f * t.y;
          o.z += f * t.z;
          o.w += f * t.w;
          L += f * M.l[w][hh];
        }
        *(float4 *)&M.o[hh][d0] = o;
        if (d0 == 0) {
          M.wm[hh] = mm;
          M.wl[hh] = L;
        }
      }
      __syncthreads();
    }
    finish_workgroup(a, b, h, chunk, j0, gn, sg.slot, sg.live, M.wm, M.wl, &M.o[0][0], kO);
    __syncthreads();  // the next segment's staging reuses the merge area
  }
}

template <int NS>
const void *wide_kernel(bool dense, bool few) {
  if (few) return dense ? (const void *)decode_wide_kernel<NS, true, true> : (const void *)decode_wide_kernel<NS, false, true>;
  return dense ? (const void *)decode_wide_kernel<NS, true, false> : (const void *)decode_wide_kernel<NS, false, false>;
}
const void *wide_kernel(int D, bool dense, bool few) {
  if (D <= 64) return wide_kernel<2>(dense, few);
  if (D <= 96) return wide_kernel<3>(dense, few);
  if (D <= 128) return wide_kernel<4>(dense, few);
  return wide_kernel<8>(dense, few);
}

// One 8-wave workgroup per CU (two waves per SIMD of up to 256 registers)
int64_t wide_resident() {
  return resident_workgroups(wide_kernel<8>(false, true), kThreadsMfma, kSlotWide);
}

}  // namespace

int64_t wide_max_resident() { return wide_resident(); }

bool wide_supported(const DecodeArgs &a) {
  if (a.D % 8 || a.D < 32) return false;
  if (a.q_dtype != CQ_F16 && a.q_dtype != CQ_BF16) return false;
  if (a.max_T >= (1 << 24) || a.stride[0] < 4 || a.stride[1] < 4) return false;
  // buffer resources address each (sequence, head) region with 32-bit offsets
  for (int i = 0; i < 2; ++i)
    if (a.cap_kf[i] * a.D * 2 >= ((int64_t)1 << 31) ||
        a.cap_pf[i] * 4 * row_words_of(a.D, a.fbits[i]) >= ((int64_t)1 << 31))
      return false;
  if ((int64_t)a.B * units_of(a.max_T) >= ((int64_t)1 << 31)) return false;  // 32-bit unit indices
  return (((uintptr_t)a.kf[0] | (uintptr_t)a.kf[1] | (uintptr_t)a.q) & 15u) == 0;
}

int launch_decode_wide(DecodeArgs &a, void *workspace, size_t ws_bytes, hipStream_t stream) {
  a.chunk_heads = kHeads;
  a.n_chunks = (a.G + kHeads - 1) / kHeads;
  const int64_t cols = (int64_t)a.H * a.n_chunks;
  const int64_t P = std::min(std::max((int64_t)1, wide_resident() / cols),
                             (int64_t)a.B * units_of(a.max_T));
  a.nsplit = (int)balanced_slots(P, a.max_T);
  a.split_len = kUnit;
  const int st = setup_workspace(a, workspace, ws_bytes);
  if (st) return st;
  const dim3 grid((unsigned)P, (unsigned)cols), blk(kThreadsMfma);
  void *args[] = {&a};
  const void *k = wide_kernel(a.D, a.fbits[0] != 4 || a.fbits[1] != 4, a.G <= 4);
  if (hipLaunchKernel(k, grid, blk, args, 0, stream) != hipSuccess) {
    (void)hipGetLastError();
    return CQ_ERR_LAUNCH;
  }
  return hipGetLastError() == hipSuccess ? CQ_OK : CQ_ERR_LAUNCH;
}

}  // namespace cq
