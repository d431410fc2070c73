// cq_flash.hip — attention of many query rows over the ChronoQuant cache for
// the calls the head_dim-128 prefill kernel (cq_prefill.hip) does not take:
// other head dims, boolean masks, dense residual rows.
//
// Reference semantics: the reconstruct fallback of chronoquant_sdpa
// (attention.py:8-20, 61-74 over cache.py:131-160): K and V rebuilt as fp16(a +
// fp16(fp16(c) * s)); fp16 queries: q' = fp16(q * fp16(scale)), scores rounded
// to fp16, masked scores fp16's lowest value, softmax in fp32, fp16 weights,
// fp16 output; bf16 queries: q' = bf16(q * bf16(scale)), then everything in
// fp32 (bf16 x fp16 promotes) to the bf16 output.
//
// Three launches on the caller's scratch:
//   rebuild_kernel  K and V of every token as fp16 rows of DP dims (head_dim
//                   rounded up to 64, 96, 128 or 256; the rest zero), once per
//                   call: a chunk's 256-row tiles read each block several
//                   times, and rebuilding it in each of them would cost more
//                   than the rows' round trip through L2.
//   flash_kernel    a workgroup of 8 waves takes 256 rows (position x q head of
//                   one kv head) and one of nsplit pieces of their keys; each
//                   wave 32 rows by v_mfma_f32_32x32x16_f16, with the K and V
//                   blocks shared through LDS.
//   combine_kernel  with several splits, the log-sum-exp merge of their
//                   unnormalised (m, l, o).
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "cq_decode_common.h"

namespace cq {
namespace {

typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef float f16v_t __attribute__((ext_vector_type(16)));
typedef float f2_t __attribute__((ext_vector_type(2)));
typedef int i4_t __attribute__((ext_vector_type(4)));
typedef short s4_t __attribute__((ext_vector_type(4)));

constexpr int kRows = 256;     // query rows per workgroup
constexpr int kThreads = 512;  // 8 waves of 32 rows
// Lazy-rescale threshold and lift of the weights, log2 units: fp16 queries' weights
// (one fp16 operand) are kept at up to 2^14 and clear of fp16's subnormals for 20
// binary orders below the running maximum; bf16 queries' (split ones) at up to 2^15,
// with both halves clear of them for 15 to 16.
template <bool Bf16>
struct Weights {
  static constexpr float kTau = Bf16 ? 1.f : 8.f;
  static constexpr float kLift = Bf16 ? 14.f : 6.f;
};
// Scores of at least -kSafe leave a hidden key, at the type's lowest value, the weight
// 0 (fp16: 104 nats and the scores' rounding above -65504).
template <bool Bf16>
constexpr float kSafe = Bf16 ? 1e38f : 65000.f;
constexpr float kFull = 0.25f;         // a weight whose fp16 pair hi + lo holds 23 bits
constexpr float kUp = 17179869184.f;   // 2^34: scale of what a pair leaves of a smaller one

enum MaskKind { kMaskNone = 0, kMaskCausal = 1, kMaskBool = 2 };

struct FlashArgs {
  const uint16_t *k, *v;  // rebuilt rows [B * H][T][DP]
  const uint16_t *q;      // [B][nq][L][D] fp16 or bf16
  uint16_t *out;          // as q
  const uint8_t *mask;    // kMaskBool: element (b, h, g, i, t) at the strides below
  int64_t ms[5];
  int32_t *blocks;        // kMaskBool: lists of visible key blocks (scan_mask_kernel); null: all
  int planes, nblk;       // ... [planes][tiles][1 + nblk]
  int B, H, G, nq, D, L, T;
  int causal;
  float scale;
  const uint32_t *top_k, *top_v;  // [B * H][ntop]: largest |K| and |V| (launch_rebuild)
  int ntop;
  int nsplit, tiles;
  float *part_ml;   // [row][nsplit][2]  (m in log2 units, l)
  float *part_acc;  // [row][nsplit][D]
};

__device__ __forceinline__ h2_t as_h2(uint32_t u) { return __builtin_bit_cast(h2_t, u); }
__device__ __forceinline__ uint32_t as_u(h2_t h) { return __builtin_bit_cast(uint32_t, h); }
__device__ __forceinline__ f16v_t mfma(h8_t a, h8_t b, f16v_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ uint4 bload128(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  const i4_t v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0);
  return uint4{(uint32_t)v[0], (uint32_t)v[1], (uint32_t)v[2], (uint32_t)v[3]};
}
// gfx950 LDS transpose read: in each group of 16 lanes, lane 4j + c addresses 4
// fp16 of row j (columns 4c ..), and lane r receives column r of rows 0..3.
__device__ __forceinline__ uint2 lds_read_tr16(const uint16_t *p) {
  const s4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4_t *)(p));
  return __builtin_bit_cast(uint2, v);
}

__device__ __forceinline__ h8_t finite_or_0(h8_t v) {
  uint4 u = __builtin_bit_cast(uint4, v);
  auto f = [](uint32_t w) {
    return ((w & 0x7c00u) == 0x7c00u ? 0u : w & 0xffffu) | ((w & 0x7c000000u) == 0x7c000000u ? 0u : w & 0xffff0000u);
  };
  return __builtin_bit_cast(h8_t, uint4{f(u.x), f(u.y), f(u.z), f(u.w)});
}

// 16-byte piece p of block row `key` sits in slot swz(p, key) of the row.  K
// rows are read by 8 or 16 lanes of consecutive keys at one piece: the low key
// bits spread them over the banks.  V rows are read four consecutive keys x 64
// bytes at a time: the low two key bits move a row to another 64 bytes.  (12
// pieces per row do that by themselves, up to the K reads' second four keys.)
template <int PR>
__device__ __forceinline__ int swz_k(int p, int key) {
  if (PR == 12) return p ^ ((key >> 2) & 3);
  if (PR == 8) return p ^ (key & 7);
  return p ^ (key & 15);
}
template <int PR>
__device__ __forceinline__ int swz_v(int p, int key) {
  if (PR == 12) return p;
  if (PR == 8) return p ^ (((key >> 1) & 1) << 2);
  return p ^ (((key & 3) << 2) | ((key >> 2) & 3));
}

// Key blocks that a 256-row tile of a boolean mask sees, as a list (its length
// first), so that the flash kernel passes over the hidden ones: a hidden key's
// weight is exactly 0 beside any visible one whose score is not near the lowest value
// itself (kSafe).  A tile with a row that sees no key lists every block (such a row
// weighs all keys alike).
// scan_mask_kernel: a workgroup per 1024 keys and 64 rows of a tile, lane = 16 keys,
// the rows dealt to its 4 waves; masks that do not depend on the q head are read once per
// position, and once for all kv heads when they do not depend on those.  It leaves
// a flag per block and per (row, 1024 keys), from which list_kernel makes the list.
// (257 queries x 2 sequences under a window of 1000 of 4001 keys: the flash kernel
// 86 -> 35 us for 4 + 3 us of scan and list.  With a tile's rows or its keys in fewer
// workgroups the scan's loads were one after the other: 40 and 15 us.)
constexpr int kScanKeys = 1024, kScanRows = 64, kScanGroups = kRows / kScanRows;

struct MaskScan {
  uint8_t *blk;  // [planes][tiles][kScanGroups][chunks * kScanKeys / keys]
  uint8_t *row;  // [planes][tiles][chunks][kRows]
  int chunks, keys;
};

__global__ __launch_bounds__(256) void scan_mask_kernel(FlashArgs a, MaskScan m) {
  __shared__ uint64_t s_seen[4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int chunk = blockIdx.x / kScanGroups, group = blockIdx.x % kScanGroups;
  const int tile = blockIdx.y, plane = blockIdx.z;
  const int b = plane / a.H, h = plane - b * a.H;  // plane 0 stands for all of them when planes == 1
  const int row0 = tile * kRows + group * kScanRows, end = min(row0 + kScanRows, a.G * a.L);
  const int64_t pt = (int64_t)plane * a.tiles + tile;
  const uint8_t *base = a.mask + b * a.ms[0] + h * a.ms[1];
  const int k0 = chunk * kScanKeys + 16 * lane;
  const bool whole = a.ms[4] == 1 && k0 + 16 <= a.T;
  // with one mask row per position, step over the positions' first rows (the
  // group's first position may begin before it)
  const int step = a.ms[2] == 0 ? a.G : 1;
  const int first = step == 1 ? row0 : row0 / a.G * a.G;
  uint32_t seen = 0;
#pragma unroll 4
  for (int r = first + step * wave; r < end; r += 4 * step) {
    const int pos = r / a.G, head = r - pos * a.G;
    const uint8_t *p = base + head * a.ms[2] + (int64_t)pos * a.ms[3];
    uint32_t w[4] = {0u, 0u, 0u, 0u};
    if (whole) {
      __builtin_memcpy(w, p + k0, 16);
    } else {
      for (int e = 0; e < 16 && k0 + e < a.T; ++e) w[0] |= p[(int64_t)(k0 + e) * a.ms[4]];
    }
    const uint32_t any = w[0] | w[1] | w[2] | w[3];
    seen |= any;
    const bool row = __any(any != 0);
    if (lane == 0)
      m.row[(pt * m.chunks + chunk) * kRows + group * kScanRows + max(r, row0) - row0] = row;
  }
  const uint64_t bal = __ballot(seen != 0);
  if (lane == 0) s_seen[wave] = bal;
  __syncthreads();
  const int per = kScanKeys / m.keys, lanes = m.keys / 16;  // blocks here, lanes of a block
  if (tid < per) {
    const uint64_t all = s_seen[0] | s_seen[1] | s_seen[2] | s_seen[3];
    m.blk[((pt * kScanGroups + group) * m.chunks + chunk) * per + tid] = ((all >> (lanes * tid)) & ((1ull << lanes) - 1)) != 0;
  }
}

// One wave per (tile, plane).
__global__ __launch_bounds__(64) void list_kernel(FlashArgs a, MaskScan m) {
  const int lane = threadIdx.x, tile = blockIdx.x, plane = blockIdx.y;
  const int64_t pt = (int64_t)plane * a.tiles + tile;
  const int row0 = tile * kRows, rows = min(kRows, a.G * a.L - row0);
  const uint8_t *flags = m.row + pt * m.chunks * kRows;
  bool blind = false;
  for (int i = lane; i < rows; i += 64) {
    // the row that stands for this one: the first of its position in the group
    const int rep = a.ms[2] == 0 ? max((row0 + i) / a.G * a.G - row0, i / kScanRows * kScanRows) : i;
    bool sees = false;
#pragma unroll 4
    for (int c = 0; c < m.chunks; ++c) sees |= flags[c * kRows + rep] != 0;
    blind |= !sees;
  }
  const bool all = __any(blind);
  const int nb = m.chunks * (kScanKeys / m.keys);
  const uint8_t *blk = m.blk + pt * kScanGroups * nb;
  int32_t *list = a.blocks + pt * (1 + a.nblk);
  int n = 0;
  for (int i0 = 0; i0 < a.nblk; i0 += 64) {
    bool on = all;
    if (i0 + lane < a.nblk) {
#pragma unroll
      for (int g = 0; g < kScanGroups; ++g) on |= blk[g * nb + i0 + lane] != 0;
    }
    on = on && i0 + lane < a.nblk;
    const uint64_t bal = __ballot(on);
    if (on) list[1 + n + __popcll(bal & ((1ull << lane) - 1))] = i0 + lane;
    n += __popcll(bal);
  }
  if (lane == 0) list[0] = n;
}

template <int DP>
struct alignas(16) FlashLds {
  static constexpr int kKeys = DP > 128 ? 32 : 64;  // keys per block
  // K-steps of a wave's q' beyond the 6 that it keeps in registers: each lane's
  // own operands (DP = 256: O^T alone takes half of the 256 registers; with 8 steps
  // in registers the masked bf16 instance spills)
  static constexpr int kQSteps = DP > 128 ? DP / 16 - 6 : 0;
  uint16_t k[2][kKeys * DP], v[2][kKeys * DP];
  uint4 q[kThreads / 64][kQSteps ? kQSteps : 1][kQSteps ? 64 : 1];
  float top[3][kThreads / 64];  // largest sum of |q'|, |K| and |V| by wave
};

// Rows R = tile * 256 + 32 wave + (lane & 31) of the G * L rows of kv head
// (b, h): position R / G, q head R % G.  S^T = K Q^T gives lane (row, half)
// the scores of keys 8 (r / 4) + 4 half + r % 4, which is the order the P.V
// product's K index takes them in (the transpose reads of V follow it), so the
// weights never leave their lane; O^T = V^T P^T keeps a row in one lane (and
// its other half), so the softmax state is per lane.
//
// Bound: a block's chain (scores, softmax, P.V, a barrier) with two waves per SIMD
// in flight: on the first shape below the matrix cores are busy for 24 % of the
// time, the VALU for 35, LDS for 12, without bank conflicts, and the waves wait for
// 49.  512 queries of 16 heads over 8192 keys of 4 heads, head_dim 256, bf16 (66.6
// GFLOP, and half as many again for the weights' low halves), with the rebuild (11)
// and the merge (12): 172 us where few scores lie 11 nats below their row's maximum
// (below), 201 with outlier channels in the keys, 280 with scores of a spread of 16,
// where the reconstruct fallback's products, softmax and conversions took 977; fp16
// 120.  257 fp16 queries x 2 sequences under a boolean window over 4001 keys: 63 us
// in all against 803; bf16 77.
//
// Split weights (bf16 queries): the fallback holds weights in fp32, so P enters
// as an fp16 pair hi + lo, two products per V operand; a pair holds 23 bits of a
// weight of at least kFull, 2^-16 or less of the largest.  What it leaves of smaller
// ones goes through a round of products of its own, scaled by kUp, and a second one
// (23 bits down to 2^-84 of the largest, some down to 2^-106): tokens behind a
// dominant one whose V is 0 are off by 9 % at a gap of 25 nats without them.  A block
// with no score 11 nats below its row's maximum needs no round.  (Where most blocks
// need them, the rounds take as long as the rest: 512 queries of 32 heads over 8192
// keys of 8 heads x 64 dims with outlier channels 158 us, 84 with the pairs alone.)
template <int DP, bool Bf16, bool Masked>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void flash_kernel(FlashArgs a) {
  using Lds = FlashLds<DP>;
  constexpr int KT = Lds::kKeys, PR = DP / 8, NK = KT / 32, ND = DP / 32, NS = DP / 16;
  constexpr int NR = NS - Lds::kQSteps;  // K-steps of q' in registers
  constexpr int kPieces = KT * PR, NP = (kPieces + kThreads - 1) / kThreads;
  __shared__ Lds lds;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r32 = lane & 31, half = lane >> 5;
  // workgroups of one (sequence, kv head, split) are a multiple of the group
  // count apart, on one XCD when that is a multiple of 8: they share its L2
  const int groups = a.B * a.H * a.nsplit;
  const int tile = (int)blockIdx.x / groups, grp = (int)blockIdx.x - tile * groups;
  const int bh = grp / a.nsplit, split = grp - bh * a.nsplit;
  const int b = bh / a.H, h = bh - b * a.H;
  const int G = a.G, L = a.L, T = a.T, GL = G * L;
  const int row0 = tile * kRows, row = row0 + 32 * wave + r32;
  const bool valid = row < GL;
  const int rr = valid ? row : GL - 1;
  const int pos = rr / G, head = rr - pos * G;
  const int64_t grow = ((int64_t)b * a.nq + h * G + head) * L + pos;

  // the rows' largest |K| and |V|, wanted further down
  const bool checked = Masked || Bf16 || a.causal;
  float top_k = 0.f, top_v = 0.f;
  if (checked && tid < a.ntop) {
    top_k = (float)a.top_k[(int64_t)bh * a.ntop + tid];
    top_v = (float)a.top_v[(int64_t)bh * a.ntop + tid];
  }

  // ---- q' (B operand of the score product): dims 16s + 8 half .. + 7 ---------
  // bf16: scaled by a power of two that brings the row's largest magnitude to
  // [2^13, 2^14), so that its fp16 form loses no bit down to 2^-31 of that;
  // cs takes the scores back, in log2 units.  low: a row of this wave has elements
  // that lose bits (a block's score products then begin with theirs).
  // sum: of the magnitudes of this half of the row.
  float sum = 0.f;
  h8_t qf[NR];
  float cs = kLog2e;
  bool low = false;
  auto raw_of = [&](int s) {
    const int d0 = 16 * s + 8 * half;
    return (valid && d0 < a.D) ? *(const uint4 *)(a.q + grow * a.D + d0) : uint4{0u, 0u, 0u, 0u};
  };
  // element e of 8 of a bf16 row, as q' times f; what its fp16 form loses
  auto scaled = [&](const uint4 &u, int e, float f) {
    const uint32_t w = e < 2 ? u.x : e < 4 ? u.y : e < 6 ? u.z : u.w;
    const float x = __uint_as_float(e & 1 ? w & 0xffff0000u : w << 16);
    return bf2f(f2bf(x * bf2f(f2bf(a.scale)))) * f;
  };
  auto lost = [](float x) {
    const float h = (float)(_Float16)x;
    return fabsf(h) < INFINITY ? x - h : 0.f;
  };
  {
    auto keep = [&](int s, h8_t v) {
      if (s < NR) qf[s] = v;
      else lds.q[wave][s - NR][Lds::kQSteps ? lane : 0] = __builtin_bit_cast(uint4, v);
    };
    if constexpr (Bf16) {
      float top = 0.f;
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const uint4 u = raw_of(s);
#pragma unroll
        for (int e = 0; e < 8; ++e) top = fmaxf(top, fabsf(scaled(u, e, 1.f)));
      }
      top = xor32_max(top);
      const int e = (int)(__float_as_uint(top) >> 23);  // biased exponent
      // 0, and infinities and NaN, stay as they are
      const int up = (e == 0 || e == 255) ? 0 : min(127 + 13 - e, 100);
      const float f = __uint_as_float((uint32_t)(127 + up) << 23);
      cs = kLog2e * __uint_as_float((uint32_t)(127 - up) << 23);
      float left = 0.f;
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const uint4 u = raw_of(s);  // (again: the rows are in cache, registers are not)
        h8_t v;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float x = scaled(u, e, f);
          v[e] = (_Float16)x;
          left = fmaxf(left, fabsf(lost(x)));
          sum += fabsf(x);
        }
        keep(s, v);
      }
      low = __any(left > 0.f);
      sum *= __uint_as_float((uint32_t)(127 - up) << 23);
    } else {
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const h8_t v = __builtin_bit_cast(h8_t, raw_of(s)) * (_Float16)a.scale;
#pragma unroll
        for (int e = 0; e < 8; ++e) sum += fabsf((float)v[e]);
        keep(s, v);
      }
    }
  }

  // ---- may hidden keys be passed over? ---------------------------------------------
  // A score is at least -sum |q'| max |K|.  Where that is not above the lowest value
  // by enough (unsafe), or V holds an infinity or NaN (vbad; 0 times it is NaN),
  // hidden keys are computed like any other.  (One word of each maximum per thread and
  // a barrier: 2 us of the shapes above, and 1 us of the rebuild that leaves them.)
  bool unsafe = false, vbad = false;
  if (checked) {
    sum = xor32_sum(sum);
    const float ms = wave_max(sum == sum ? sum : INFINITY), mk = wave_max(top_k), mv = wave_max(top_v);
    if (lane == 0) lds.top[0][wave] = ms, lds.top[1][wave] = mk, lds.top[2][wave] = mv;
    __syncthreads();
    float m[3] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < kThreads / 64; ++i)
#pragma unroll
      for (int j = 0; j < 3; ++j) m[j] = fmaxf(m[j], lds.top[j][i]);
    vbad = __builtin_amdgcn_readfirstlane((int)m[2]) >= 0x7c00;
    const float bound = m[0] * h2f((uint16_t)m[1]);
    unsafe = vbad || __builtin_amdgcn_readfirstlane(!(bound < kSafe<Bf16>));  // (NaN: not safe)
  }
  const float low_score = Bf16 ? -1.7e38f : -65504.f;

  // ---- key range ----------------------------------------------------------------
  const int qbase = T - L;
  const int lim = a.causal ? qbase + pos : T - 1;           // last key this row sees
  const int lim_all = a.causal ? qbase + row0 / G : T - 1;  // ... every row sees
  const int last = min(row0 + kRows, GL) - 1;
  const int key_end = a.causal && !unsafe ? qbase + last / G + 1 : T;
  // blocks in the order they are taken: all up to key_end, or the tile's list
  const int32_t *list = nullptr;
  if constexpr (Masked) {
    if (a.blocks && !unsafe)
      list = a.blocks + ((int64_t)(a.planes == 1 ? 0 : bh) * a.tiles + tile) * (1 + a.nblk);
  }
  const int n_all = list ? __builtin_amdgcn_readfirstlane(list[0]) : (key_end + KT - 1) / KT;
  auto block_id = [&](int kb) { return list ? __builtin_amdgcn_readfirstlane(list[1 + kb]) : kb; };
  const int kb_lo = (int)((int64_t)split * n_all / a.nsplit);
  const int kb_hi = (int)((int64_t)(split + 1) * n_all / a.nsplit);

  // ---- block staging: piece tid + 512 i of the block's rows, contiguous ----------
  const uint32_t kv_bytes = (uint32_t)T * (uint32_t)(DP * 2);
  const __amdgpu_buffer_rsrc_t rk = make_rsrc(a.k + (int64_t)bh * T * DP, kv_bytes);
  const __amdgpu_buffer_rsrc_t rv = make_rsrc(a.v + (int64_t)bh * T * DP, kv_bytes);
  int wk[NP], wv[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const int pid = tid + kThreads * i, key = pid / PR, p = pid - key * PR;
    wk[i] = key * DP + 8 * swz_k<PR>(p, key);
    wv[i] = key * DP + 8 * swz_v<PR>(p, key);
  }
  uint4 gk[NP], gv[NP];
  auto load_block = [&](int kb) {
    const uint32_t base = (uint32_t)kb * (uint32_t)(KT * DP * 2) + 16u * tid;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      if (kPieces % kThreads == 0 || tid + kThreads * i < kPieces) {
        gk[i] = bload128(rk, base + 16u * kThreads * i);
        gv[i] = bload128(rv, base + 16u * kThreads * i);
      }
    }
  };
  auto store_block = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      if (kPieces % kThreads == 0 || tid + kThreads * i < kPieces) {
        *(uint4 *)&lds.k[buf][wk[i]] = gk[i];
        *(uint4 *)&lds.v[buf][wv[i]] = gv[i];
      }
    }
  };

  const uint8_t *mrow = nullptr;
  int64_t mst = 0;
  if constexpr (Masked) {
    mrow = a.mask + b * a.ms[0] + h * a.ms[1] + head * a.ms[2] + (int64_t)pos * a.ms[3];
    mst = a.ms[4];
  }

  float m_run = -INFINITY, l_run = 0.f;
  f16v_t acc[ND];
#pragma unroll
  for (int dt = 0; dt < ND; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[dt][r] = 0.f;

  // This lane's operands in a block.  K: rows 32 kt + r32, piece 2s + half.  V (transpose
  // reads): keys 16 j + 4 half + jj (+ 8), columns 32 dt + 16 g + 4 c.  The swizzles are
  // the same for every kt and j, and for rows of a power of two of bytes a step's place
  // is the first one's with s or dt brought in by an exclusive or.  At 256 dims the 48
  // places are made anew from it at each use: kept, they and the accumulators leave too
  // few of the 256 registers for the rest (40 to 144 bytes of spills per lane, a block's
  // loads among them).
  const int jj = (lane & 15) >> 2, g1 = (lane >> 4) & 1, c4 = lane & 3;
  constexpr bool kPow2 = PR != 12, kAnew = DP > 128;
  auto k_at = [&](int s) { return r32 * DP + 8 * swz_k<PR>(2 * s + half, r32); };
  auto v_at = [&](int dt, int more) {
    const int key = 4 * half + jj + more;
    return key * DP + 8 * swz_v<PR>(4 * dt + 2 * g1 + (c4 >> 1), key) + 4 * (c4 & 1);
  };
  int k_first = k_at(0), v_first = v_at(0, 0);

  int id = 0, id_next = 0;  // this block's place in the keys, the next one's
  // bad_c: V holds infinities or NaN.  They meet the weights' high halves alone (a low
  // half or a rest may be 0 or of the other sign, where the weight is neither).  (A
  // loop of its own: 4 us of 197 on the shape above without any such value.)
  auto block = [&](int kb, auto buf_c, auto bad_c) {
    constexpr int cur = decltype(buf_c)::value;
    constexpr bool bad = decltype(bad_c)::value;
    const int k0 = id * KT;
    if (kb + 1 < kb_hi) load_block(id_next);  // uniform
    id = id_next;
    id_next = block_id(min(kb + 2, kb_hi - 1));

    // mask bytes of keys k0 + 32 kt + 8 q + 4 half .. + 3 (1: visible)
    uint32_t mb[NK][4];
    if constexpr (Masked) {
      if (mst == 1 && k0 + KT <= T) {
#pragma unroll
        for (int kt = 0; kt < NK; ++kt)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            __builtin_memcpy(&mb[kt][q], mrow + k0 + 32 * kt + 8 * q + 4 * half, 4);
      } else {
#pragma unroll
        for (int kt = 0; kt < NK; ++kt)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            mb[kt][q] = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int key = k0 + 32 * kt + 8 * q + 4 * half + e;
              if (key < T) mb[kt][q] |= (uint32_t)(mrow[(int64_t)key * mst] != 0) << (8 * e);
            }
          }
      }
    }

    // ---- scores ------------------------------------------------------------------
    float sc[NK][16];
    h2_t s2[NK][8];
#pragma unroll
    for (int kt = 0; kt < NK; ++kt) {
      f16v_t d;
#pragma unroll
      for (int r = 0; r < 16; ++r) d[r] = 0.f;
      if constexpr (Bf16) {
        if (low) {  // (below 2^-24; scaled by kUp exact down to 2^-65 of the row's largest)
#pragma unroll 1
          for (int s = 0; s < NS; ++s) {
            const uint4 kv = *(const uint4 *)&lds.k[cur][32 * kt * DP + k_at(s)];
            const uint4 u = raw_of(s);
            h8_t v;
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = (_Float16)(lost(scaled(u, e, kLog2e / cs)) * kUp);
            d = mfma(__builtin_bit_cast(h8_t, kv), v, d);
          }
#pragma unroll
          for (int r = 0; r < 16; ++r) d[r] *= 1.f / kUp;
        }
      }
      if constexpr (kAnew) asm volatile("" : "+v"(k_first));
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const uint4 kv = *(const uint4 *)&lds.k[cur][32 * kt * DP + (kPow2 ? k_first ^ (16 * s) : k_at(s))];
        const h8_t q8 = s < NR ? qf[s < NR ? s : 0] : __builtin_bit_cast(h8_t, lds.q[wave][s < NR ? 0 : s - NR][Lds::kQSteps ? lane : 0]);
        d = mfma(__builtin_bit_cast(h8_t, kv), q8, d);
      }
      if constexpr (Bf16) {
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[kt][r] = d[r] * cs;
      } else {
#pragma unroll
        for (int r = 0; r < 16; r += 2) s2[kt][r >> 1] = __builtin_convertvector(f2_t{d[r], d[r + 1]}, h2_t);
      }
    }
    auto put = [&](int kt, int r, float x) {
      if constexpr (Bf16) sc[kt][r] = x;
      else s2[kt][r >> 1][r & 1] = (_Float16)x;
    };
    if constexpr (Masked) {
      // hidden keys take the lowest finite value (a row that sees no key
      // weighs all of them alike); -inf is for keys past the end
#pragma unroll
      for (int kt = 0; kt < NK; ++kt)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (!((mb[kt][r >> 2] >> (8 * (r & 3))) & 0xffu)) put(kt, r, low_score);
    }
    auto past = [&](int end, float x) {  // keys beyond a row's end
#pragma unroll
      for (int kt = 0; kt < NK; ++kt)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (k0 + 32 * kt + 8 * (r >> 2) + 4 * half + (r & 3) > end) put(kt, r, x);
    };
    // (uniform: only a tile's last blocks)
    if constexpr (!Masked) {
      if (k0 + KT - 1 > lim_all) past(lim, unsafe ? low_score : -INFINITY);
    }
    if (k0 + KT > T) past(T - 1, -INFINITY);
    float mx;
    if constexpr (Bf16) {
      mx = sc[0][0];
#pragma unroll
      for (int kt = 0; kt < NK; ++kt)
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = max_nn(mx, sc[kt][r]);
    } else {
      h2_t m2 = s2[0][0];
#pragma unroll
      for (int kt = 0; kt < NK; ++kt)
#pragma unroll
        for (int i = 0; i < 8; ++i) m2 = __builtin_elementwise_maximum(m2, s2[kt][i]);
      mx = max_nn((float)m2.x, (float)m2.y) * kLog2e;
    }
    mx = xor32_max(mx);
    // ---- lazy running max ----------------------------------------------------------
    if (__any(mx > m_run + Weights<Bf16>::kTau)) {
      const float m_new = fmaxf(m_run, mx);
      const float f = (m_run == -INFINITY) ? 0.f : fast_exp2(m_run - m_new);
      l_run *= f;
#pragma unroll
      for (int dt = 0; dt < ND; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[dt][r] *= f;
      m_run = m_new;
    }
    const float mref = ((m_run == -INFINITY) ? 0.f : m_run) - Weights<Bf16>::kLift;
    bool deep = false;  // a weight below kFull (uniform; 0s count as well)
    if constexpr (Bf16) {
      float mn = sc[0][0];
#pragma unroll
      for (int kt = 0; kt < NK; ++kt)
#pragma unroll
        for (int r = 0; r < 16; ++r) mn = fminf(mn, sc[kt][r]);
      deep = __any(mn < mref - 2.f);
    }
    // ---- weights and P.V, 16 keys a step --------------------------------------------
    // (tight: V operands one at a time, as the registers of a rare round allow)
    auto product = [&](int j, const h2_t (&ph)[4], const h2_t (&pl)[4], bool tight) {
      const h8_t bh8 = __builtin_bit_cast(h8_t, uint4{as_u(ph[0]), as_u(ph[1]), as_u(ph[2]), as_u(ph[3])});
      h8_t bl8;
      if constexpr (Bf16)
        bl8 = __builtin_bit_cast(h8_t, uint4{as_u(pl[0]), as_u(pl[1]), as_u(pl[2]), as_u(pl[3])});
      if constexpr (kAnew) asm volatile("" : "+v"(v_first));
      const uint16_t *v16 = &lds.v[cur][16 * j * DP];
#pragma unroll
      for (int dt = 0; dt < ND; ++dt) {
        const int at = kPow2 ? v_first ^ (32 * dt) : v_at(dt, 0);
        // 8 keys on: the swizzle's third bit turns, where it has one
        const int at2 = kAnew ? (at ^ 16) + 8 * DP : v_at(dt, 8);
        const uint2 v1 = lds_read_tr16(v16 + at);
        const uint2 v2 = lds_read_tr16(v16 + at2);
        const h8_t va = __builtin_bit_cast(h8_t, uint4{v1.x, v1.y, v2.x, v2.y});
        const h8_t vl = bad ? finite_or_0(va) : va;
        acc[dt] = mfma(bad && tight ? vl : va, bh8, acc[dt]);
        if constexpr (Bf16) acc[dt] = mfma(vl, bl8, acc[dt]);
        if (tight) __builtin_amdgcn_sched_barrier(0);
      }
    };
    // the fp16 pair of x0, x1; rest: what it leaves of those below kFull
    auto split = [&](float &x0, float &x1, h2_t &hi, h2_t &lo, bool rest) {
      hi = __builtin_convertvector(f2_t{x0, x1}, h2_t);
      if constexpr (bad) {  // (0 for a weight of 0 alone)
        if (hi.x == (_Float16)0.f && x0 > 0.f) hi.x = (_Float16)0x1p-24f;
        if (hi.y == (_Float16)0.f && x1 > 0.f) hi.y = (_Float16)0x1p-24f;
      }
      const float d0 = x0 - (float)hi.x, d1 = x1 - (float)hi.y;
      lo = __builtin_convertvector(f2_t{d0, d1}, h2_t);
      if (rest) {
        x0 = fabsf(x0) < kFull ? d0 - (float)lo.x : 0.f;
        x1 = fabsf(x1) < kFull ? d1 - (float)lo.y : 0.f;
      }
    };
    const h2_t ones = {(_Float16)1.f, (_Float16)1.f};
#pragma unroll
    for (int j = 0; j < KT / 16; ++j) {
      h2_t ph[4], pl[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int kt = j >> 1, r = 8 * (j & 1) + 2 * i;
        if constexpr (Bf16) {
          float p0 = fast_exp2(sc[kt][r] - mref), p1 = fast_exp2(sc[kt][r + 1] - mref);
          l_run += p0 + p1;
          split(p0, p1, ph[i], pl[i], deep);
          if (deep) sc[kt][r] = p0, sc[kt][r + 1] = p1;
        } else {
          const h2_t x = s2[kt][r >> 1];
          ph[i] = h2_t{(_Float16)fast_exp2(__builtin_fmaf((float)x.x, kLog2e, -mref)),
                       (_Float16)fast_exp2(__builtin_fmaf((float)x.y, kLog2e, -mref))};
          l_run = __builtin_amdgcn_fdot2(ph[i], ones, l_run, false);
        }
      }
      product(j, ph, pl, false);
    }
    if constexpr (Bf16) {
      // the rests, kUp larger a round, into acc as much larger: |acc| <= 2^55 (2^15 a
      // weight, 2^16 a value, 2^24 keys) stays a number in both rounds
      float down = 1.f;
#pragma unroll 1
      for (int round = deep ? 0 : 2; round < 2; ++round) {
        float any = 0.f;
#pragma unroll
        for (int kt = 0; kt < NK; ++kt)
#pragma unroll
          for (int r = 0; r < 16; ++r) any = fmaxf(any, fabsf(sc[kt][r]));
        if (!__any(any > 0.f)) break;
        down *= 1.f / kUp;
#pragma unroll
        for (int dt = 0; dt < ND; ++dt)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[dt][r] *= kUp;
#pragma unroll
        for (int j = 0; j < KT / 16; ++j) {
          h2_t ph[4], pl[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int kt = j >> 1, r = 8 * (j & 1) + 2 * i;
            sc[kt][r] *= kUp;
            sc[kt][r + 1] *= kUp;
            split(sc[kt][r], sc[kt][r + 1], ph[i], pl[i], true);
          }
          product(j, ph, pl, true);
        }
      }
      if (down != 1.f) {
#pragma unroll
        for (int dt = 0; dt < ND; ++dt)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[dt][r] *= down;
      }
    }
    if (kb + 1 < kb_hi) store_block(cur ^ 1);
    __syncthreads();
  };

  if (kb_lo < kb_hi) {  // uniform
    id = block_id(kb_lo);
    id_next = block_id(min(kb_lo + 1, kb_hi - 1));
    load_block(id);
    store_block(0);
  }
  __syncthreads();
  auto run = [&](auto bad_c) {
    for (int kb = kb_lo; kb < kb_hi;) {
      block(kb++, std::integral_constant<int, 0>{}, bad_c);
      if (kb >= kb_hi) break;
      block(kb++, std::integral_constant<int, 1>{}, bad_c);
    }
  };
  if (Bf16 && vbad) run(std::integral_constant<bool, Bf16>{});
  else run(std::false_type{});

  // ---- output: lane (row, half) holds dims 32 dt + 8 q + 4 half .. + 3 ---------------
  l_run = xor32_sum(l_run);
  if (!valid) return;
  if (a.nsplit > 1) {
    const int64_t pr = grow * a.nsplit + split;
    if (half == 0) *(float2 *)(a.part_ml + 2 * pr) = make_float2(m_run, l_run);
    float *o = a.part_acc + pr * a.D;
#pragma unroll
    for (int dt = 0; dt < ND; ++dt)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int d0 = 32 * dt + 8 * q + 4 * half;
        if (d0 < a.D)
          *(float4 *)(o + d0) = make_float4(acc[dt][4 * q], acc[dt][4 * q + 1], acc[dt][4 * q + 2],
                                            acc[dt][4 * q + 3]);
      }
    return;
  }
  // (scores of -inf alone: NaN, as the fallback's softmax gives)
  const float inv = l_run > 0.f ? 1.f / l_run : NAN;
  uint16_t *o = a.out + grow * a.D;
#pragma unroll
  for (int dt = 0; dt < ND; ++dt)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int d0 = 32 * dt + 8 * q + 4 * half;
      uint16_t w[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = acc[dt][4 * q + e] * inv;
        w[e] = Bf16 ? f2bf(x) : f2h(x);
      }
      if (d0 < a.D)
        *(uint2 *)(o + d0) = uint2{(uint32_t)w[0] | ((uint32_t)w[1] << 16),
                                   (uint32_t)w[2] | ((uint32_t)w[3] << 16)};
    }
}

// Log-sum-exp merge of the splits: thread = (row, 4 dims).  Bound: reading the
// partials once.
template <bool Bf16>
__global__ __launch_bounds__(256) void combine_kernel(const float *part_ml, const float *part_acc,
                                                      uint16_t *out, int D, int nsplit, float empty,
                                                      int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int d4 = D / 4;
  const int64_t row = i / d4;
  const int d0 = 4 * (int)(i - row * d4);
  const float2 *ml = (const float2 *)part_ml + row * nsplit;
  const float *pa = part_acc + row * nsplit * D + d0;
  float M = -INFINITY;
  for (int s = 0; s < nsplit; ++s) M = fmaxf(M, ml[s].x);
  float Ls = 0.f;
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
  for (int s = 0; s < nsplit; ++s) {
    const float2 x = ml[s];
    const float4 v = *(const float4 *)(pa + (int64_t)s * D);
    const float w = (x.x == -INFINITY) ? 0.f : fast_exp2(x.x - M);
    Ls += w * x.y;
    o.x += w * v.x;
    o.y += w * v.y;
    o.z += w * v.z;
    o.w += w * v.w;
  }
  const float inv = Ls > 0.f ? 1.f / Ls : (Ls == 0.f ? empty : Ls);
  const float ov[4] = {o.x * inv, o.y * inv, o.z * inv, o.w * inv};
  uint16_t w[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) w[e] = Bf16 ? f2bf(ov[e]) : f2h(ov[e]);
  *(uint2 *)(out + row * D + d0) =
      uint2{(uint32_t)w[0] | ((uint32_t)w[1] << 16), (uint32_t)w[2] | ((uint32_t)w[3] << 16)};
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
int padded_dim(int D) { return D <= 64 ? 64 : D <= 96 ? 96 : D <= 128 ? 128 : 256; }

struct FlashPlan {
  int dp, tiles, nsplit;
  int nblk, chunks;
  int ntop;
  size_t kv, ml, acc, lists, tops;  // bytes: K (and V) rows, partial (m, l), partial o, block lists, tops
  size_t bytes() const { return 2 * kv + ml + acc + lists + tops; }
};

constexpr int kMaxFlashSplits = 32;
static_assert(kMaxTops <= kThreads, "a thread reads one top");
constexpr size_t kMaxListBytes = 64 << 20;

// Key splits: one workgroup per CU, so the grid runs in ceil(groups * ns /
// CUs) rounds of ceil(blocks / ns) key blocks each plus a fixed part (the
// prologue and the epilogue, about 5 blocks' time; writing and merging partials
// another 5).  Against 1 to 32 splits on 15 shapes (head_dim 64 to 256, 300 to 32768
// keys, 2 to 256 groups, masked or not) it takes the fastest or one at most 5 % slower,
// except for few rows over few keys, where it does not see the merge grow with the
// splits: 8 groups of 32 blocks, 29.5 us with 32 and 22.9 with 8; 4 of 16, 33.0 with 16
// and 29.5 with 8.  (Masked calls are planned for all their blocks, not the listed.)
FlashPlan flash_plan(int64_t B, int64_t H, int64_t G, int64_t D, int64_t L, int64_t T) {
  FlashPlan p;
  p.dp = padded_dim((int)D);
  p.tiles = (int)((G * L + kRows - 1) / kRows);
  const int64_t cus = std::max<int64_t>(1, resident_workgroups(
      reinterpret_cast<const void *>(flash_kernel<128, false, false>), kThreads, kSlotFlash));
  const int64_t groups = (int64_t)p.tiles * B * H, keys = p.dp > 128 ? 32 : 64;
  const int64_t blocks = (T + keys - 1) / keys;
  int64_t best = 1, best_cost = 0;
  for (int64_t ns = 1; ns <= kMaxFlashSplits && ns <= blocks; ++ns) {
    const int64_t cost = (groups * ns + cus - 1) / cus * ((blocks + ns - 1) / ns + (ns > 1 ? 10 : 5));
    if (ns == 1 || cost < best_cost) best = ns, best_cost = cost;
  }
  p.nsplit = (int)best;
  const size_t rows = (size_t)(B * H * G * L);
  p.kv = round256((size_t)(B * H * T) * p.dp * 2);
  p.nblk = (int)blocks;
  const int64_t chunks = (T + kScanKeys - 1) / kScanKeys;
  p.chunks = (int)chunks;
  p.lists = (size_t)(B * H * p.tiles) *
            ((1 + blocks) * 4 + chunks * (kScanGroups * kScanKeys / keys + kRows));  // lists, blk, row
  p.lists = p.lists <= kMaxListBytes ? round256(p.lists) : 0;
  p.ntop = rebuild_tops(T, p.dp);
  p.tops = round256((size_t)(2 * B * H * p.ntop) * 4);
  p.ml = best > 1 ? round256(rows * best * 8) : 0;
  p.acc = best > 1 ? round256(rows * best * D * 4) : 0;
  return p;
}

int flash_shape(const cq_cache_desc *c, int n_q_heads, int64_t n_q, int64_t seq_len) {
  const int D = c->head_dim;
  if (D % 8 || D < 8) return CQ_ERR_UNSUPPORTED;
  if (n_q_heads < 1 || n_q_heads % c->n_kv_heads) return CQ_ERR_SHAPE;
  const int64_t G = n_q_heads / c->n_kv_heads;
  if (n_q < 1 || seq_len < 1) return CQ_ERR_SHAPE;
  // 32-bit row indices, byte offsets into one kv head's rows, and grid
  if (G * n_q >= ((int64_t)1 << 30) || seq_len * padded_dim(D) * 2 >= ((int64_t)1 << 31) - (1 << 16))
    return CQ_ERR_UNSUPPORTED;
  const int64_t tiles = (G * n_q + kRows - 1) / kRows;
  if (tiles * c->batch * c->n_kv_heads * kMaxFlashSplits >= ((int64_t)1 << 31)) return CQ_ERR_UNSUPPORTED;
  return CQ_OK;
}

template <int DP, bool Bf16>
void launch_flash(const FlashArgs &a, bool masked, dim3 grid, hipStream_t s) {
  if (masked) flash_kernel<DP, Bf16, true><<<grid, dim3(kThreads), 0, s>>>(a);
  else flash_kernel<DP, Bf16, false><<<grid, dim3(kThreads), 0, s>>>(a);
}
template <bool Bf16>
void launch_flash(const FlashArgs &a, int dp, bool masked, dim3 grid, hipStream_t s) {
  if (dp == 64) launch_flash<64, Bf16>(a, masked, grid, s);
  else if (dp == 96) launch_flash<96, Bf16>(a, masked, grid, s);
  else if (dp == 128) launch_flash<128, Bf16>(a, masked, grid, s);
  else launch_flash<256, Bf16>(a, masked, grid, s);
}

}  // namespace

void launch_combine(bool bf16, const float *part_ml, const float *part_acc, uint16_t *out,
                    int64_t rows, int D, int nsplit, float empty, hipStream_t s) {
  const int64_t n = rows * (D / 4);
  const dim3 grid((unsigned)((n + 255) / 256)), blk(256);
  if (bf16) combine_kernel<true><<<grid, blk, 0, s>>>(part_ml, part_acc, out, D, nsplit, empty, n);
  else combine_kernel<false><<<grid, blk, 0, s>>>(part_ml, part_acc, out, D, nsplit, empty, n);
}

}  // namespace cq

using namespace cq;

extern "C" size_t cq_flash_scratch_size(const cq_cache_desc *cache, int32_t n_q_heads, int64_t n_q,
                                        int64_t seq_len) {
  if (validate_cache(cache) || flash_shape(cache, n_q_heads, n_q, seq_len)) return 0;
  return flash_plan(cache->batch, cache->n_kv_heads, n_q_heads / cache->n_kv_heads, cache->head_dim,
                    n_q, seq_len).bytes();
}

extern "C" int cq_flash_attn(const cq_cache_desc *cache, const void *q, int32_t q_dtype,
                             int32_t n_q_heads, int64_t n_q, float scale, int32_t mask_kind,
                             const uint8_t *mask, const int64_t *mask_strides, int64_t seq_len,
                             void *out, void *scratch, size_t scratch_bytes, cq_stream_t stream) {
  int st = validate_cache(cache);
  if (st) return st;
  if (!q || !out) return CQ_ERR_ARG;
  if (q_dtype != CQ_F16 && q_dtype != CQ_BF16) return CQ_ERR_DTYPE;
  if (mask_kind < kMaskNone || mask_kind > kMaskBool) return CQ_ERR_ARG;
  if (mask_kind == kMaskBool && (!mask || !mask_strides)) return CQ_ERR_ARG;
  st = flash_shape(cache, n_q_heads, n_q, seq_len);
  if (st) return st;
  if (mask_kind == kMaskCausal && seq_len < n_q) return CQ_ERR_SHAPE;
  for (const cq_component *p : {&cache->k, &cache->v})
    if (num_keyframes(seq_len, p->stride) > p->cap_keyframes ||
        num_pframes(seq_len, p->stride) > p->cap_pframes)
      return CQ_ERR_CAPACITY;
  if (((uintptr_t)q | (uintptr_t)out) & 15) return CQ_ERR_ALIGN;
  const int64_t G = n_q_heads / cache->n_kv_heads;
  const FlashPlan p = flash_plan(cache->batch, cache->n_kv_heads, G, cache->head_dim, n_q, seq_len);
  if (!scratch || scratch_bytes < p.bytes()) return CQ_ERR_WORKSPACE;
  if ((uintptr_t)scratch & 255) return CQ_ERR_ALIGN;
  const hipStream_t s = (hipStream_t)stream;
  char *w = (char *)scratch;
  FlashArgs a;
  a.k = (const uint16_t *)w;
  a.v = (const uint16_t *)(w + p.kv);
  a.part_ml = (float *)(w + 2 * p.kv);
  a.part_acc = (float *)(w + 2 * p.kv + p.ml);
  a.q = (const uint16_t *)q;
  a.out = (uint16_t *)out;
  a.mask = mask;
  for (int i = 0; i < 5; ++i) a.ms[i] = mask_kind == kMaskBool ? mask_strides[i] : 0;
  a.B = cache->batch;
  a.H = cache->n_kv_heads;
  a.G = (int)G;
  a.nq = n_q_heads;
  a.D = cache->head_dim;
  a.L = (int)n_q;
  a.T = (int)seq_len;
  a.causal = mask_kind == kMaskCausal;
  a.scale = scale;
  a.nsplit = p.nsplit;
  a.tiles = p.tiles;
  a.nblk = p.nblk;
  a.planes = a.ms[0] == 0 && a.ms[1] == 0 ? 1 : a.B * a.H;
  a.blocks = nullptr;
  if (mask_kind == kMaskBool && p.lists && a.planes <= 65535 && p.tiles <= 65535) {
    a.blocks = (int32_t *)(w + 2 * p.kv + p.ml + p.acc);
    const size_t n = (size_t)a.planes * p.tiles;
    MaskScan m;
    m.chunks = p.chunks;
    m.keys = p.dp > 128 ? 32 : 64;
    m.blk = (uint8_t *)(a.blocks + n * (1 + p.nblk));
    m.row = m.blk + n * kScanGroups * p.chunks * (kScanKeys / m.keys);
    scan_mask_kernel<<<dim3((unsigned)(p.chunks * kScanGroups), (unsigned)p.tiles, (unsigned)a.planes), dim3(256), 0, s>>>(a, m);
    list_kernel<<<dim3((unsigned)p.tiles, (unsigned)a.planes), dim3(64), 0, s>>>(a, m);
  }
  uint32_t *tops = (uint32_t *)(w + 2 * p.kv + p.ml + p.acc + p.lists);
  a.ntop = p.ntop;
  a.top_k = tops;
  a.top_v = tops + (int64_t)a.B * a.H * p.ntop;
  st = launch_rebuild(*cache, seq_len, p.dp, (uint16_t *)w, (uint16_t *)(w + p.kv), tops,
                      tops + (int64_t)a.B * a.H * p.ntop, s);
  if (st) return st;
  const dim3 grid((unsigned)(p.tiles * a.B * a.H * p.nsplit));
  const bool masked = mask_kind == kMaskBool;
  if (q_dtype == CQ_BF16) launch_flash<true>(a, p.dp, masked, grid, s);
  else launch_flash<false>(a, p.dp, masked, grid, s);
  if (p.nsplit > 1)
    launch_combine(q_dtype == CQ_BF16, a.part_ml, a.part_acc, a.out, (int64_t)a.B * a.nq * a.L, a.D,
                   p.nsplit, NAN, s);
  return hipGetLastError() == hipSuccess ? CQ_OK : CQ_ERR_LAUNCH;
}
