// INT8-QK / f16-PV attention for the query blocks that would leave most of the chip idle: the whole
// call of a short sequence, and the last, partial round of a longer one. The operands, the result and its
// tolerance are those of k_attention_hm (attention_hm.hip); what differs is who does the work, and the
// last bits: each group of keys has its own running max, the scores are multiplied by their scales
// directly (there by one FMA that also takes out the accumulators' bias), and the row sum adds the
// probabilities in f32 before they are rounded to f16 for PV (there the rounded ones). A call's rows can
// come from both kernels, so a row's last bits depend on how its call is divided. Against 64 bits, 1,024
// tokens of 8 heads: 2.9e-4 of the result here, 3.0e-4 there.
//
// k_attention_hm gives 256 queries of one head to a workgroup, which walks every key: a call of B
// blocks takes ceil(B / CUs) rounds of a whole walk, however few blocks the last round holds. Here
// a workgroup's eight waves are QW (one or two) tiles of 32 queries times KS = 8 / QW groups of keys:
// group g walks the 64-key stages g, g + KS, ..., each wave with an online softmax of its own, and the KS
// partial results of a tile are combined through LDS at the end. A block's work is then spread
// over 8 / QW workgroups, each of which takes 1 / KS of the walk, without device memory for the
// partial results.
//
// The waves of a workgroup walk different keys, so nothing is shared through LDS: a lane loads its
// MFMA operands straight from memory (L2, in practice), whole 128-byte lines of K and of V^T per
// stage. Per stage: the V^T operands are requested, QK runs on the K operands requested half a stage
// before, and the two 32-key halves follow, softmax and PV each, with the next stage's K operands
// requested between them: each request has about half a stage to land. What bounds it is what a CU
// can pull through its L1 (about 20 bytes a clock), so a stage costs more than in k_attention_hm and
// the calls that fill the chip stay there (the rule and its measurements are at split_plan below).
// 16x16 MFMAs, whose operand loads cover 64 bytes of a row instead of 32, measured 10 % slower.
//
// QK uses v_mfma_i32_32x32x32_i8 on K rows in swap23 order, so that a lane's accumulator registers
// 8g..8g+7 are keys 16g + 8(lane/32) + 0..7 of their 32-key half, PV's B operand with V^T in
// natural key order. The FP6 form (kFp6) reads 32-byte blocks of 24 bytes of e2m3 codes and
// accumulates from zero.
#include <algorithm>
#include <type_traits>

#include "internal.hpp"

namespace h3 {
namespace {

constexpr int kWaves = 8;
constexpr int kThreads = 64 * kWaves;
constexpr int kTileQ = 32;
constexpr int kBlockQ = 256;        // the query block of k_attention_hm
constexpr int kKeys = 64;           // keys per stage
constexpr int kORow = 128 + 4;      // floats per query of a partial result (rows 4 banks apart)
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kSumLimit = 256.0f;        // a lane's stage sum above this: raise the running max
constexpr int kRsrcWord3 = 0x00020000;     // raw buffer: 32-bit data format, no swizzle
constexpr int kCpolNt = 2;                 // buffer store cache policy: non-temporal

typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef unsigned int v2u __attribute__((ext_vector_type(2)));
typedef int v6i __attribute__((ext_vector_type(6)));
typedef int v8i __attribute__((ext_vector_type(8)));

struct Args {
  const char* qi;
  const float* qs;
  const char* ki;
  const float* ks;
  const uint16_t* vt;
  uint16_t* out;
  uint32_t tokens;      // keys, and readable query rows
  uint32_t rows;        // query rows written
  uint32_t capacity;    // row pitch of V^T
  uint32_t out_stride;
  uint32_t kv_head_limit, head_limit;
  // code rows: byte pitch of a token's row and of a head; scales: element pitch of both
  uint32_t k_row, q_row;
  uint64_t k_head, q_head;
  uint32_t ks_key, ks_head, qs_row, qs_head;
  // Units: the full blocks from `first` on (block = head * full + query block) in `per_full` pieces
  // of qw_full tiles, then the heads' last, partial blocks in `per_rest` pieces of qw_rest tiles.
  uint32_t first, full, units_full, per_full, qw_full, per_rest, qw_rest;
  uint32_t units, per_xcd;  // all units; ceil(units / 8)
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes,
                                           kRsrcWord3);
}
__device__ __forceinline__ uint32_t swap23(uint32_t m) {
  return (m & ~12u) | ((m & 4u) << 1) | ((m & 8u) >> 1);
}
// The max of the two lanes that hold a query (lane % 32), on the vector pipe.
__device__ __forceinline__ float query_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false,
                                                  false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// A lane's share of a 32-row operand of K or Q, of row lane % 32: INT8, bytes 16 (lane / 32) .. +15
// of each 32-channel quarter; FP6, the 24 bytes of codes of 32-byte blocks lane / 32 and + 2.
template <bool kFp6>
struct Rows {
  v4i c0, c1, c2, c3;
};
template <>
struct Rows<true> {
  v8i c0, c1;
};
__device__ __forceinline__ v4i load16(__amdgpu_buffer_rsrc_t from, uint32_t off) {
  return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(from, off, 0, 0));
}
__device__ __forceinline__ v8i load24(__amdgpu_buffer_rsrc_t from, uint32_t off) {
  const v4i lo = load16(from, off);
  const v2u hi = __builtin_bit_cast(v2u, __builtin_amdgcn_raw_buffer_load_b64(from, off + 16, 0, 0));
  return v8i{lo[0], lo[1], lo[2], lo[3], (int)hi[0], (int)hi[1], 0, 0};
}
template <bool kFp6>
__device__ __forceinline__ Rows<kFp6> load_rows(__amdgpu_buffer_rsrc_t from, uint32_t off) {
  if constexpr (kFp6)
    return {load24(from, off), load24(from, off + 64)};
  else
    return {load16(from, off), load16(from, off + 32), load16(from, off + 64),
            load16(from, off + 96)};
}

// S^T of 32 keys and 32 queries, exact: S in int32 (INT8, |S| <= 128^3), S / 4 in f32 (FP6).
template <bool kFp6>
using Scores = std::conditional_t<kFp6, v16f, v16i>;
template <bool kFp6>
__device__ __forceinline__ Scores<kFp6> scores(const Rows<kFp6>& k, const Rows<kFp6>& q) {
  Scores<kFp6> s = {};
  if constexpr (kFp6) {  // formats 2 = FP6 e2m3; scales 127 = 2^0
    s = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(k.c0, q.c0, s, 2, 2, 0, 127, 0, 127);
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(k.c1, q.c1, s, 2, 2, 0, 127, 0, 127);
  } else {
    s = __builtin_amdgcn_mfma_i32_32x32x32_i8(k.c0, q.c0, s, 0, 0, 0);
    s = __builtin_amdgcn_mfma_i32_32x32x32_i8(k.c1, q.c1, s, 0, 0, 0);
    s = __builtin_amdgcn_mfma_i32_32x32x32_i8(k.c2, q.c2, s, 0, 0, 0);
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(k.c3, q.c3, s, 0, 0, 0);
  }
}

template <bool kFp6>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_attention_split(Args g) {
  __shared__ __attribute__((aligned(16))) float part[kWaves][kTileQ][kORow];
  __shared__ float part_m[kWaves][kTileQ], part_l[kWaves][kTileQ];
  __shared__ __attribute__((aligned(16))) float strip[kWaves][kKeys];  // a wave's key scales

  // The unit: head, first query, tiles. The hardware deals workgroup b to XCD b % 8; each XCD takes
  // a contiguous range of the units, so that the units of a head stream its K and V^T through one
  // L2 (256 units of
  // 2,048 keys: 41.7 us, 44.6 dealt out singly).
  const uint32_t unit = (blockIdx.x & 7u) * g.per_xcd + (blockIdx.x >> 3);
  if (unit >= g.units) return;  // the whole workgroup
  const bool is_full = unit < g.units_full;
  const uint32_t per = is_full ? g.per_full : g.per_rest;
  const uint32_t u = is_full ? unit : unit - g.units_full;
  const uint32_t qw = is_full ? g.qw_full : g.qw_rest;
  const uint32_t block = u / per + (is_full ? g.first : 0u);
  const uint32_t head_y = is_full ? block / g.full : block;
  const uint32_t qb = is_full ? block % g.full : g.full;
  const uint32_t q0 = qb * kBlockQ + (u % per) * qw * kTileQ;  // first query of the unit
  const uint32_t kv_head = head_y % g.kv_head_limit;
  const uint32_t head = kv_head % g.head_limit;

  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t groups = kWaves / qw;
  const uint32_t tile = wave / groups, group = wave % groups;
  const uint32_t lane = threadIdx.x & 63, n = lane & 31, half = lane >> 5;
  const uint32_t stages = (g.tokens + kKeys - 1) / kKeys;

  v16f o[4];  // O^T: channels 32 db + 8 (r / 4) + 4 half + r % 4 of query n
#pragma unroll
  for (int db = 0; db < 4; ++db) o[db] = v16f{};
  float m = -1.0e30f, l = 0.0f;

  const uint32_t qt = q0 + tile * kTileQ;  // the wave's first query
  if (qt < g.rows && group < stages) {
    const uint32_t q = min(qt + n, g.tokens - 1);
    constexpr uint32_t kPiece = kFp6 ? 32 : 16;  // bytes between the lane halves' operand pieces
    const Rows<kFp6> qop = load_rows<kFp6>(
        rsrc(g.qi + head * g.q_head + (uint64_t)qt * g.q_row, 31 * g.q_row + 128),
        (q - qt) * g.q_row + kPiece * half);
    const float qsl = g.qs[(uint64_t)q * g.qs_row + (uint64_t)head * g.qs_head] * kLog2e;
    const char* kbase = g.ki + kv_head * g.k_head;
    const float* sbase = g.ks + (uint64_t)kv_head * g.ks_head;
    const uint32_t blk = 128 * g.capacity;  // halves of a head's V^T
    const uint16_t* vbase = g.vt + (uint64_t)kv_head * blk;
    const uint32_t koff = swap23(n) * g.k_row + kPiece * half;
    const uint32_t voff = n * g.capacity * 2 + 16 * half;
    const uint32_t soff = lane * g.ks_key * 4;

    // K operands and key scales of stage st; rows past the last key read as zero
    Rows<kFp6> kop0, kop1;
    float ks_lane;
    auto request_k = [&](uint32_t st) __attribute__((always_inline)) {
      const uint32_t k0 = st * kKeys, live = min(g.tokens - k0, (uint32_t)kKeys);
      const __amdgpu_buffer_rsrc_t rk =
          rsrc(kbase + (uint64_t)k0 * g.k_row, (live - 1) * g.k_row + 128);
      kop0 = load_rows<kFp6>(rk, koff);
      kop1 = load_rows<kFp6>(rk, koff + 32 * g.k_row);
      ks_lane = __builtin_bit_cast(
          float, __builtin_amdgcn_raw_buffer_load_b32(
                     rsrc(sbase + (uint64_t)k0 * g.ks_key, ((live - 1) * g.ks_key + 1) * 4), soff,
                     0, 0));
    };
    request_k(group);

    for (uint32_t st = group; st < stages; st += groups) {
      const uint32_t k0 = st * kKeys, live = min(g.tokens - k0, (uint32_t)kKeys);
      // V^T operands: channel block db, 16-key group kg. The descriptor ends with the head's
      // block; columns past the last key are zero or the next channel row's and meet p = 0.
      const __amdgpu_buffer_rsrc_t rv = rsrc(vbase + k0, (blk - k0) * 2);
      v8h vop[4][4];
      auto request_v = [&](int kg) __attribute__((always_inline)) {
#pragma unroll
        for (int db = 0; db < 4; ++db)
          vop[kg][db] = __builtin_bit_cast(
              v8h, __builtin_amdgcn_raw_buffer_load_b128(rv, voff + db * 64 * g.capacity, 32 * kg, 0));
      };
      request_v(0);
      request_v(1);
      strip[wave][lane] = lane < live ? ks_lane : 1.0f;
      const Scores<kFp6> s0 = scores<kFp6>(kop0, qop), s1 = scores<kFp6>(kop1, qop);
      __builtin_amdgcn_sched_barrier(0);
      request_v(2);  // into the K operands' registers
      request_v(3);
      __builtin_amdgcn_sched_barrier(0);
      // One 32-key half: the probabilities of the scores in `raw`, then PV.
      auto consume = [&](int b, const Scores<kFp6>& raw) __attribute__((always_inline)) {
        // t = S * qs * log2(e), and -inf (times a scale of 1) for a key past the sequence
        v16f t = __builtin_convertvector(raw, v16f);
#pragma unroll
        for (int r = 0; r < 16; ++r) t[r] *= qsl;
        if (live < (uint32_t)kKeys) {
#pragma unroll
          for (int r = 0; r < 16; ++r)
            t[r] = 32u * b + 16 * (r >> 3) + 8 * half + (r & 7) < live ? t[r] : -INFINITY;
        }
        // key scales of registers 4i .. 4i+3
        auto scale4 = [&](int i) __attribute__((always_inline)) {
          return *reinterpret_cast<const float4*>(
              &strip[wave][32 * b + 16 * (i >> 1) + 8 * half + 4 * (i & 1)]);
        };
        v8h p[2];
        float ts;
        auto probabilities = [&](float negm) __attribute__((always_inline)) {
          ts = 0.0f;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float4 k4 = scale4(i);
            const float kk[4] = {k4.x, k4.y, k4.z, k4.w};
            float y[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
              y[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(t[4 * i + e], kk[e], negm));
            ts += (y[0] + y[1]) + (y[2] + y[3]);
#pragma unroll
            for (int e = 0; e < 4; ++e) p[i >> 1][4 * (i & 1) + e] = (_Float16)y[e];
          }
        };
        // As in k_attention_hm: probabilities against the running max so far; a lane whose sum
        // (which bounds each of them) passes 2^8 raises it and computes them again.
        bool raise = b == 0 && st == group;
        if (!raise) {
          probabilities(-m);
          raise = __any(!(ts <= kSumLimit));
        }
        if (raise) {
          float tmax = -INFINITY;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float4 k4 = scale4(i);
            tmax = fmaxf(tmax, fmaxf(fmaxf(t[4 * i] * k4.x, t[4 * i + 1] * k4.y),
                                     fmaxf(t[4 * i + 2] * k4.z, t[4 * i + 3] * k4.w)));
          }
          const float m_new = fmaxf(m, query_max(tmax));
          const float alpha = __builtin_amdgcn_exp2f(m - m_new);
#pragma unroll
          for (int db = 0; db < 4; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[db][r] *= alpha;
          l *= alpha;
          m = m_new;
          probabilities(-m);
        }
        l += ts;
#pragma unroll
        for (int kg = 0; kg < 2; ++kg)
#pragma unroll
          for (int db = 0; db < 4; ++db)
            o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vop[2 * b + kg][db], p[kg], o[db], 0, 0, 0);
      };
      consume(0, s0);
      __builtin_amdgcn_sched_barrier(0);
      if (st + groups < stages) request_k(st + groups);  // into V^T's first registers
      __builtin_amdgcn_sched_barrier(0);
      consume(1, s1);
    }
  }

  // ---- combine the groups of each tile: weights 2^(m - max m), sums in group order
  if (half == 0) part_m[wave][n] = m;
  __syncthreads();
  float top = -1.0e30f;
  for (uint32_t k = 0; k < groups; ++k) top = fmaxf(top, part_m[tile * groups + k][n]);
  const float weight = __builtin_amdgcn_exp2f(m - top);
  const float l_both = (l + __shfl_xor(l, 32)) * weight;
  if (half == 0) part_l[wave][n] = l_both;
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      *reinterpret_cast<float4*>(&part[wave][n][32 * db + 8 * i + 4 * half]) =
          make_float4(o[db][4 * i] * weight, o[db][4 * i + 1] * weight, o[db][4 * i + 2] * weight,
                      o[db][4 * i + 3] * weight);
  __syncthreads();
  const uint32_t live_rows = g.rows > q0 ? min(g.rows - q0, qw * kTileQ) : 0u;
  const __amdgpu_buffer_rsrc_t ro =
      rsrc(g.out + (uint64_t)q0 * g.out_stride, live_rows * g.out_stride * 2);
  for (uint32_t piece = threadIdx.x; piece < qw * kTileQ * 16; piece += kThreads) {
    const uint32_t row = piece >> 4, chunk = piece & 15;  // eight channels of one query
    const uint32_t w0 = (row >> 5) * groups, r = row & 31;
    float sum[8] = {}, lsum = 0.0f;
    for (uint32_t k = 0; k < groups; ++k) {
      const float4 a = *reinterpret_cast<const float4*>(&part[w0 + k][r][8 * chunk]);
      const float4 b = *reinterpret_cast<const float4*>(&part[w0 + k][r][8 * chunk + 4]);
      lsum += part_l[w0 + k][r];
      sum[0] += a.x; sum[1] += a.y; sum[2] += a.z; sum[3] += a.w;
      sum[4] += b.x; sum[5] += b.y; sum[6] += b.z; sum[7] += b.w;
    }
    const float inv = 1.0f / lsum;
    v8h h;
#pragma unroll
    for (int e = 0; e < 8; ++e) h[e] = (_Float16)(sum[e] * inv);
    if (row < live_rows)
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, h), ro,
                                             (row * g.out_stride + head * 128 + 8 * chunk) * 2, 0,
                                             kCpolNt);
  }
}

inline uint32_t div_up(uint32_t a, uint32_t b) { return (a + b - 1) / b; }

// The rule of split_plan prices a call's ways of being divided in us, S stages of 64 keys a block. Fitted to
// every way of 1,125 INT8 calls (1 to 24,000 tokens, 1 to 64 heads, all or some of the rows) behind their
// operands' kernels in captured graphs, to 6.5 % in the root mean square; no call was measured slower than
// undivided by it, in the FP6 form neither (175 calls).
//   k_attention_hm      one block per CU, 5.75 + 1.14 S, to which a share f of the CUs at work adds 0.30 f^2
//                       a stage (the engine clock falls) and 1.15 f in each of the first eight (every block
//                       at once asks for operands just written); after full rounds a last round of share f
//                       takes 0.67 + 0.32 f of one (its blocks start as CUs free up)
//   k_attention_split   5.6 a round of units, 0.45 f in each of the first eight stages, and what its operands
//                       take through the CU's L1: for each live tile and stage an eighth of 5.3 us where
//                       V^T's rows are whole 128-byte lines apart (capacity % 64 == 0: the 32 rows of a load
//                       then lie at the same place of their lines) and of 3.7 (1 + f / 4) where not (1,792
//                       tokens of 4 heads: 25.4 against 21.5 us, 6,000 of 2: 133 against 105)
// so 1,024 tokens of 8 heads take 16.5 us here against 26.3, and 8,193 of 16 heads, whose last round
// would hold 16 blocks of one row each, 530 against 566. 9,375 tokens of one head are faster undivided, 163
// us against 198, and so are most calls of 3,000 keys that fill an eighth of the chip.
constexpr float kMainFixed = 5.75f, kMainStage = 1.14f, kMainFull = 0.30f, kMainCold = 1.15f;
constexpr float kMainLast = 0.67f, kMainLastShare = 0.32f;
constexpr float kSplitFixed = 5.6f, kSplitCold = 0.45f;
constexpr float kSplitAligned = 5.3f, kSplitStage = 3.7f, kSplitFull = 0.25f;
constexpr float kSecondLaunch = 0.6f;
constexpr uint32_t kColdStages = 8;

// Time of `blocks` blocks of `stages` stages on k_attention_hm.
float main_time(uint32_t blocks, uint32_t stages, uint32_t cus) {
  if (blocks == 0) return 0.0f;
  const uint32_t rounds = blocks / cus, extra = blocks % cus;
  const float share = (float)extra / cus;
  auto round = [&](float f) { return kMainFixed + stages * (kMainStage + kMainFull * f * f); };
  const float cold = kMainCold * std::min(stages, kColdStages);
  if (rounds == 0) return cold * share + round(share);
  return cold + round(1.0f) * (rounds + (extra ? kMainLast + kMainLastShare * share : 0.0f));
}

// The time after which `na` units of `da` each, then `nb` of `db`, have run on `cus` CUs in order: the
// CUs that hold no unit of the last round of the first kind take the second kind's from then on.
float makespan(uint32_t na, float da, uint32_t nb, float db, uint32_t cus) {
  const uint32_t rounds = na / cus, extra = na % cus;
  const float early = rounds * da, late = early + (extra ? da : 0.0f);
  float end = late, next_early = early + db, next_late = late + db;
  for (uint32_t left = nb; left > 0;) {
    const bool from_early = extra == 0 || next_early <= next_late;
    float& next = from_early ? next_early : next_late;
    end = std::max(late, next);
    next += db;
    left -= std::min(left, from_early ? cus - extra : extra);
  }
  return end;
}

}  // namespace

SplitPlan split_plan(uint32_t tokens, uint32_t rows, uint32_t heads, uint32_t capacity, uint32_t cus) {
  const uint32_t stages = div_up(tokens, kKeys);
  const uint32_t full = rows / kBlockQ, rest_tiles = div_up(rows % kBlockQ, kTileQ);
  const uint32_t full_blocks = full * heads, rest_blocks = rest_tiles ? heads : 0u;
  SplitPlan best{false, 0, 0, 0};
  const uint32_t mains[2] = {full_blocks / cus * cus, full_blocks};
  // a split has to gain more than the prices' error: 6 % of what follows the full rounds, which every way
  // has, and a microsecond
  const float whole = main_time(full_blocks + rest_blocks, stages, cus);
  float best_time = whole - std::max(1.0f, 0.06f * (whole - main_time(mains[0], stages, cus)));
  for (uint32_t main : mains)
    for (uint32_t qf = 1; qf <= 2; qf *= 2)
      for (uint32_t qr = 1; qr <= 2; qr *= 2) {
        const uint32_t nf = (full_blocks - main) * (kWaves / qf);
        const uint32_t nr = rest_blocks * div_up(rest_tiles, qr);
        if (nf + nr == 0) continue;
        const float share = std::min(1.0f, (float)(nf + nr) / cus);
        const float stage = capacity % 64 == 0 ? kSplitAligned : kSplitStage * (1.0f + kSplitFull * share);
        const float fixed = kSplitFixed + kSplitCold * share * std::min(stages, kColdStages);
        const float df = fixed + stage * stages * qf / kWaves;
        const float dr = fixed + stage * stages * std::min(qr, rest_tiles) / kWaves;
        const float t = main_time(main, stages, cus) + (main ? kSecondLaunch : 0.0f) +
                        makespan(nf, df, nr, dr, cus);
        if (t < best_time) {
          best_time = t;
          best = {true, main, qf, qr};
        }
      }
  return best;
}

hipError_t launch_attention_split(const SplitOperands& x, const SplitPlan& plan,
                                  hipStream_t stream) {
  Args g{};
  g.qi = static_cast<const char*>(x.qi);
  g.qs = x.qs;
  g.ki = static_cast<const char*>(x.ki);
  g.ks = x.ks;
  g.vt = x.vt;
  g.out = x.out;
  g.tokens = x.tokens;
  g.rows = x.rows;
  g.capacity = x.capacity;
  g.out_stride = x.out_stride;
  g.kv_head_limit = x.kv_head_limit;
  g.head_limit = x.head_limit;
  g.k_row = x.k_row;
  g.q_row = x.q_row;
  g.k_head = x.k_head;
  g.q_head = x.q_head;
  g.ks_key = x.ks_key;
  g.ks_head = x.ks_head;
  g.qs_row = x.qs_row;
  g.qs_head = x.qs_head;
  const uint32_t full = x.rows / kBlockQ, rest_tiles = div_up(x.rows % kBlockQ, kTileQ);
  g.first = plan.main_blocks;
  g.full = full;
  g.qw_full = plan.qw_full;
  g.per_full = kWaves / plan.qw_full;
  g.units_full = (full * x.heads - plan.main_blocks) * g.per_full;
  g.qw_rest = plan.qw_rest;
  g.per_rest = std::max(1u, div_up(rest_tiles, plan.qw_rest));
  const uint32_t units = g.units_full + (rest_tiles ? x.heads * g.per_rest : 0u);
  if (units == 0) return hipSuccess;
  g.units = units;
  g.per_xcd = div_up(units, 8);
  const dim3 grid(8 * g.per_xcd);
  if (x.fp6)
    hipLaunchKernelGGL(k_attention_split<true>, grid, dim3(kThreads), 0, stream, g);
  else
    hipLaunchKernelGGL(k_attention_split<false>, grid, dim3(kThreads), 0, stream, g);
  return hipGetLastError();
}

}  // namespace h3
