// INT8 QKV projection with the compact Q/K-rows + V^T epilogue, on gfx950 int8 MFMA.
//
// Semantics follow kernels/gemm_packed_256.loom:14-412 instantiated as h3_gemm_i8_qkv_256
// (kernels/gemm_packed_256.loom:3429-3471; dispatch src/dispatch.rs:756-790 and 1025-1060):
//   acc[m][n]  = sum_k a[m][k] * w[n][k]                       (int8 x int8, exact int32)
//   v          = ((float)acc * w_scale[n]) * a_scale[m] + 0.0   (three IEEE f32 operations)
//   v          = clamp(v, -65472, 65472) when v is finite; inf and NaN pass unchanged
//   columns n < 2N/3 (Q and K): out[m][n], row pitch 2N/3 f16
//   columns n >= 2N/3 (V):      vt[n - 2N/3][m] at element offset M*2N/3, row pitch
//                               cap = ceil(M/256)*256; rows M <= m < cap are written as zero.
// That layout is what Stack::prepare_fused_operands reads on the compact route
// (src/stack.rs:634-661, 1034-1040, 1561-1600): Q/K rows for the RoPE quantizer with a row
// stride of 2*inner, V^T already in the attention's operand layout, no transpose pass.
//
// Design. A workgroup computes a tile with 8 waves, 2 along M x 4 along N, each of kMB x kNB blocks
// of v_mfma_i32_32x32x32_i8: 256 x 256 (128 x 64 per wave), or 128 x 128 and 64 x 128 where the larger
// ones leave CUs idle. K advances 128 bytes per step through a ring of two or four LDS stages filled
// by LDS-DMA (buffer_load ... lds); rows are 16-byte chunks XOR-swizzled by (row/2)%8 so the 32 rows a
// half-wave reads hit distinct banks. Buffer descriptors end at the last valid row, so rows past M
// (or past N) load as zero. The operand order of the MFMA is chosen per region so each lane ends up
// holding four consecutive output elements along the stored direction: W.A^T for Q/K tiles (4
// consecutive channels of one token) and A.W^T for V tiles (4 consecutive tokens of one channel),
// each written as one 8-byte store.
//
// What bounds it: at full occupancy the matrix cores' power (54 % busy at an engine clock of 1.5 GHz,
// 31,104 tokens: 1.95-2.05 POP/s against torch._int_mm's 2.10); with one tile per CU or fewer, what a
// CU can load (20 to 25 bytes a clock) and the latency of a step.
#include <algorithm>
#include <cmath>

#include "internal.hpp"

namespace h3 {
namespace {

constexpr int kBK = 128;                       // K bytes per step
constexpr int kWaves = 8;                      // 2 (M) x 4 (N)
constexpr int kThreads = 64 * kWaves;
constexpr int kGroupM = 4;                     // m-tiles that share one sweep over the n-tiles
constexpr int kCapRows = 256;                  // V^T is padded to a multiple of this many tokens
constexpr int kRsrcWord3 = 0x00020000;         // raw buffer, 32-bit data format, no swizzle
constexpr int kWaitAll = 0 | (7 << 4) | (0 << 8);  // s_waitcnt vmcnt(0) lgkmcnt(0)

// A tile of kMB x kNB 32-row blocks per wave.
template <int kMB, int kNB>
struct Tile {
  static constexpr int kBM = 2 * 32 * kMB;                    // tile rows (tokens)
  static constexpr int kBN = 4 * 32 * kNB;                    // tile columns (output channels)
  static constexpr int kStage = (kBM + kBN) * kBK;            // A rows, then W rows
  static constexpr int kLoads = kStage / 1024 / kWaves;       // 1 KiB DMA loads per wave per step
};

typedef __attribute__((address_space(3))) void lds_void;

struct Args {
  const int8_t* a;
  const int8_t* w;
  const float* ws;
  const float* as;
  uint16_t* out;
  uint32_t m;         // tokens
  uint32_t n;         // output channels (3 * inner)
  uint32_t k;         // reduction length (multiple of 64)
  uint32_t k_stride;  // bytes per operand row
  uint32_t qk_width;  // 2N/3: row pitch of the Q/K rows, first V channel
  uint32_t cap;       // ceil(M/256)*256: row pitch of V^T
  uint32_t tiles_m, tiles_n_qk, tiles_n, total, per_xcd;
};

// A buffer descriptor from wave-uniform values, read back from the first lane so that the
// compiler keeps it in scalar registers.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, uint32_t bytes) {
  const uint64_t v = reinterpret_cast<uint64_t>(base);
  const uint64_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint64_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(lo | (hi << 32)), (short)0,
                                           __builtin_amdgcn_readfirstlane((int)bytes), kRsrcWord3);
}

// LDS byte offset, inside a 128-byte row, of logical 16-byte chunk c for swizzle sw.
__device__ __forceinline__ uint32_t chunk_off(uint32_t c, uint32_t sw) { return 16 * (c ^ sw); }

// f32 epilogue of one accumulator (kernels/gemm_packed_256.loom:370-397).
__device__ __forceinline__ _Float16 finish(int acc, float ws, float as) {
  float v = (float)acc * ws;
  v = v * as;
  v = v + 0.0f;
  if (__builtin_fabsf(v) < __builtin_inff()) v = __builtin_fminf(__builtin_fmaxf(v, -65472.0f), 65472.0f);
  return (_Float16)v;
}

// The operands of one 32-byte substep of a wave, double-buffered by the substep's parity.
template <int kMB, int kNB>
struct Operands {
  v4i a[2][kMB], w[2][kNB];
};
// Operands of substep ks of the stage `st`.
template <int kMB, int kNB>
__device__ __forceinline__ void read_operands(Operands<kMB, kNB>& op, const char* st, int ks,
                                              uint32_t arow, uint32_t wrow, uint32_t half,
                                              uint32_t sw) {
  const uint32_t at = chunk_off(2 * ks + half, sw);
#pragma unroll
  for (int mb = 0; mb < kMB; ++mb)
    op.a[ks & 1][mb] = *reinterpret_cast<const v4i*>(st + (arow + 32 * mb) * kBK + at);
#pragma unroll
  for (int nb = 0; nb < kNB; ++nb)
    op.w[ks & 1][nb] =
        *reinterpret_cast<const v4i*>(st + (Tile<kMB, kNB>::kBM + wrow + 32 * nb) * kBK + at);
}
template <bool kTrans, int kMB, int kNB>
__device__ __forceinline__ void mma_one(const Operands<kMB, kNB>& op, int ks, int mb, int nb,
                                        v16i (&acc)[kMB][kNB]) {
  acc[mb][nb] = kTrans ? __builtin_amdgcn_mfma_i32_32x32x32_i8(op.w[ks & 1][nb], op.a[ks & 1][mb],
                                                               acc[mb][nb], 0, 0, 0)
                       : __builtin_amdgcn_mfma_i32_32x32x32_i8(op.a[ks & 1][mb], op.w[ks & 1][nb],
                                                               acc[mb][nb], 0, 0, 0);
}
template <bool kTrans, int kMB, int kNB>
__device__ __forceinline__ void mma(const Operands<kMB, kNB>& op, int ks, v16i (&acc)[kMB][kNB]) {
#pragma unroll
  for (int mb = 0; mb < kMB; ++mb)
#pragma unroll
    for (int nb = 0; nb < kNB; ++nb)
      mma_one<kTrans>(op, ks, mb, nb, acc);
}

template <bool kTrans, int kMB, int kNB, int kRing>
__device__ __forceinline__ void tile(const Args& a, uint32_t m0, uint32_t n0, char* s0, char* s1,
                                     char* s2, char* s3) {
  using T = Tile<kMB, kNB>;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave_m = wave >> 2, wave_n = wave & 3;
  const uint32_t half = lane >> 5;
  const uint32_t arow = wave_m * 32 * kMB + (lane & 31);  // A row of block 0 (stage row)
  const uint32_t wrow = wave_n * 32 * kNB + (lane & 31);  // W row of block 0 (stage row - kBM)
  const uint32_t sw = (lane >> 1) & 7;                    // (row/2)%8, the same for every block

  // DMA map: load t of wave w fills stage bytes [(kLoads w + t) * 1024, + 1024), eight rows of A or
  // of W; lane l writes row r = (kLoads w + t) * 8 + l/8, position l%8, which holds logical chunk
  // (l%8) ^ ((r/2)%8).
  const uint32_t a_left = min(a.m - m0, (uint32_t)T::kBM);
  const uint32_t w_left = a.n > n0 ? min(a.n - n0, (uint32_t)T::kBN) : 0u;
  const int8_t* a_base = a.a + (size_t)m0 * a.k_stride;
  const int8_t* w_base = a.w + (size_t)n0 * a.k_stride;
  const uint32_t a_bytes = a_left * a.k_stride, w_bytes = w_left * a.k_stride;
  auto is_a = [&](int t) { return (T::kLoads * wave + t) * 8 < (uint32_t)T::kBM; };
  uint32_t voff[T::kLoads];
#pragma unroll
  for (int t = 0; t < T::kLoads; ++t) {
    const uint32_t r = (T::kLoads * wave + t) * 8 + (lane >> 3);
    const uint32_t row = is_a(t) ? r : r - T::kBM;
    voff[t] = row * a.k_stride + 16 * ((lane & 7) ^ ((r >> 1) & 7));
  }
  // A wave's loads are all of A or all of W (kSame), or, with 64-row tiles, of either.
  // Step at K byte k0: the descriptors start at k0 and end at the last valid row's end, so rows
  // past the tile's valid ones read zero and nothing past the operand is addressed. In a final
  // 64-byte step the lanes of logical chunks 4..7 (bytes k0+64..k0+127, past K) are sent out of
  // range and write zeros.
  constexpr bool kSame = (T::kBM / 8) % T::kLoads == 0;
  struct Loads {
    __amdgpu_buffer_rsrc_t a, w;  // kSame: a is the wave's own, w is not used
    bool half_step;
  };
  const int8_t* own_base = is_a(0) ? a_base : w_base;
  const uint32_t own_bytes = is_a(0) ? a_bytes : w_bytes;
  const uint32_t steps = (a.k + kBK - 1) / kBK;
  const bool tail = a.k % kBK != 0;
  auto loads_of = [&](uint32_t i) {  // step i; past the last step the descriptors are empty
    const uint32_t k0 = i * kBK;
    const int8_t* base = kSame ? own_base : a_base;
    const uint32_t bytes = kSame ? own_bytes : a_bytes;
    Loads l;
    l.a = rsrc(base + k0, i < steps && bytes > k0 ? bytes - k0 : 0u);
    l.w = kSame ? l.a : rsrc(w_base + k0, i < steps && w_bytes > k0 ? w_bytes - k0 : 0u);
    l.half_step = tail && i + 1 == steps;
    return l;
  };
  auto load = [&](const Loads& l, char* st, int t) __attribute__((always_inline)) {
    const uint32_t piece = T::kLoads * wave + t, r = piece * 8 + (lane >> 3);
    const bool past_k = l.half_step && (((lane & 7) ^ ((r >> 1) & 7)) >= 4);
    const uint32_t off = past_k ? 0x80000000u : voff[t];
    const __amdgpu_buffer_rsrc_t from = kSame || is_a(t) ? l.a : l.w;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(from, (lds_void*)(st + piece * 1024), 16, off, 0, 0, 0);
  };
  auto stage = [&](char* st, uint32_t i) __attribute__((always_inline)) {
    const Loads l = loads_of(i);
#pragma unroll
    for (int t = 0; t < T::kLoads; ++t) load(l, st, t);
  };

  v16i acc[kMB][kNB];
#pragma unroll
  for (int mb = 0; mb < kMB; ++mb)
#pragma unroll
    for (int nb = 0; nb < kNB; ++nb)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[mb][nb][r] = 0;

  // K steps of 128 bytes; K is a multiple of 64, so the last step may hold only 64 bytes (its
  // other half loads as zero). Step i sits in ring stage i % kRing and is consumed in four substeps
  // of 32 bytes, each reading the next one's operands ahead of its MFMAs. A step's one barrier stands
  // before its last substep's MFMAs: by then every operand of the step has been read and the next
  // step's loads have landed, so right behind it the loads of step i + kRing go into the stage just
  // read, the next step's first operands are read, and both run under the last substep's MFMAs.
  // vmcnt: the loads of the steps after the next one (or, ahead of step 0, after it) stay in flight.
  constexpr int kWaitNext = kWaitAll | ((kRing - 2) * T::kLoads);
  constexpr int kWaitFirst = kWaitAll | ((kRing - 1) * T::kLoads);
  static_assert((kRing - 1) * T::kLoads < 16, "the vmcnt field's low four bits hold the count");
  Operands<kMB, kNB> op;
  auto step = [&](char* cur, const char* nxt, uint32_t i) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < 3; ++ks) {
      read_operands(op, cur, ks + 1, arow, wrow, half, sw);
      __builtin_amdgcn_sched_barrier(0);  // the next substep's reads go out before these MFMAs
      mma<kTrans>(op, ks, acc);
    }
    __builtin_amdgcn_s_waitcnt(kWaitNext);  // step i + 1's loads; the later ones stay in flight
    asm volatile("s_barrier" ::: "memory");
    read_operands(op, nxt, 0, arow, wrow, half, sw);  // after the last step: unused
    const Loads l = loads_of(i + kRing);
    __builtin_amdgcn_sched_barrier(0);
    // The loads of step i + kRing, two behind each of the first MFMAs: a wave takes about 65 cycles to
    // issue one, which in a burst ahead of the MFMAs left the matrix cores idle (256 x 256 tiles: 1,543
    // -> 1,521 us at 31,104 tokens, 6,447 -> 6,343 at 129,024, with the barrier moved; one behind each
    // of the eight leaves the last ones less time to land, 2 % slower where the operands come from
    // HBM). Smaller tiles have fewer MFMAs than loads and run 2 % better with the burst.
    if constexpr (kMB * kNB >= T::kLoads) {
#pragma unroll
      for (int x = 0; x < kMB * kNB; ++x) {
        mma_one<kTrans>(op, 3, x / kNB, x % kNB, acc);
#pragma unroll
        for (int t = 2 * x; t < 2 * x + 2 && t < T::kLoads; ++t) load(l, cur, t);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma unroll
      for (int t = 0; t < T::kLoads; ++t) load(l, cur, t);
      __builtin_amdgcn_sched_barrier(0);
      mma<kTrans>(op, 3, acc);
    }
  };
  if (steps > 0) {
    stage(s0, 0);
    stage(s1, 1);
    if (kRing == 4) {
      stage(s2, 2);
      stage(s3, 3);
    }
    __builtin_amdgcn_s_waitcnt(kWaitFirst);
    asm volatile("s_barrier" ::: "memory");
    read_operands(op, s0, 0, arow, wrow, half, sw);
    uint32_t i = 0;
    if constexpr (kRing == 2) {
#pragma clang loop unroll(disable)
      for (; i + 1 < steps; i += 2) {
        step(s0, s1, i);
        step(s1, s0, i + 1);
      }
      if (i < steps) step(s0, s1, i);
    } else {
#pragma clang loop unroll(disable)
      for (; i + 3 < steps; i += 4) {
        step(s0, s1, i);
        step(s1, s2, i + 1);
        step(s2, s3, i + 2);
        step(s3, s0, i + 3);
      }
      if (i < steps) step(s0, s1, i);
      if (i + 1 < steps) step(s1, s2, i + 1);
      if (i + 2 < steps) step(s2, s3, i + 2);
    }
    __builtin_amdgcn_s_waitcnt(kWaitAll);  // no load into LDS outlives the workgroup
  }

  if (kTrans) {
    // Q/K tile: block (mb, nb) holds C^T: lane column = token, registers 4g+i = channels
    // 8g + 4*half + i of the block.
#pragma unroll
    for (int mb = 0; mb < kMB; ++mb) {
      const uint32_t m = m0 + arow + 32 * mb;
      if (m >= a.m) continue;
      const float asv = a.as[m];
      uint16_t* dst = a.out + (size_t)m * a.qk_width;
#pragma unroll
      for (int nb = 0; nb < kNB; ++nb) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const uint32_t n = n0 + wave_n * 32 * kNB + 32 * nb + 8 * g + 4 * half;
          v4h o;
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i] = finish(acc[mb][nb][4 * g + i], a.ws[n + i], asv);
          *reinterpret_cast<v4h*>(dst + n) = o;
        }
      }
    }
  } else {
    // V tile: block (mb, nb) holds C: lane column = channel, registers 4g+i = tokens
    // 8g + 4*half + i of the block; tokens >= M are stored as zero up to the capacity.
    uint16_t* vt = a.out + (size_t)a.m * a.qk_width;
#pragma unroll
    for (int nb = 0; nb < kNB; ++nb) {
      const uint32_t n = n0 + wave_n * 32 * kNB + 32 * nb + (lane & 31);
      if (n >= a.n) continue;
      const float wsv = a.ws[n];
      uint16_t* dst = vt + (size_t)(n - a.qk_width) * a.cap;
#pragma unroll
      for (int mb = 0; mb < kMB; ++mb) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const uint32_t m = m0 + wave_m * 32 * kMB + 32 * mb + 8 * g + 4 * half;
          v4h o;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const uint32_t mi = m + i;
            const float asv = a.as[mi < a.m ? mi : a.m - 1];
            o[i] = mi < a.m ? finish(acc[mb][nb][4 * g + i], wsv, asv) : (_Float16)0.0f;
          }
          *reinterpret_cast<v4h*>(dst + m) = o;
        }
      }
    }
    // The last tile of tokens also writes the zeros up to the capacity. Tiles of their own for them
    // took slots from the others: 513 tokens x 12,288 are 480 tiles of 128 x 128, which fit two to a
    // CU, and 96 more did not (K 4,096: 62.7 us with them, 40.5 so).
    if (m0 + T::kBM >= a.m) {
      const uint32_t first = m0 + T::kBM, per = (a.cap - first) / 4;
      for (uint32_t i = threadIdx.x; i < T::kBN * per; i += kThreads) {
        const uint32_t n = n0 + i / per;
        if (n < a.n)
          *reinterpret_cast<v4h*>(vt + (size_t)(n - a.qk_width) * a.cap + first + 4 * (i % per)) = v4h{};
      }
    }
  }
}

template <int kMB, int kNB, int kRing>
__global__ __launch_bounds__(kThreads) void k_gemm_i8_qkv(Args a) {
  using T = Tile<kMB, kNB>;
  __shared__ __attribute__((aligned(16))) char s0[T::kStage];
  __shared__ __attribute__((aligned(16))) char s1[T::kStage];
  __shared__ __attribute__((aligned(16))) char s2[kRing == 4 ? T::kStage : 16];
  __shared__ __attribute__((aligned(16))) char s3[kRing == 4 ? T::kStage : 16];
  // XCD-aware remap (block b runs on XCD b % 8): each XCD takes a contiguous range of the
  // rasterised tiles, so the tiles resident on one XCD share A and W rows in its L2.
  const uint32_t b = blockIdx.x;
  const uint32_t w = (b & 7u) * a.per_xcd + (b >> 3);
  if (w >= a.total) return;
  const uint32_t span = kGroupM * a.tiles_n;
  const uint32_t gm = w / span, r = w % span;
  const uint32_t m_in = min((uint32_t)kGroupM, a.tiles_m - gm * kGroupM);
  const uint32_t m_tile = gm * kGroupM + r % m_in;
  const uint32_t n_tile = r / m_in;
  const uint32_t m0 = m_tile * T::kBM;
  if (n_tile < a.tiles_n_qk) {
    tile<true, kMB, kNB, kRing>(a, m0, n_tile * T::kBN, s0, s1, s2, s3);
  } else {
    tile<false, kMB, kNB, kRing>(a, m0, a.qk_width + (n_tile - a.tiles_n_qk) * T::kBN, s0, s1, s2,
                                 s3);
  }
}

template <int kMB, int kNB, int kRing>
hipError_t launch_tiles(Args g, hipStream_t stream) {
  using T = Tile<kMB, kNB>;
  g.tiles_m = (g.m + T::kBM - 1) / T::kBM;
  g.tiles_n_qk = (g.qk_width + T::kBN - 1) / T::kBN;
  g.tiles_n = g.tiles_n_qk + (g.n - g.qk_width + T::kBN - 1) / T::kBN;
  g.total = g.tiles_m * g.tiles_n;
  g.per_xcd = (g.total + 7) / 8;
  hipLaunchKernelGGL((k_gemm_i8_qkv<kMB, kNB, kRing>), dim3(g.per_xcd * 8), dim3(kThreads), 0, stream, g);
  return hipGetLastError();
}

// Up to 32 tokens: the projection is bound by reading W (10 us at K = 4,096, N = 12,288), and a tile
// walks the whole K on one CU. Here a workgroup takes 32 channels, its eight waves every eighth
// 128-byte piece of K each, operands loaded straight into registers, and the eight partial products
// are added through LDS (int32: exact in any order). One token: 14.4 us against 21.6 on 64 x 128
// tiles and 46 on 256 x 256; at 64 tokens two such workgroups per channel block are already slower
// than the tiles (26.5 against 25 us).
constexpr int kRedRow = 32 + 4;  // ints per token of a partial product (token rows 4 banks apart)
__global__ __launch_bounds__(kThreads) void k_gemm_i8_qkv_few(Args a) {
  __shared__ __attribute__((aligned(16))) int red[kWaves][32][kRedRow];
  const uint32_t w = (blockIdx.x & 7u) * a.per_xcd + (blockIdx.x >> 3);
  if (w >= a.total) return;  // the whole workgroup
  const uint32_t n0 = w * 32;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t lane = threadIdx.x & 63, row = lane & 31, half = lane >> 5;
  // the descriptors end with the last valid row: tokens past M read as zero
  const __amdgpu_buffer_rsrc_t ra = rsrc(a.a, a.m * a.k_stride);
  const __amdgpu_buffer_rsrc_t rw = rsrc(a.w + (size_t)n0 * a.k_stride, 32 * a.k_stride);
  const uint32_t off = row * a.k_stride + 16 * half;
  v16i acc = {};
  auto load = [](__amdgpu_buffer_rsrc_t from, uint32_t at) {
    return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(from, at, 0, 0));
  };
  const uint32_t halves = a.k / 64;  // K is a multiple of 64: the last piece may be half of one
  for (uint32_t k0 = wave * kBK; k0 < a.k; k0 += kWaves * kBK) {
    const int parts = k0 / 64 + 1 < halves ? 4 : 2;  // 32-byte parts of the piece
    v4i wf[4], af[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const uint32_t at = p < parts ? off + k0 + 32 * p : 0x80000000u;  // past K: reads zero
      wf[p] = load(rw, at);
      af[p] = load(ra, at);
    }
#pragma unroll
    for (int p = 0; p < 4; ++p)
      acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(wf[p], af[p], acc, 0, 0, 0);
  }
  // lane column = token, registers 4g + i = channels 8g + 4 half + i
#pragma unroll
  for (int g = 0; g < 4; ++g)
    *reinterpret_cast<v4i*>(&red[wave][row][8 * g + 4 * half]) =
        v4i{acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]};
  __syncthreads();
  if (n0 < a.qk_width) {  // Q/K: four channels of a token
    const uint32_t m = threadIdx.x >> 3, c = 4 * (threadIdx.x & 7);
    if (m >= a.m) return;  // threads 256.. and tokens past M
    v4i sum = *reinterpret_cast<const v4i*>(&red[0][m][c]);
#pragma unroll
    for (int x = 1; x < kWaves; ++x) sum += *reinterpret_cast<const v4i*>(&red[x][m][c]);
    const float asv = a.as[m];
    v4h o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = finish(sum[e], a.ws[n0 + c + e], asv);
    *reinterpret_cast<v4h*>(a.out + (size_t)m * a.qk_width + n0 + c) = o;
  } else {  // V: four tokens of a channel, zeros past M up to the capacity
    uint16_t* vt = a.out + (size_t)a.m * a.qk_width + (size_t)(n0 - a.qk_width) * a.cap;
    const uint32_t per = a.cap / 4;
    for (uint32_t i = threadIdx.x; i < 32 * per; i += kThreads) {
      const uint32_t c = i / per, m = 4 * (i % per);
      v4h o = {};
      if (m < a.m) {
        const float wsv = a.ws[n0 + c];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (m + e >= a.m) break;
          int sum = 0;
#pragma unroll
          for (int x = 0; x < kWaves; ++x) sum += red[x][m + e][c];
          o[e] = finish(sum, wsv, a.as[m + e]);
        }
      }
      *reinterpret_cast<v4h*>(vt + (size_t)c * a.cap + m) = o;
    }
  }
}

hipError_t launch_few(Args g, hipStream_t stream) {
  g.total = g.n / 32;
  g.per_xcd = (g.total + 7) / 8;
  hipLaunchKernelGGL(k_gemm_i8_qkv_few, dim3(g.per_xcd * 8), dim3(kThreads), 0, stream, g);
  return hipGetLastError();
}

}  // namespace

// The tiling that prices lowest, in us, s steps of 128 bytes of K: fixed costs, what a tile costs besides its
// steps (its fill and its epilogue, which nothing overlaps at one 256 x 256 tile per CU), and its steps.
// n0, n1: 256 x 256 and 128 x 128 tiles per CU. 256 x 256 run one to a CU, in rounds; 128 x 128 on a ring
// of two stages two to a CU; on a ring of four one, its loads four steps ahead. 64 x 128 where the others
// leave three CUs of four idle. Past one round of 256 x 256 a smaller tile has to be 2 % cheaper, and 12 %
// where A, W and the output are more than 200 MiB: it reads A and W more often, from HBM then, where the
// 256 MB behind the L2s no longer holds what the launch touches. Fitted to 64 to 8,192 tokens at seven
// (N, K); checked behind the quantizer with W from four buffers on 1,700 shapes of 33 to 64,000 tokens, 1 to
// 56 heads, K 128 to 7,680: 3.7 % over the best tile in the mean, nearly all of it small calls that 64 x 128
// would suit; 11 of them slower than on 256 x 256 by more than 1 %, by 6.7 % at most (without the rule for
// 200 MiB 68, by 17 %). us on 256 x 256 / 128 x 128 ring 2 / ring 4, K 4,096, N 12,288: 129 tokens 57 / 29 /
// 22, 513 64 / 41 / 44, 1,025 76 / 73 / 77, 5,000 246 / 279 / 298; 2,049 of K 1,024, N 21,504 113 / 87 / 108;
// 641 of K 7,168, N 21,504 110 / 120 / 124; 34,453 of K 1,984, N 5,760 520 / 611 / 662.
GemmTiling gemm_tiling(uint32_t m, uint32_t n, uint32_t k, uint32_t compute_units) {
  if (m <= 32) return GemmTiling::kFew;
  const float cus = compute_units, s = k / 128.0f;
  auto tiles = [&](uint32_t bm, uint32_t bn) {
    const uint32_t qk_width = n / 3 * 2;
    const uint32_t qk = (qk_width + bn - 1) / bn, v = (n - qk_width + bn - 1) / bn;
    return (m + bm - 1) / bm * (qk + v) / cus;
  };
  if (tiles(64, 128) <= 0.25f) return GemmTiling::k64x128;
  const float n0 = tiles(256, 256), n1 = tiles(128, 128);
  const float rounds = n0 <= 3.0f ? 0.84f * std::ceil(n0) + 0.16f * n0 : n0 + 0.2f;
  const float t0 = n0 <= 1.0f ? 28.75f + s * (0.89f + 0.61f * n0)
                              : 8.91f + rounds * (19.84f + 1.43f * s);
  const float t2 = 7.01f + 3.43f * n1 +
                   s * (n1 <= 2.0f   ? 0.64f + 0.29f * std::max(n1 - 1.0f, 0.0f)
                        : n1 <= 4.0f ? 1.48f + 0.18f * (n1 - 2.0f)
                                     : 0.21f + 0.475f * n1);
  const float t4 = 7.6f + 4.95f * n1 +
                   s * (n1 <= 1.0f   ? 0.35f
                        : n1 <= 2.0f ? 0.85f
                        : n1 <= 4.0f ? 1.17f + 0.36f * (n1 - 2.0f)
                                     : 0.1f + 0.475f * n1);
  const bool large = (float)m * k + (float)n * k + 2.0f * m * n >= 200.0f * 1048576.0f;
  if (std::min(t2, t4) > (large ? 0.88f : n0 > 1.0f ? 0.98f : 1.0f) * t0) return GemmTiling::k256x256;
  return t2 <= t4 ? GemmTiling::k128x128Ring2 : GemmTiling::k128x128Ring4;
}

hipError_t launch_gemm_i8_qkv(uint32_t m, uint32_t n, uint32_t k, uint32_t k_stride,
                              const int8_t* a, const int8_t* w, const float* ws, const float* as,
                              uint16_t* out, hipStream_t stream) {
  Args g;
  g.a = a;
  g.w = w;
  g.ws = ws;
  g.as = as;
  g.out = out;
  g.m = m;
  g.n = n;
  g.k = k;
  g.k_stride = k_stride;
  g.qk_width = n / 3 * 2;
  g.cap = (m + kCapRows - 1) / kCapRows * kCapRows;
  switch (gemm_tiling(m, n, k, device_cus())) {
    case GemmTiling::kFew: return launch_few(g, stream);
    case GemmTiling::k64x128: return launch_tiles<1, 1, 4>(g, stream);
    case GemmTiling::k128x128Ring4: return launch_tiles<2, 1, 4>(g, stream);
    case GemmTiling::k128x128Ring2: return launch_tiles<2, 1, 2>(g, stream);
    default: return launch_tiles<4, 2, 2>(g, stream);
  }
}

}  // namespace h3
