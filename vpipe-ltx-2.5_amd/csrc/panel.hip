// The linear between the M <= 128 kernel and the 256 x 256 tile on gfx950:
// y = x . W^T (+ bias) (+ GELU) (+ y_in), W group-affine codes (w8 / w4) or
// dense bf16, for shapes whose output holds too few large tiles to fill the
// CUs.
//
// A workgroup owns R x C = 32 RB x 32 CB outputs and a whole run of K. Its
// four waves split that run into contiguous ranges of 64-wide chunks; each
// wave computes all R x C outputs over its own range and the four partial
// tiles are summed once through LDS, in wave order. So the CUs are filled without
// split-K partials in memory or a second launch, and the K loop has no
// barrier: each wave feeds itself.
//
//   - Every operand goes straight from global memory into the wave's own LDS
//     (buffer_load ... lds, 16 bytes per lane) through a ring of NS slots of
//     4 KB: a slot holds 32 rows x 64 of X, or a chunk's codes of all C
//     columns (a dense weight: one slot per 32 columns). The slot that a unit
//     leaves is refilled at once with the unit NS places ahead, so 20 to
//     30 KB per wave stay in flight. Units past the
//     wave's range are loaded through an empty buffer range (zeros, no
//     traffic): the loop has no branch and every wait is a constant.
//   - Fragments are read one unit ahead of the MFMAs that take them; the next
//     chunk's codes are dequantized, w = bf16(fma(scale, q, zero point)), and
//     the slots refilled in the gaps between the current chunk's MFMAs.
//   - Scales and zero points arrive as 16-byte windows of eight groups of
//     one column (at whatever 2-byte offset the column's row starts), four
//     windows deep: one instruction per eight groups and 64 columns. Loaded two
//     bytes at a time they cost one cache line per column and chunk.
//
// What bounds it: the L2 -> LDS stream of a workgroup's operands, K (2 R + C
// bits / 8) bytes at 70 to 125 GB/s per CU (0.84 us per 80 KB round of chunks at
// 128 x 64 w8, where the MFMAs alone take 0.46 and everything but the loads
// 0.63), and 4 to 7 us of launch, first loads and the final sum.
//
// Reference semantics: MetalOps::linear(QWeight) (src/ltx25-metal-ops.cc:
// 531-569), both of its routes.
#include "common.h"

#include <type_traits>
#include <utility>

namespace ltx25 {
namespace {

constexpr int kChunk = 64;            // K per chunk
constexpr int kWaves = 4;             // per workgroup, one per SIMD
constexpr int kThreads = kWaves * 64;
constexpr int kSlot = 4096;           // bytes per ring slot
constexpr int kLdsBytes = 160 * 1024;
constexpr int kWindows = 4;           // scale windows of 8 groups in LDS
constexpr uint32_t kOob = 0x80000000u;

typedef uint32_t __attribute__((address_space(3))) lds_u32;

struct PanelParams {
  const void* x;            // bf16 [M][K]
  const void* w;            // codes [N][K * bits / 8], or bf16 [wn][K]
  const void* scales;       // aligned down to 16 bytes
  const void* qbias;        // aligned down to 16 bytes
  int s_mis, q_mis;         // elements from those addresses to the first scale / zero point
  const void* bias;
  const uint16_t* y_in;
  uint16_t* y;
  float* partial;           // [splits][M][N] when split
  int M, N, K, wn;
  int gshift, gcols;
  int k_chunk;              // K per workgroup (multiple of 64)
  int bias_type, epilogue;
  int tiles_m, tiles_n, splits;
  int by_m;                 // 1: an XCD takes whole rows of tiles, 0: whole columns
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* p, size_t bytes)
{
  // loads at offsets past `bytes` return zeros
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)(uint32_t)bytes,
                                           0x00020000);
}

template <typename F, int... I>
__device__ __forceinline__ void unroll_seq(F&& f, std::integer_sequence<int, I...>)
{
  (f(std::integral_constant<int, I>{}), ...);
}

template <int N, typename F>
__device__ __forceinline__ void unroll(F&& f)
{
  unroll_seq(f, std::make_integer_sequence<int, N>{});
}

// s_waitcnt vmcnt(N), the other counters left alone
template <int N>
__device__ __forceinline__ void wait_vm()
{
  static_assert(N >= 0 && N < 64, "vmcnt has six bits");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <int BITS, int RB, int CB>
struct Panel {
  static constexpr bool kQuant = BITS != 16;
  static constexpr int kR = 32 * RB;
  static constexpr int kC = 32 * CB;
  static constexpr int kWLoads = BITS == 16 ? 4 * CB : BITS == 8 ? 2 * CB : CB;  // 1 KB loads
  static constexpr int kWSlots = BITS == 16 ? CB : 1;
  static constexpr int kUnits = kWSlots + RB;                    // slots per chunk
  static constexpr int kWinBytes = kC * 16;                      // one window, one array
  static constexpr int kWinAll = kQuant ? 2 * kWindows * kWinBytes : 0;
  static constexpr int kWaveLds = kLdsBytes / kWaves;
  static constexpr int kSlots = (kWaveLds - kWinAll) / kSlot;
  static_assert(kWLoads * 1024 <= kWSlots * kSlot, "the codes fit their slots");
  static_assert(kR * kC * 4 <= kSlots * kSlot, "a partial tile fits the ring");
  // The stream of units: chunk by chunk, the weight and then X(t, 0 .. RB - 1).
  // Codes run a chunk ahead, W(0), then W(t + 1) before X(t, ..), to be
  // dequantized under the MFMAs of the chunk before theirs; a dense weight's
  // fragments are read as they are, W(t) before X(t, ..).
  static constexpr int kAhead = kQuant ? 1 : 0;
  static constexpr int kPre = kQuant ? kWSlots : 0;              // units before chunk 0's part
  static constexpr int loads_at(int pos)
  {
    if (pos < kPre) { return kWLoads / kWSlots; }
    return (pos - kPre) % kUnits < kWSlots ? kWLoads / kWSlots : 4;
  }
  // loads of the units at places a .. b - 1 of a chunk's part of the stream, and
  // the place of the unit that load l of those from place a on belongs to
  static constexpr int loads_upto(int a, int b)
  {
    int n = 0;
    for (int q = a; q < b; ++q) { n += loads_at(kPre + q); }
    return n;
  }
  static constexpr int unit_of(int a, int l)
  {
    int q = a;
    while (loads_upto(a, q + 1) <= l) { ++q; }
    return q;
  }
  // loads issued after the unit at `pos`: those of the kSlots - 1 units behind
  // it, less `held`, the units read before it whose slots wait for their refill
  static constexpr int later(int pos, int held)
  {
    int n = 0;
    for (int d = 1; d < kSlots - held; ++d) { n += loads_at(pos + d); }
    return n;
  }
};

template <int BITS, int RB, int CB, bool SPLIT>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
panel_kernel(PanelParams p)
{
  using P = Panel<BITS, RB, CB>;
  constexpr bool QUANT = P::kQuant;
  constexpr int R = P::kR;
  constexpr int C = P::kC;
  constexpr int NS = P::kSlots;
  constexpr int U = P::kUnits;
  constexpr int WS = P::kWSlots;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kLdsBytes];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int h = lane >> 5;
  const int l32 = lane & 31;
  uint8_t* const ring = lds + wave * P::kWaveLds;
  uint8_t* const win = ring + NS * kSlot;   // [scales, zero points][window % 4][column]

  // Workgroup ids are dealt round-robin to the 8 XCDs: each gets a contiguous
  // range of (outer tile, split, inner tile), so the workgroups that share the
  // larger operand's rows or columns meet in one L2.
  int tm, tn, split;
  {
    const int total = (int)gridDim.x;
    const int total8 = total & ~7;
    const int b = (int)blockIdx.x;
    const int pid = b < total8 ? (b & 7) * (total8 >> 3) + (b >> 3) : b;
    const int inner = p.by_m ? p.tiles_n : p.tiles_m;
    const int i = pid % inner;
    const int os = pid / inner;
    split = SPLIT ? os % p.splits : 0;
    const int o = SPLIT ? os / p.splits : os;
    tm = p.by_m ? o : i;
    tn = p.by_m ? i : o;
  }
  const int m0 = tm * R;
  const int n0 = tn * C;
  const int kbeg = split * p.k_chunk;
  const int nch = (min(p.K, kbeg + p.k_chunk) - kbeg) / kChunk;
  const int c_lo = nch * wave / kWaves;
  const int cnt = nch * (wave + 1) / kWaves - c_lo;   // this wave's chunks
  const int kw0 = kbeg + c_lo * kChunk;

  const uint32_t wrow = (uint32_t)((size_t)p.K * BITS / 8);
  const __amdgpu_buffer_rsrc_t none = rsrc(p.x, 0);
  const __amdgpu_buffer_rsrc_t xr = rsrc(p.x, (size_t)p.M * p.K * 2);
  const __amdgpu_buffer_rsrc_t wr = rsrc(p.w, (size_t)p.wn * wrow);

  // ---- loads. An X slot is 32 rows of 128 bytes; load j covers rows 8 j .. 8 j +
  // 7, lane l lands at byte 16 l of it and fetches the row's 16-byte piece
  // (l % 8) ^ ((row / 2) % 8): the fragment reads below are then free of bank
  // conflicts. A dense weight's slots are the same with columns for rows.
  // Codes are C rows of 64 (w8) or 32 (w4) bytes, pieces XORed by (row / 4) % 4
  // or (row / 8) % 2.
  uint32_t xoff[4 * RB];
#pragma unroll
  for (int j = 0; j < 4 * RB; ++j) {
    const int r = 8 * j + (lane >> 3);
    xoff[j] = (uint32_t)(m0 + r) * (uint32_t)(p.K * 2) + (((lane & 7) ^ ((r >> 1) & 7)) * 16);
  }
  uint32_t woff[P::kWLoads];
#pragma unroll
  for (int j = 0; j < P::kWLoads; ++j) {
    if constexpr (BITS == 16) {
      const int r = 8 * j + (lane >> 3);
      woff[j] = (uint32_t)(n0 + r) * wrow + (((lane & 7) ^ ((r >> 1) & 7)) * 16);
    } else if constexpr (BITS == 8) {
      const int r = 16 * j + (lane >> 2);
      woff[j] = (uint32_t)(n0 + r) * wrow + (((lane & 3) ^ ((r >> 2) & 3)) * 16);
    } else {
      const int r = 32 * j + (lane >> 1);
      woff[j] = (uint32_t)(n0 + r) * wrow + (((lane & 1) ^ ((r >> 3) & 1)) * 16);
    }
  }
  auto dma = [&](__amdgpu_buffer_rsrc_t r, uint8_t* dst, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_u32*)dst, 16, (int)voff, (int)soff, 0, 0);
  };
  // load k of the unit q places after the start of chunk t's part of the stream
  auto load_one = [&](int t, auto q, auto k, uint8_t* dst) {
    constexpr int Q = decltype(q)::value;
    constexpr int L = decltype(k)::value;
    constexpr int pos = Q % U;
    if constexpr (pos < WS) {
      const int c = t + Q / U + P::kAhead;
      dma(c < cnt ? wr : none, dst + L * 1024, woff[P::kWLoads / WS * pos + L],
          (uint32_t)(kw0 + c * kChunk) * BITS / 8);
    } else {
      const int c = t + Q / U;
      dma(c < cnt ? xr : none, dst + L * 1024, xoff[4 * (pos - WS) + L],
          (uint32_t)(kw0 + c * kChunk) * 2u);
    }
  };
  auto load_at = [&](int t, auto q, uint8_t* dst) {
    unroll<P::loads_at(P::kPre + decltype(q)::value)>([&](auto k) { load_one(t, q, k, dst); });
  };

  // ---- scale windows. Column c's scales of this wave start at element
  // c * gcols + first group; window w holds elements 8 (that / 8) + 8 w .. + 7.
  // One load covers a window of 64 columns, or two windows of 32.
  const __amdgpu_buffer_rsrc_t sr =
      rsrc(p.scales, QUANT ? (((size_t)p.N * p.gcols + p.s_mis) * 2 + 3) & ~(size_t)3 : 0);
  const __amdgpu_buffer_rsrc_t qr =
      rsrc(p.qbias, QUANT ? (((size_t)p.N * p.gcols + p.q_mis) * 2 + 3) & ~(size_t)3 : 0);
  uint32_t soff0 = kOob, qoff0 = kOob;
  if constexpr (QUANT) {
    const int n = n0 + (CB == 2 ? lane : l32);
    const uint32_t e = (uint32_t)n * (uint32_t)p.gcols + (uint32_t)(kw0 >> p.gshift);
    if (n < p.N) {
      soff0 = ((e + p.s_mis) >> 3) * 16u + (CB == 1 ? h * 16u : 0u);
      qoff0 = ((e + p.q_mis) >> 3) * 16u + (CB == 1 ? h * 16u : 0u);
    }
  }
  constexpr int kWinStep = CB == 2 ? 1 : 2;   // windows per load
  auto load_win = [&](int w) {
    if constexpr (QUANT) {
      uint8_t* const dst = win + (w % kWindows) * P::kWinBytes;
      dma(sr, dst, soff0 + 16u * w, 0);
      dma(qr, dst + kWindows * P::kWinBytes, qoff0 + 16u * w, 0);
    }
  };
  // byte offset of chunk 0's scale in the windows' sequence, per 32-column
  // block: twice the element's place in its window, the lane's K half counted
  uint32_t sph[CB], qph[CB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    const uint32_t e = (uint32_t)(n0 + 32 * cb + l32) * (uint32_t)p.gcols +
                       (uint32_t)(kw0 >> p.gshift);
    const uint32_t hg = p.gshift == 5 ? h : 0;   // groups of 32: two per chunk
    sph[cb] = (((e + p.s_mis) & 7u) + hg) * 2u;
    qph[cb] = (((e + p.q_mis) & 7u) + hg) * 2u;
  }
  const int gpc = p.gshift == 5 ? 2 : 1;         // groups per chunk

  // ---- fragments: unit row l32, 16-byte piece 4 h + s at (4 h + s) ^ ((l32 / 2) % 8)
  int fo[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) { fo[s] = l32 * 128 + (((4 * h + s) ^ ((l32 >> 1) & 7)) * 16); }
  constexpr int kCw = BITS == 16 ? 4 : BITS == 8 ? 2 : 1;   // 16-byte pieces per lane and block
  i32x4 cw[2][CB][kCw];       // codes (or dense fragments) of a chunk, by its parity
  uint32_t sv[2][CB], qv[2][CB];
  i32x4 wq[2][CB][4];         // dequantized fragments (dense: cw itself)
  bf16x8 xf[2][4];
  auto read_x = [&](auto b, const uint8_t* src) {
#pragma unroll
    for (int s = 0; s < 4; ++s) { xf[decltype(b)::value][s] = *(const bf16x8*)(src + fo[s]); }
  };
  auto read_w = [&](auto par, auto s, const uint8_t* src) {
    constexpr int B = decltype(par)::value;
    if constexpr (BITS == 16) {
#pragma unroll
      for (int k = 0; k < 4; ++k) { cw[B][decltype(s)::value][k] = *(const i32x4*)(src + fo[k]); }
    } else {
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) {
        const int r = 32 * cb + l32;
#pragma unroll
        for (int k = 0; k < kCw; ++k) {
          if constexpr (BITS == 8) {
            cw[B][cb][k] = *(const i32x4*)(src + r * 64 + (((2 * h + k) ^ ((r >> 2) & 3)) * 16));
          } else {
            cw[B][cb][k] = *(const i32x4*)(src + r * 32 + ((h ^ ((r >> 3) & 1)) * 16));
          }
        }
      }
    }
  };
  // chunk t's scales and zero points
  auto read_scales = [&](auto par, int t) {
    if constexpr (QUANT) {
      constexpr int B = decltype(par)::value;
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) {
        const uint32_t es = sph[cb] + 2u * (uint32_t)(gpc * t);
        const uint32_t eq = qph[cb] + 2u * (uint32_t)(gpc * t);
        const uint8_t* const b = win + (32 * cb + l32) * 16;
        sv[B][cb] = *(const uint16_t*)(b + ((es >> 4) & 3u) * P::kWinBytes + (es & 14u));
        qv[B][cb] = *(const uint16_t*)(b + (kWindows + ((eq >> 4) & 3u)) * P::kWinBytes +
                                       (eq & 14u));
      }
    }
  };
  // pair f of a chunk's dequantization: codes 2 (f % 4) and + 1 of fragment
  // (f / 16, f / 4 % 4)
  auto dequant2 = [&](auto par, auto f) {
    constexpr int B = decltype(par)::value;
    constexpr int cb = decltype(f)::value / 16;
    constexpr int s = decltype(f)::value / 4 % 4;
    constexpr int pr = decltype(f)::value % 4;
    const float sc = __uint_as_float(sv[B][cb] << 16);
    const float qb = __uint_as_float(qv[B][cb] << 16);
    uint32_t c0, c1;
    if constexpr (BITS == 8) {
      const uint32_t w = (uint32_t)cw[B][cb][s / 2][2 * (s & 1) + pr / 2] >> (16 * (pr & 1));
      c0 = w & 0xffu;
      c1 = (w >> 8) & 0xffu;
    } else {
      const uint32_t w = (uint32_t)cw[B][cb][0][s] >> (8 * pr);
      c0 = w & 0xfu;
      c1 = (w >> 4) & 0xfu;
    }
    uint32_t v = pack_bf16x2(fmaf(sc, (float)c0, qb), fmaf(sc, (float)c1, qb));
    asm volatile("" : "+v"(v));   // computed here, not sunk to the MFMA that takes it
    wq[B][cb][s][pr] = (int)v;
  };

  f32x16 acc[RB][CB];
#pragma unroll
  for (int i = 0; i < RB; ++i) {
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
#pragma unroll
      for (int r = 0; r < 16; ++r) { acc[i][cb][r] = 0.0f; }
    }
  }

  // ---- prologue: the first windows, the whole ring, W(0), W(1), X(0, 0)
  for (int w = 0; w < kWindows; w += kWinStep) { load_win(w); }
  unroll<NS>([&](auto j) {
    constexpr int J = decltype(j)::value;
    // before chunk 0's part, W(0): the place that part - 1 gives it
    load_at(J < P::kPre ? -1 : 0, std::integral_constant<int, J < P::kPre ? J : J - P::kPre>{},
            ring + J * kSlot);
  });
  int rp = 0;   // byte offset of the slot of the next unit to read
  int rf = 0;   // and of the next one to refill
  auto advance = [&](int& r) { r = r + kSlot == NS * kSlot ? 0 : r + kSlot; };
  auto lgkm0 = [&]() { __builtin_amdgcn_s_waitcnt(0xc07f); };   // lgkmcnt(0)
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  unroll<P::kPre>([&](auto j) {
    constexpr int J = decltype(j)::value;
    wait_vm<P::later(J, J)>();
    read_w(I0{}, j, ring + rp);
    if constexpr (J == 0) { read_scales(I0{}, 0); }
    advance(rp);
  });
  if constexpr (QUANT) {
    __builtin_amdgcn_sched_barrier(0);
    lgkm0();
    unroll<P::kPre>([&](auto j) {
      load_at(0, std::integral_constant<int, decltype(j)::value + NS - P::kPre>{}, ring + rf);
      advance(rf);
    });
    __builtin_amdgcn_sched_barrier(0);
    unroll<16 * CB>([&](auto f) { dequant2(I0{}, f); });
  }
  // issue the reads of the units at places A .. B - 1 of chunk t's part of the
  // stream; `held` units before them are read and not refilled yet
  auto read_units = [&](int t, auto par, auto a, auto b, auto xb, auto held) {
    constexpr int A = decltype(a)::value;
    unroll<decltype(b)::value - A>([&](auto d) {
      constexpr int Q = A + decltype(d)::value;
      wait_vm<P::later(P::kPre + Q, decltype(held)::value + Q - A)>();
      if constexpr (Q < WS) {
        read_w(par, std::integral_constant<int, Q>{}, ring + rp);
        if constexpr (Q == 0) { read_scales(par, t + P::kAhead); }
      } else {
        read_x(xb, ring + rp);
      }
      advance(rp);
    });
  };
  // Chunk t (parity PAR), a step per 32-row block: the next unit's reads are
  // issued, then the block's MFMAs go out one by one, and in the gap after
  // each go its shares of chunk t + 1's dequantization and of the refills of
  // the slots that the step before has read. A lone wave per SIMD has nothing
  // else to fill the matrix pipe while a load waits to be taken.
  auto chunk = [&](int t, auto par) {
    constexpr int PAR = decltype(par)::value;
    using Nxt = std::integral_constant<int, PAR ^ 1>;
    if constexpr (QUANT) {
      // Scales are read two chunks ahead, from group g on: the windows before
      // g / 8 are done with, and the next ones take their places.
      const int g = gpc * (t + 2);
      if ((g & (8 * kWinStep - 1)) == 0) { load_win((g >> 3) + kWindows - kWinStep); }
    }
    unroll<RB>([&](auto ii) {
      constexpr int i = decltype(ii)::value;
      constexpr int xb = RB == 1 ? PAR : (i & 1);
      // units to refill: part t's weight and X(t, 0) at the first step, then X(t, i)
      constexpr int q0 = i == 0 ? 0 : WS + i;
      constexpr int q1 = WS + i + 1;
      using Held = std::integral_constant<int, q1 - q0>;
      if constexpr (i + 1 < RB) {
        read_units(t, Nxt{}, std::integral_constant<int, q1>{},
                   std::integral_constant<int, q1 + 1>{}, std::integral_constant<int, xb ^ 1>{},
                   Held{});
      } else {
        // chunk t + 1's part begins: W(t + 2) (dense: W(t + 1)), then X(t + 1, 0)
        read_units(t + 1, std::integral_constant<int, QUANT ? PAR : PAR ^ 1>{}, I0{},
                   std::integral_constant<int, WS + 1>{}, std::integral_constant<int, xb ^ 1>{},
                   Held{});
      }
      __builtin_amdgcn_sched_barrier(0);
      constexpr int G = 4 * CB;                      // gaps
      constexpr int D0 = QUANT ? i * 16 * CB / RB : 0;
      constexpr int ND = QUANT ? (i + 1) * 16 * CB / RB - D0 : 0;   // pairs to dequantize
      constexpr int NL = P::loads_upto(q0 + NS, q1 + NS);           // refill loads
      unroll<G>([&](auto gg) {
        constexpr int g = decltype(gg)::value;
        constexpr int S = g / CB;
        constexpr int cb = g % CB;
        const bf16x8 w = __builtin_bit_cast(bf16x8, QUANT ? wq[PAR][cb][S] : cw[PAR][cb][S % kCw]);
        acc[i][cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w, xf[xb][S], acc[i][cb], 0, 0, 0);
        unroll<(g + 1) * NL / G - g * NL / G>([&](auto d) {
          // load l of this step's, unit by unit
          constexpr int l = g * NL / G + decltype(d)::value;
          constexpr int q = P::unit_of(q0 + NS, l);
          constexpr int k = l - P::loads_upto(q0 + NS, q);
          load_one(t, std::integral_constant<int, q>{}, std::integral_constant<int, k>{},
                   ring + rf);
          if constexpr (k + 1 == P::loads_at(P::kPre + q)) { advance(rf); }
        });
        unroll<(g + 1) * ND / G - g * ND / G>([&](auto d) {
          dequant2(Nxt{}, std::integral_constant<int, D0 + g * ND / G + decltype(d)::value>{});
        });
        __builtin_amdgcn_sched_barrier(0);
      });
      lgkm0();
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  // W(1) (dense: W(0)) and X(0, 0), then the chunks, two parities at a time
  read_units(0, std::integral_constant<int, P::kAhead>{}, I0{}, std::integral_constant<int, WS + 1>{},
             I0{}, I0{});
  __builtin_amdgcn_sched_barrier(0);
  lgkm0();
  __builtin_amdgcn_sched_barrier(0);
  int t = 0;
  for (; t + 2 <= cnt; t += 2) {
    chunk(t, I0{});
    chunk(t + 1, I1{});
  }
  if (t < cnt) { chunk(t, I0{}); }

  // ---- the partial tiles, summed through LDS in wave order. Block (i, cb),
  // registers 4 g .. 4 g + 3 of lane l: row 32 i + l % 32, columns 32 cb + 8 g +
  // 4 (l / 32) + 0..3; run (i, cb, g) of 64 lanes x 16 bytes, lanes XORed by the
  // run so that the reads of a row's runs fall in different banks.
  constexpr int kCpt = R * C / kThreads < 8 ? R * C / kThreads : 8;   // consecutive columns per item
  constexpr int kItems = R * C / kCpt / kThreads;
  constexpr int kFv = kCpt < 4 ? kCpt : 4;
  typedef float fv __attribute__((ext_vector_type(kFv)));
  // every item of a thread has the same columns: one branch on the bias type,
  // its loads at clamped columns together
  static_assert(kThreads % (C / kCpt) == 0, "a thread's items share their columns");
  const int c = tid % (C / kCpt) * kCpt;
  const int n = n0 + c;
  float bv[kCpt];
#pragma unroll
  for (int j = 0; j < kCpt; ++j) { bv[j] = 0.0f; }
  if constexpr (!SPLIT) {
    if (p.bias_type == kBiasF32) {
      const float* const bf = (const float*)p.bias;
#pragma unroll
      for (int j = 0; j < kCpt; ++j) { bv[j] = bf[min(n + j, p.N - 1)]; }
    } else if (p.bias_type == kBiasBf16) {
      const uint16_t* const bh = (const uint16_t*)p.bias;
#pragma unroll
      for (int j = 0; j < kCpt; ++j) { bv[j] = bf16_to_f32(bh[min(n + j, p.N - 1)]); }
    }
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");   // the ring's last loads landed
#pragma unroll
  for (int i = 0; i < RB; ++i) {
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int run = (i * CB + cb) * 4 + g;
        const f32x4 v = {acc[i][cb][4 * g], acc[i][cb][4 * g + 1], acc[i][cb][4 * g + 2],
                         acc[i][cb][4 * g + 3]};
        *(f32x4*)(ring + run * 1024 + ((lane ^ ((run & 7) << 1)) * 16)) = v;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < kItems; ++it) {
    const int r = (tid + it * kThreads) / (C / kCpt);
    float v[kCpt];
#pragma unroll
    for (int j = 0; j < kCpt; ++j) { v[j] = 0.0f; }
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
#pragma unroll
      for (int s = 0; s < kCpt; s += kFv) {
        const int run = ((r >> 5) * CB + (c >> 5)) * 4 + ((c & 31) >> 3);
        const int ln = (r & 31) + 32 * (((c + s) >> 2) & 1);
        const fv a = *(const fv*)(lds + w * P::kWaveLds + run * 1024 +
                                  ((ln ^ ((run & 7) << 1)) * 16) + (c & 3) * 4);
#pragma unroll
        for (int j = 0; j < kFv; ++j) { v[s + j] += a[j]; }
      }
    }
    const int m = m0 + r;
    if (m >= p.M || n >= p.N) { continue; }
    if constexpr (SPLIT) {
      float* prow = p.partial + ((size_t)split * p.M + m) * p.N;
      if ((p.N & 3) == 0 && n + kCpt <= p.N) {
#pragma unroll
        for (int s = 0; s < kCpt; s += kFv) {
          fv o;
#pragma unroll
          for (int j = 0; j < kFv; ++j) { o[j] = v[s + j]; }
          *(fv*)(prow + n + s) = o;
        }
      } else {
#pragma unroll
        for (int j = 0; j < kCpt; ++j) {
          if (n + j < p.N) { prow[n + j] = v[j]; }
        }
      }
    } else {
      uint16_t* const yrow = p.y + (size_t)m * p.N;
      const uint16_t* const yin = p.y_in != nullptr ? p.y_in + (size_t)m * p.N : nullptr;
#pragma unroll
      for (int j = 0; j < kCpt; ++j) {
        if (yin != nullptr && n + j < p.N) { v[j] += bf16_to_f32(yin[n + j]); }
        v[j] += bv[j];
      }
      if (p.epilogue == kEpiGelu) {
#pragma unroll
        for (int j = 0; j < kCpt; ++j) { v[j] = gelu_tanh(v[j]); }
      }
      if ((p.N & 7) == 0 && n + kCpt <= p.N) {
        uint32_t o[kCpt / 2];
#pragma unroll
        for (int j = 0; j < kCpt / 2; ++j) { o[j] = pack_bf16x2(v[2 * j], v[2 * j + 1]); }
        __builtin_memcpy(__builtin_assume_aligned(yrow + n, 2 * kCpt), o, 2 * kCpt);
      } else {
#pragma unroll
        for (int j = 0; j < kCpt; ++j) {
          if (n + j < p.N) { yrow[n + j] = f32_to_bf16(v[j]); }
        }
      }
    }
  }
}

template <int BITS, int RB, int CB>
hipError_t launch_cfg(const PanelParams& p, dim3 grid, hipStream_t stream, hipEvent_t done)
{
  return p.splits > 1
             ? launch_done(panel_kernel<BITS, RB, CB, true>, grid, kThreads, stream, nullptr, p)
             : launch_done(panel_kernel<BITS, RB, CB, false>, grid, kThreads, stream, done, p);
}

template <int BITS>
hipError_t launch_bits(const PanelParams& p, int rb, int cb, dim3 grid, hipStream_t stream,
                       hipEvent_t done)
{
  if (cb == 2) {
    return rb == 4   ? launch_cfg<BITS, 4, 2>(p, grid, stream, done)
           : rb == 2 ? launch_cfg<BITS, 2, 2>(p, grid, stream, done)
                     : launch_cfg<BITS, 1, 2>(p, grid, stream, done);
  }
  return rb == 4   ? launch_cfg<BITS, 4, 1>(p, grid, stream, done)
         : rb == 2 ? launch_cfg<BITS, 2, 1>(p, grid, stream, done)
                   : launch_cfg<BITS, 1, 1>(p, grid, stream, done);
}

// The panels, with the time of one workgroup as measured on w8g64 calls whose
// workgroups fill the CUs at most once (captured bursts, rotated weights): a
// fixed part (launch, first loads, the sum of the partial tiles) and a part
// per chunk of a wave's range, both in us. 320 x 4096 -> 4096 (128 x 64): 22.6
// against 34.4 on the 128 x 128 split-K tile; 1000 x 4096 -> 512 (64 x 32) 13.1
// against 18.8; 16 x 8192 -> 16384 (32 x 64) 39.7 against 71.2.
struct PanelCost {
  int rows, cols;
  float fixed, per_chunk;
};
constexpr PanelCost kPanels[] = {
    {32, 32, 3.9f, 0.40f}, {64, 32, 4.2f, 0.52f},  {128, 32, 5.0f, 0.75f},
    {32, 64, 5.0f, 0.75f}, {64, 64, 5.3f, 0.78f}, {128, 64, 6.5f, 1.00f},
};
// Splitting K across workgroups as well: the reduction launch, and its f32
// partials written and read at 3 TB/s.
constexpr float kSplitUs = 3.5f;
constexpr float kPartialUsPerByte = 2.0f / 3e6f;
constexpr int kMinK = 1024;        // K per workgroup

}  // namespace

bool plan_panel(int M, int N, int K, int cu_count, GemmPlan& plan)
{
  // Below 1024 of K the fixed part outweighs what the in-workgroup split saves,
  // and the larger tiles sum K in one order.
  // The kernel's byte offsets are 32-bit, rows past the last panel's end
  // included, a dense weight's too.
  constexpr size_t kFourGib = (size_t)1 << 32;
  if (M < 1 || N < 1 || K < kMinK || K % kChunk != 0 || (size_t)(M + 128) * K * 2 >= kFourGib ||
      (size_t)(N + 64) * K * 2 >= kFourGib) {
    return false;
  }
  const long chunks = K / kChunk;
  float best = 0.0f;
  bool found = false;
  for (const PanelCost& c : kPanels) {
    if (c.rows >= M + 32 && c.rows > 32) { continue; }   // whole row blocks of nothing
    const long tiles = (long)((M + c.rows - 1) / c.rows) * ((N + c.cols - 1) / c.cols);
    for (long s = 1; s == 1 || K / s >= kMinK; ++s) {
      const long per = (chunks + s - 1) / s;
      if ((chunks + per - 1) / per != s) { continue; }
      // Past one round of workgroups (160 KB of LDS each, one per CU) a second
      // one repeats the fixed part: 8160 x 4096 -> 512 in two rounds of 128 x 64
      // 44.6 us, 41 on the 128 x 128 tile.
      if (tiles * s > cu_count) { break; }
      const float us = c.fixed + c.per_chunk * (float)((per + kWaves - 1) / kWaves) +
                       (s > 1 ? kSplitUs + (float)(s * M) * (float)N * 4.0f * kPartialUsPerByte : 0.0f);
      if (!found || us < best) {
        found = true;
        best = us;
        plan.panel_rows = c.rows;
        plan.panel_cols = c.cols;
        plan.splits = (int)s;
        plan.k_chunk = (int)per * kChunk;
      }
    }
  }
  if (!found) { return false; }
  plan.tile = 1;
  plan.workspace_bytes = plan.splits > 1 ? (size_t)plan.splits * M * N * sizeof(float) : 0;
  return true;
}

hipError_t launch_panel(const GemmDesc& d, const GemmPlan& plan, float* workspace,
                        hipStream_t stream)
{
  const int rb = plan.panel_rows / 32;
  const int cb = plan.panel_cols / 32;
  const size_t four = (size_t)1 << 32;
  if ((rb != 1 && rb != 2 && rb != 4) || (cb != 1 && cb != 2) ||
      d.M < 1 || d.N < 1 || d.K < kChunk || d.K % kChunk != 0 || plan.k_chunk % kChunk != 0 ||
      plan.k_chunk < kChunk || (long)plan.splits * plan.k_chunk < d.K || d.x2 != nullptr ||
      (d.bits != 8 && d.bits != 4 && d.bits != 16) || (plan.splits > 1 && workspace == nullptr) ||
      (size_t)(d.M + 128) * d.K * 2 >= four || (size_t)(d.N + 64) * d.K * d.bits / 8 >= four) {
    return hipErrorInvalidValue;
  }
  PanelParams p = {};
  p.x = d.x;
  p.w = d.w;
  if (d.bits != 16) {
    p.scales = (const void*)((uintptr_t)d.scales & ~(uintptr_t)15);
    p.qbias = (const void*)((uintptr_t)d.qbias & ~(uintptr_t)15);
    p.s_mis = (int)((uintptr_t)d.scales & 15) / 2;
    p.q_mis = (int)((uintptr_t)d.qbias & 15) / 2;
    while ((1 << p.gshift) < d.group) { ++p.gshift; }
    p.gcols = d.K / d.group;
  }
  p.bias = d.bias;
  p.bias_type = d.bias != nullptr ? d.bias_type : kBiasNone;
  p.epilogue = d.epilogue;
  p.y_in = d.y_in;
  p.y = d.y;
  p.partial = workspace;
  p.M = d.M;
  p.N = d.N;
  p.K = d.K;
  p.wn = d.wn > 0 && d.wn < d.N ? d.wn : d.N;
  p.k_chunk = plan.k_chunk;
  p.tiles_m = (d.M + 32 * rb - 1) / (32 * rb);
  p.tiles_n = (d.N + 32 * cb - 1) / (32 * cb);
  p.by_m = (size_t)d.M * 16 > (size_t)d.N * d.bits;
  p.splits = plan.splits;
  const dim3 grid((unsigned)(p.tiles_m * p.tiles_n * plan.splits));
  const hipError_t e = d.bits == 8    ? launch_bits<8>(p, rb, cb, grid, stream, d.done)
                       : d.bits == 16 ? launch_bits<16>(p, rb, cb, grid, stream, d.done)
                                      : launch_bits<4>(p, rb, cb, grid, stream, d.done);
  if (e != hipSuccess || plan.splits <= 1) { return e; }
  return launch_splitk_reduce(workspace, plan.splits, d.bias, p.bias_type, d.epilogue, d.y_in,
                              d.y, d.M, d.N, stream, d.done);
}

}  // namespace ltx25
