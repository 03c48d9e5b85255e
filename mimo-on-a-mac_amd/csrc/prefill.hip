// Prefill MoE: (token, k) routes sorted by slot, grouped gate/up + SwiGLU and down GEMMs on bf16 MFMA, bf16 expert
// outputs, fixed-order weighted combine back to token order.
//
// Reference: _moe_prefill engine/mimo_stream/model.py:230-271 and _pair_outputs :221-228 (three sorted
// gather_qmm calls, bf16 SwiGLU intermediate, bf16 expert outputs, inverse permutation, (Y.f32 * w).sum(1)).
//
// The dispatch cuts each slot's sorted routes into row tiles of at most 128 routes and writes the tile table.  A block
// (4 waves, two blocks per CU) owns one row tile and 256 weight rows, 64 per wave.  Weights go from HBM straight to
// the registers of the one wave that uses them and are turned into bf16 there (exactly: an E2M1 value times a power
// of two); the bf16 activation rows, which all four waves use, go through an LDS ring.
//
// What bounds it: up to ~700 tokens HBM (512 tokens: gate/up and down read 3.4 GB in ~680 us, 5 TB/s; the loads alone
// took 405 us of gate/up's 460, now 438); above, the MFMAs at the ~1.9 GHz that the chip's power leaves (60% busy at 6250
// tokens) and the copies that they hide only in part (gate/up 1516 us; without activation copies 1327, without weight
// loads 1296, without both 1184).  A layer step took 379 / 775 / 1273 / 2839 us at 24 / 512 / 2048 / 6250 tokens with
// two E4M3 planes per activation on the block-scaled MFMA and two launches per GEMM, and takes 313 / 702 / 1102 / 2431.
#include <algorithm>
#include <atomic>

#include "device.h"
#include "host.h"
#include "layer.h"
#include "router.h"

namespace mimo {

struct PrefillArgs {
  const uint16_t* x;      // [T, H] bf16
  const int32_t* perm;    // sorted position -> flat route
  const int4* tiles;      // the tile table (TileSpec)
  int wcap, k, H, I;
  // slots [0, S0) address the bank's pools, later ones the staging bank's (pool index 1, slot - S0)
  int S0;
  const uint32_t *gate_w[2], *up_w[2], *down_w[2];
  const uint8_t *gate_s[2], *up_s[2], *down_s[2];
  const uint16_t* sigtab;
  uint16_t* h;            // [P, I] bf16, sorted route order
  uint16_t* Y;            // [P, H] bf16 expert outputs, sorted route order
};

// Row tiles: a slot with at most PF_NARROW_MAX routes is one narrow tile, a larger one is cut into wide tiles of
// PF_WIDE_ROWS (PF_SMALL_ROWS) routes and a remainder.  A tile runs the shape of its NJ = ceil(routes / 16) chunks of 16 routes.
//
// A K-step is 128 codes.  Per step a wave loads 16 bytes per lane of each of its 4 weight tiles of 16 rows (lane
// (i, g) = (l % 16, l / 16): codes 32 g .. of row i, which share one E8M0 scale), DEPTH steps ahead of their use, and
// the block copies the routes' 256-byte row pieces into one of STAGES ring slots, STAGES - 1 steps ahead.  The four
// v_mfma_f32_16x16x32_bf16 of a step take dword m of every lane's weights (codes 32 g + 8 m ..) and the same columns
// of the routes, so the pairing is right whatever order the unit sums in.
//
// In LDS the 16-byte chunk 4 g + m of route r sits at position (4 m + g) ^ (r & 15) of its 256-byte row: the operand
// reads are then free of bank conflicts (with the chunk 4 g + m at (4 g + m) ^ (r & 15) they took twice the cycles).  The
// scale bytes are not: 16 rows of 32 bytes, 8 cycles a read, 6 of them conflicts, for 4 reads a step (0.18 to 0.39 conflict
// cycles per access cycle over the kernels).
constexpr int PF_NARROW_MAX = 32;
constexpr int PF_WIDE_ROWS = 128;
// Routes per slot up to which the streaming configuration runs (three blocks per CU, tiles of up to 64 routes), against
// the other: Zipf routes at 512 tokens (16 a slot) 720 us a layer against 750, 640 (20) 773 against 808, 768 (24) 810
// against 835, 1024 (32) 906 against 918; near-uniform ones at 700 tokens 779 against 792, at 1000 (31) 872 against 864.
// Its tiles are not smaller: at 32 routes a popular slot's weights were read and converted twice as often (Zipf, 512
// tokens: 763 us, 733 with 48).
constexpr int PF_SMALL_AVG = 24;
constexpr int PF_SMALL_ROWS = 64;
// It also runs when the wide tiles are fewer blocks than CUs (full tiles times gate/up output blocks): half the rows make
// twice the blocks.  H 4096, I 384, 64 slots: 800 tokens on 6 slots (112 blocks) 111 us a layer against 132, spread over
// all 134 against 129, 1700 spread (239) 200 against 215; H 7168, I 256, 32 slots, 800 tokens (50) 144 against 177; H 256,
// I 2048, 16 slots, 800 tokens (200) 53 against 63.  Above: H 768, I 384, 12 slots, 6000 tokens (422) 97 against 89.
constexpr int PF_FEW_BLOCKS = 256;
constexpr int PF_UNIT = 16;                          // routes per MFMA chunk
constexpr int PF_ROWS = 256;                         // weight rows per block
// the part of the bf16 sigmoid table that is not constant: |x| in [2^-9, 128) (below, 0.5; above, 0 or 1)
constexpr int PF_SIG_LO = 118 << 7, PF_SIG_N = 16 << 7;

constexpr int PF_SCW = 8;                            // steps per scale window
constexpr int PF_SC = PF_ROWS * 4 * PF_SCW;          // bytes of one window of the block's scales

// What the shapes of one kernel have in common: blocks per CU and the LDS of the activation ring (two scale windows
// follow it).
template <bool SMALL> struct PfKind {
  static constexpr int BLOCKS = SMALL ? 3 : 2;
  static constexpr int RING = SMALL ? 32768 : 65536;
  static constexpr int LDS = RING + 2 * PF_SC;
  static_assert(BLOCKS * LDS <= 163840, "blocks per CU within 160 KB of LDS");
};

template <int NJ, bool SMALL> struct PfShape : PfKind<SMALL> {
  using Kind = PfKind<SMALL>;
  static constexpr int STAGE = NJ * PF_UNIT * 256;
  static constexpr int STAGES = NJ >= 6 || (NJ >= 3 && SMALL) ? 2 : (NJ >= 3 || SMALL ? 3 : 4);
  static constexpr int AHEAD = STAGES - 1;
  static constexpr int DEPTH = NJ >= 6 || (NJ >= 3 && SMALL) ? 2 : (NJ >= 3 || SMALL ? 4 : 8);
  // Weights are requested LU steps at a time, 64 LU consecutive bytes of a row back to back, once the registers of LU
  // steps are free; EARLY steps of them before the first activation rows (whose addresses take a round trip to the
  // route list).
  static constexpr int LU = NJ >= 6 || (NJ >= 3 && SMALL) ? 1 : 2;
  static constexpr int EARLY = LU;
  // weight loads issued in the AHEAD steps before step u of a round of DEPTH
  static constexpr int newer(int u) {
    int n = 0;
    for (int v = 1; v <= AHEAD; ++v) n += ((u - v + DEPTH) % DEPTH) % LU == LU - 1 ? 4 * LU : 0;
    return n;
  }
  static constexpr int WB = SMALL ? 1 : 2;       // converted weights: of this dword, and of the next
  // the sigmoid entries: beside the ring where there is room, else over it once the K loop is done
  static constexpr bool TAB_LATE = STAGES * STAGE + 4 * PF_SIG_N > Kind::RING;
  static constexpr int TAB = TAB_LATE ? 0 : STAGES * STAGE;
  static_assert(STAGES * STAGE <= Kind::RING && 4 * PF_SIG_N <= Kind::RING, "ring");
  static_assert(DEPTH % LU == 0 && AHEAD <= DEPTH && 4 * (DEPTH - EARLY) >= 4 * ((AHEAD + LU - 1) / LU) * LU,
                "loads counted by the waits");
  static_assert(AHEAD <= PF_SCW, "scale windows landed in time");
};

// at most n of the most recent vector memory loads still in flight; n is a constant once the step loop is unrolled
__device__ __forceinline__ void pf_wait(int n) {
  switch (n) {
#define PF_W(c) case c: __builtin_amdgcn_s_waitcnt(vm_keep(c)); break;
#define PF_W8(c) PF_W(c) PF_W(c + 1) PF_W(c + 2) PF_W(c + 3) PF_W(c + 4) PF_W(c + 5) PF_W(c + 6) PF_W(c + 7)
    PF_W8(1) PF_W8(9) PF_W8(17) PF_W8(25) PF_W8(33) PF_W8(41) PF_W8(49)
#undef PF_W8
#undef PF_W
    default: __builtin_amdgcn_s_waitcnt(vm_keep(0)); break;
  }
}

__device__ __forceinline__ uint32_t pf_pack2(float lo, float hi) {
  return (uint32_t)f32_to_bf16(lo) | ((uint32_t)f32_to_bf16(hi) << 16);
}

// One (row tile, output block).  GATEUP: activations = the routes' token rows, weights = 128 gate and the same 128 up
// rows; epilogue SwiGLU to bf16 h.  !GATEUP: activations = the routes' h rows, weights = 256 down rows; bf16 outputs.
// Wave w, weight tile t, lane row i: GATEUP projection t / 2, output 32 w + 8 (i / 4) + 4 (t % 2) + i % 4; else output
// 64 w + 16 (i / 4) + 4 t + i % 4.  A lane's accumulators are then 8 (GATEUP) or 16 consecutive outputs of a route.
template <bool GATEUP, int NJ, bool SMALL>
__device__ __forceinline__ void pf_tile(const PrefillArgs& a, uint8_t* pl, int slot, int beg, int nvalid, int ob) {
  using Sh = PfShape<NJ, SMALL>;
  constexpr int D = Sh::DEPTH, AHEAD = Sh::AHEAD;
  const int lane = threadIdx.x & 63, g = lane >> 4, i = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K = GATEUP ? a.H : a.I;
  const int nK = K / 128, KS = K / 32, RB = K / 2;   // steps; scale and weight bytes per row
  const int ncol = GATEUP ? a.I : a.H;               // weight rows per slot and projection
  const int n0 = ob * (GATEUP ? PF_ROWS / 2 : PF_ROWS);
  auto out_row = [&](int t, int r) {
    return GATEUP ? 32 * wave + 8 * (r >> 2) + 4 * (t & 1) + (r & 3) : 64 * wave + 16 * (r >> 2) + 4 * t + (r & 3);
  };
  // token rows of the wave's copies: 4 NJ consecutive routes of the tile, one per lane (padding repeats the first)
  const int r0 = 4 * NJ * wave;
  int tok;
  {
    const int r = r0 + (lane & 31);
    const int p = beg + (r < nvalid ? r : 0);
    tok = GATEUP ? a.perm[p] : p;
  }
  const int pool = slot >= a.S0;                     // tile-uniform: the bank or the staging bank
  const size_t row0 = (size_t)(slot - (pool ? a.S0 : 0)) * ncol + n0;
  const uint8_t* w0 = reinterpret_cast<const uint8_t*>(GATEUP ? a.gate_w[pool] : a.down_w[pool]) + row0 * RB;
  const uint8_t* w1 = reinterpret_cast<const uint8_t*>(GATEUP ? a.up_w[pool] : a.down_w[pool]) + row0 * RB;
  const uint8_t* s0p = (GATEUP ? a.gate_s[pool] : a.down_s[pool]) + row0 * KS;
  const uint8_t* s1p = (GATEUP ? a.up_s[pool] : a.down_s[pool]) + row0 * KS;
  // the block's weight rows as buffers: a step past the row ends reads offset kPast, outside them, and fetches nothing
  constexpr int kPast = 0x40000000;
  const int wbytes = (GATEUP ? PF_ROWS / 2 : PF_ROWS) * RB;
  const __amdgpu_buffer_rsrc_t rs0 = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(w0), 0, wbytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs1 = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(w1), 0, wbytes, 0x00020000);
  int woff[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) woff[t] = out_row(t, i) * RB + 16 * g;
  const bool s16 = (KS & 15) == 0 && ((((uintptr_t)a.gate_s[pool] | (uintptr_t)a.up_s[pool] | (uintptr_t)a.down_s[pool]) & 15) == 0);
  v4i braw[D][4];
  auto issue_w = [&](int u, int s) __attribute__((always_inline)) {   // steps s .. s + LU - 1 into registers u ..
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int v = 0; v < Sh::LU; ++v)
        braw[u + v][t] = __builtin_bit_cast(
            v4i, __builtin_amdgcn_raw_buffer_load_b128(t < 2 ? rs0 : rs1, woff[t] + (s + v < nK ? 64 * (s + v) : kPast), 0, 0));
  };
  // Scale window w (steps PF_SCW w ..): SB bytes of each of the wave's 64 rows, tile row 16 t + i at SB (16 t + i) of
  // the wave's part of buffer w % 2; bytes past the row's end read its start (they are never used)
  constexpr int SB = 4 * PF_SCW;
  uint8_t* scl = pl + Sh::RING + wave * (PF_SC / 4);
  auto issue_scales = [&](int w) __attribute__((always_inline)) {
    uint8_t* dst = scl + (w % 2) * PF_SC;
    int ln = lane;
    asm volatile("" : "+v"(ln));                     // the addresses are not kept in registers between windows
    if (s16) {                                       // 16-byte pieces, SB / 16 lanes per row
#pragma unroll
      for (int c = 0; c < SB / 16; ++c) {
        const int q = 1024 / SB * c + ln / (SB / 16), at = SB * w + 16 * (ln % (SB / 16));
        lds_copy16(2 * c >= SB / 16 ? s1p : s0p, out_row(q >> 4, q & 15) * KS + (at < KS ? at : 0), dst + 1024 * c);
      }
    } else {                                         // rows of any multiple of 4 bytes: 4-byte pieces
#pragma unroll 1
      for (int c = 0; c < SB / 4; ++c) {
        const int q = 256 / SB * c + ln / (SB / 4), at = SB * w + 4 * (ln % (SB / 4));
        lds_copy4(2 * c >= SB / 4 ? s1p : s0p, out_row(q >> 4, q & 15) * KS + (at < KS ? at : 0), dst + 256 * c);
      }
    }
  };
  const uint8_t* act = reinterpret_cast<const uint8_t*>(GATEUP ? a.x : a.h);
  uint32_t a_off[NJ];
  auto issue_a = [&](int s) __attribute__((always_inline)) {
    uint8_t* st = pl + (s % Sh::STAGES) * Sh::STAGE;
#pragma unroll
    for (int c = 0; c < NJ; ++c) lds_copy16(act, a_off[c] + 256u * s, st + 1024 * (NJ * wave + c));
  };
  // operand addresses: route rows 16 j + i, chunk 4 g + m; scale byte of tile row 16 t + i, step s: + 4 (s % 8) + g
  const int aoff = 256 * i + 16 * (g ^ i);
  const uint8_t* scr = scl + SB * i + g;

  v4f acc[NJ][4];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[j][t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  uint32_t big = 2;                                  // least of 254 - scale byte (byte 255: NaN whatever the weight)
  issue_scales(0);
#pragma unroll
  for (int u = 0; u < Sh::EARLY; u += Sh::LU) issue_w(u, u);
  __builtin_amdgcn_sched_barrier(0);
  {
    const int token = GATEUP ? tok / a.k : tok;
    int ln = lane;
    asm volatile("" : "+v"(ln));                   // kept out of the registers that live across the K loop
#pragma unroll
    for (int c = 0; c < NJ; ++c) {
      const int rl = 4 * c + (ln >> 4), r = r0 + rl;
      const uint32_t row = (uint32_t)__shfl(token, rl, 64) * (uint32_t)(2 * K);
      const int at = (ln ^ r) & 15;        // 4 m + g of the lane's position
      a_off[c] = row + (r < nvalid ? 16u * (uint32_t)(4 * (at & 3) + (at >> 2)) : 0u);
    }
  }
#pragma unroll
  for (int s = 0; s < AHEAD; ++s)
    if (s < nK) issue_a(s);
  if constexpr (GATEUP && !Sh::TAB_LATE) {
#pragma unroll
    for (int c = 0; c < 2; ++c)
      lds_copy16(a.sigtab + PF_SIG_LO + (wave >= 2 ? 32768 : 0), 2048 * (wave & 1) + 1024 * c + 16 * lane,
                 pl + Sh::TAB + 2048 * wave + 1024 * c);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = Sh::EARLY; u < D; u += Sh::LU) issue_w(u, u);
  __builtin_amdgcn_sched_barrier(0);

  for (int sb = 0; sb < nK; sb += D) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      const int s = sb + u;                        // past nK (a last round of fewer than D steps): nothing multiplied
      // The activation copies of step s have landed once no more than the loads issued after them are in flight:
      // the weights requested since and, away from the end, AHEAD - 1 steps' copies.
      if (s + AHEAD <= nK) pf_wait(Sh::newer(u) + (AHEAD - 1) * NJ);
      else pf_wait(Sh::newer(u));
      __syncthreads();                             // step s landed everywhere; the slot of step s - 1 is free
      // the step's weights are waited for here, before any newer copy is issued
      asm volatile("" : "+v"(braw[u][0]), "+v"(braw[u][1]), "+v"(braw[u][2]), "+v"(braw[u][3])::"memory");
      if (s + AHEAD < nK) issue_a(s + AHEAD);
      if (s % PF_SCW == 0 && s + PF_SCW < nK) issue_scales(s / PF_SCW + 1);
      __builtin_amdgcn_sched_barrier(0);
      if (s < nK) {
        const uint8_t* st = pl + (s % Sh::STAGES) * Sh::STAGE;
        const uint8_t* sp = scr + (s / PF_SCW % 2) * PF_SC + 4 * (s % PF_SCW);
        float sc[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const uint32_t e = sp[16 * SB * t];
          big = min(big, 254u - e);
          sc[t] = e8m0_f32(e);
        }
        // 4 NJ groups of a route chunk times the 4 weight tiles: a group's activation operand is read PX groups ahead
        // and the next dword's weights are converted a tile at a time, both while earlier MFMAs run
        constexpr int G = 4 * NJ, PX = NJ == 1 ? 1 : 3;
        auto read_x = [&](int f) { return *reinterpret_cast<const bf16x8*>(st + (aoff ^ (64 * (f / NJ))) + 4096 * (f % NJ)); };
        bf16x8 X[PX + 1], W[Sh::WB][4];
#pragma unroll
        for (int f = 0; f < PX; ++f) X[f] = read_x(f);
#pragma unroll
        for (int t = 0; t < 4; ++t) W[0][t] = fp4_bf16x8(braw[u][t][0], sc[t]);
#pragma unroll
        for (int f = 0; f < G; ++f) {
          const int m = f / NJ, j = f % NJ;
          __builtin_amdgcn_sched_barrier(0);
          if (f + PX < G) X[(f + PX) & PX] = read_x(f + PX);
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            if (Sh::WB == 2 && m < 3 && t * NJ / 4 == j) W[(m + 1) & 1][t] = fp4_bf16x8(braw[u][t][m + 1], sc[t]);
            if (Sh::WB == 1 && m > 0 && j == 0) W[0][t] = fp4_bf16x8(braw[u][t][m], sc[t]);
          }
#pragma unroll
          for (int t = 0; t < 4; ++t)
            acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(W[m % Sh::WB][t], X[f & PX], acc[j][t], 0, 0, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (u % Sh::LU == Sh::LU - 1) issue_w(u - Sh::LU + 1, s + D - Sh::LU + 1);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // Scale bytes 253 and 254 (weights that bf16 cannot hold): the tile's sums are taken again in parts, rows, weights and
  // scales straight from memory
  const bool over = __ballot(big <= 1u) != 0;
  uint32_t* flag = reinterpret_cast<uint32_t*>(pl + Sh::LDS - 16);
  wait_vm_all();
  __syncthreads();                                   // every wave is done with the ring and the scales
  if (lane == 0) flag[wave] = over ? 1u : 0u;
  if constexpr (GATEUP && Sh::TAB_LATE) {
#pragma unroll
    for (int c = 0; c < 2; ++c)
      lds_copy16(a.sigtab + PF_SIG_LO + (wave >= 2 ? 32768 : 0), 2048 * (wave & 1) + 1024 * c + 16 * lane,
                 pl + Sh::TAB + 2048 * wave + 1024 * c);
    wait_vm_all();
  }
  __syncthreads();
  if (__builtin_amdgcn_readfirstlane(flag[0] | flag[1] | flag[2] | flag[3])) {
    int ln = lane;
    asm volatile("" : "+v"(ln));                     // nothing of this is kept in registers across the K loop
    const int gl = ln >> 4, il = ln & 15;
    uint32_t xrow[NJ];                               // byte offsets of the lane's routes 16 j + i, codes 32 g ..
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int p = beg + (PF_UNIT * j + il < nvalid ? PF_UNIT * j + il : 0);
      xrow[j] = (uint32_t)(GATEUP ? a.perm[p] / a.k : p) * (uint32_t)(2 * K) + 64u * gl;
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[j][t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    }
#pragma unroll 1
    for (int part = 0; part < 2; ++part) {
      const bool hp = part == 0;
#pragma unroll 1
      for (int s = 0; s < nK; ++s)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const uint32_t e = (t < 2 ? s0p : s1p)[out_row(t, il) * KS + 4 * s + gl];
          const uint8_t* wp = (t < 2 ? w0 : w1) + (size_t)out_row(t, il) * RB + 16 * gl + 64 * s;
          const float sc = part_scale(e, hp);
#pragma unroll 1
          for (int m = 0; m < 4; ++m) {
            const uint32_t w = *reinterpret_cast<const uint32_t*>(wp + 4 * m);
            const bf16x8 W = fp4_bf16x8(huge_scale(e) == hp ? w : 0u, sc);
#pragma unroll
            for (int j = 0; j < NJ; ++j)
              acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                  W, *reinterpret_cast<const bf16x8*>(act + xrow[j] + 256u * s + 16 * m), acc[j][t], 0, 0, 0);
          }
        }
      if (hp) {
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int t = 0; t < 4; ++t) acc[j][t] = acc[j][t] * 4.0f;
      }
    }
  }

  // epilogue: lane (i, g) holds route 16 j + i at outputs 8 g .. (GATEUP) or 16 g .. of the wave
  if constexpr (GATEUP) {
    const uint16_t* tab = reinterpret_cast<const uint16_t*>(pl + Sh::TAB);
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      float hv[8];
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint16_t gt = f32_to_bf16(acc[j][b][q]);
          const int mag = min(max((int)(gt & 0x7FFF), PF_SIG_LO), PF_SIG_LO + PF_SIG_N - 1) - PF_SIG_LO;
          const float sig = bf16_to_f32(tab[mag + ((gt & 0x8000) ? PF_SIG_N : 0)]);
          hv[4 * b + q] = round_bf16(bf16_to_f32(gt) * sig) * round_bf16(acc[j][2 + b][q]);
        }
      const int r = PF_UNIT * j + i;
      if (r < nvalid)
        *reinterpret_cast<uint4*>(a.h + (size_t)(beg + r) * a.I + n0 + 32 * wave + 8 * g) =
            make_uint4(pf_pack2(hv[0], hv[1]), pf_pack2(hv[2], hv[3]), pf_pack2(hv[4], hv[5]), pf_pack2(hv[6], hv[7]));
    }
  } else {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int r = PF_UNIT * j + i;
      if (r >= nvalid) continue;
      uint4* dst = reinterpret_cast<uint4*>(a.Y + (size_t)(beg + r) * a.H + n0 + 64 * wave + 16 * g);
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const v4f p = acc[j][2 * b], q = acc[j][2 * b + 1];
        dst[b] = make_uint4(pf_pack2(p[0], p[1]), pf_pack2(p[2], p[3]), pf_pack2(q[0], q[1]), pf_pack2(q[2], q[3]));
      }
    }
  }
}

// One launch per GEMM.  Workgroups go to the 8 XCDs round robin (hardware block b runs on XCD b % 8); XCD x takes the
// x-th share of the wide (tile, output block) pairs, of equal cost (by count, a popular slot's tiles left one XCD up to
// 13% more work than the average at 2048 tokens), then the x-th eighth of the narrow ones, a tile's output blocks one
// after the other (they share its activations in L2).  The 1-D grid has room for the tile table's capacity; blocks past
// the used pairs exit at once.
template <bool GATEUP, bool SMALL>
__global__ void __launch_bounds__(256, PfKind<SMALL>::BLOCKS) prefill_gemm_kernel(PrefillArgs a) {
  extern __shared__ __align__(256) uint8_t pl[];
  const int x = blockIdx.x & 7;
  int j = blockIdx.x >> 3;
  const int4 hdr = a.tiles[0], c0 = a.tiles[1 + x], c1 = a.tiles[1 + min(x + 1, 7)];
  const int nw = __builtin_amdgcn_readfirstlane(hdr.x), nn = __builtin_amdgcn_readfirstlane(hdr.y);
  const int obn = GATEUP ? a.I / (PF_ROWS / 2) : a.H / PF_ROWS;   // output blocks per tile
  auto start = [&](int4 c) {                     // first pair of a share
    return __builtin_amdgcn_readfirstlane(c.x * obn + (c.y * obn + 8 * c.z - 1) / (8 * c.z));
  };
  int at = kTileHead, l = 0, n = 0;
  if (nw > 0) {
    l = start(c0);
    n = (x < 7 ? start(c1) : nw * obn) - l;
  }
  l += j;
  if (j >= n) {
    const int per = (nn * obn + 7) / 8;
    j -= n;
    at += a.wcap;
    l = x * per + j;
    if (j >= per || l >= nn * obn) return;
  }
  const int tile = l / obn, ob = l - tile * obn;
  const int4 tt = a.tiles[at + tile];
  const int slot = __builtin_amdgcn_readfirstlane(tt.x), beg = __builtin_amdgcn_readfirstlane(tt.y);
  const int nv = __builtin_amdgcn_readfirstlane(tt.z - tt.y);
  if constexpr (SMALL) {
    if (nv <= 16) pf_tile<GATEUP, 1, true>(a, pl, slot, beg, nv, ob);
    else if (nv <= 32) pf_tile<GATEUP, 2, true>(a, pl, slot, beg, nv, ob);
    else if (nv <= 48) pf_tile<GATEUP, 3, true>(a, pl, slot, beg, nv, ob);
    else pf_tile<GATEUP, 4, true>(a, pl, slot, beg, nv, ob);
  } else {
    if (nv <= 32) pf_tile<GATEUP, 2, false>(a, pl, slot, beg, nv, ob);
    else if (nv <= 48) pf_tile<GATEUP, 3, false>(a, pl, slot, beg, nv, ob);
    else if (nv <= 64) pf_tile<GATEUP, 4, false>(a, pl, slot, beg, nv, ob);
    else if (nv <= 80) pf_tile<GATEUP, 5, false>(a, pl, slot, beg, nv, ob);
    else if (nv <= 96) pf_tile<GATEUP, 6, false>(a, pl, slot, beg, nv, ob);
    else if (nv <= 112) pf_tile<GATEUP, 7, false>(a, pl, slot, beg, nv, ob);
    else pf_tile<GATEUP, 8, false>(a, pl, slot, beg, nv, ob);
  }
}

// ------------------------------------------------------------------ weighted combine in route order
// y[t] = bf16(sum_j fp32(Y[inv[t*k + j]]) * w[t, j]), j ascending (model.py:269-271).  A thread owns 8 outputs
// (16-byte loads); all k route rows are requested before the sum.
__global__ void __launch_bounds__(256) prefill_combine_kernel(const uint16_t* __restrict__ Y, const int32_t* __restrict__ inv,
                                                              const float* __restrict__ w, int k, int H,
                                                              const uint16_t* resid, uint16_t* y) {
#pragma clang fp contract(off)
  const int t = blockIdx.y;
  const int m = (blockIdx.x * 256 + threadIdx.x) * 8;
  if (m >= H) return;
  float acc[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  constexpr int KB = 8;                          // routes whose rows are in flight at once
  for (int j0 = 0; j0 < k; j0 += KB) {
    uint4 v[KB];
    float wj[KB];
#pragma unroll
    for (int jj = 0; jj < KB; ++jj) {
      const int j = j0 + jj < k ? j0 + jj : j0;
      v[jj] = *reinterpret_cast<const uint4*>(Y + (size_t)inv[t * k + j] * H + m);
      wj[jj] = w[t * k + j];
    }
#pragma unroll
    for (int jj = 0; jj < KB; ++jj) {
      if (j0 + jj >= k) break;
      const uint32_t u[4] = {v[jj].x, v[jj].y, v[jj].z, v[jj].w};
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float lo = __uint_as_float(u[q] << 16), hi = __uint_as_float(u[q] & 0xFFFF0000u);
        const float plo = lo * wj[jj], phi = hi * wj[jj];
        acc[2 * q] = acc[2 * q] + plo;
        acc[2 * q + 1] = acc[2 * q + 1] + phi;
      }
    }
  }
  uint16_t yb[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) yb[q] = f32_to_bf16(acc[q]);
  if (resid) {                       // h = x + y of the decoder layer (resid may alias y: read before the write)
    const uint4 rv = *reinterpret_cast<const uint4*>(resid + (size_t)t * H + m);
    const uint32_t r[4] = {rv.x, rv.y, rv.z, rv.w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      yb[2 * q] = residual_bf16((uint16_t)r[q], yb[2 * q]);
      yb[2 * q + 1] = residual_bf16((uint16_t)(r[q] >> 16), yb[2 * q + 1]);
    }
  }
  uint4 o;
  o.x = (uint32_t)yb[0] | ((uint32_t)yb[1] << 16);
  o.y = (uint32_t)yb[2] | ((uint32_t)yb[3] << 16);
  o.z = (uint32_t)yb[4] | ((uint32_t)yb[5] << 16);
  o.w = (uint32_t)yb[6] | ((uint32_t)yb[7] << 16);
  *reinterpret_cast<uint4*>(y + (size_t)t * H + m) = o;
}

// ------------------------------------------------------------------ host
struct PrefillWs {
  int32_t *hist, *perm, *inv, *offsets, *status, *slot_inds;
  int4* tiles;
  float *logits, *w;
  int32_t* inds;
  uint16_t *h, *Y;
};

// Tile capacities: a slot of c > PF_NARROW_MAX routes is ceil(c / PF_WIDE_ROWS) wide tiles, at most
// P / PF_WIDE_ROWS + #{s : c_s > PF_NARROW_MAX} together; at most one narrow tile per slot.
struct PfTiling {
  int wcap, scap, rows;
  bool small;
};
static int pf_wide_cap(int64_t P, int S, int rows) {
  return (int)(P / rows + std::min<int64_t>(S, P / (PF_NARROW_MAX + 1)) + 1);
}
static PfTiling pf_tiling(int64_t P, int S, int I) {
  PfTiling t;
  t.small = P <= (int64_t)PF_SMALL_AVG * S || P * I < (int64_t)PF_FEW_BLOCKS * PF_WIDE_ROWS * (PF_ROWS / 2);
  t.rows = t.small ? PF_SMALL_ROWS : PF_WIDE_ROWS;
  t.wcap = pf_wide_cap(P, S, t.rows);
  t.scap = (int)std::min<int64_t>(S, P);
  return t;
}

// The need grows with T alone: a workspace sized for the longest chunk holds every shorter one.
static PrefillWs carve_prefill(Carve& c, int T, int k, int S, int H, int I, int E) {
  PrefillWs w{};
  const size_t P = (size_t)T * k;
  const PfTiling tl = pf_tiling((int64_t)P, S, I);
  w.status = c.take<int32_t>(1);
  w.hist = reinterpret_cast<int32_t*>(c.take<char>(dispatch_workspace((int)P, S)));
  w.perm = c.take<int32_t>(P);
  w.inv = c.take<int32_t>(P);
  w.offsets = c.take<int32_t>(S + 1);
  // with the capacity that tiles of PF_SMALL_ROWS need in either configuration
  w.tiles = c.take<int4>(kTileHead + (size_t)pf_wide_cap((int64_t)P, S, PF_SMALL_ROWS) + tl.scap);
  if (E > 0) {
    w.inds = c.take<int32_t>(P);
    w.w = c.take<float>(P);
    w.slot_inds = c.take<int32_t>(P);
  }
  // the selection has read the logits before h and Y are written: they share their room
  Carve over = c;
  w.h = c.take<uint16_t>(P * I);
  w.Y = c.take<uint16_t>(P * H);
  if (E > 0) {
    w.logits = over.take<float>((size_t)std::max(T, kRlParts * std::min(T, kRlPartsMax)) * E);
    c.off = std::max(c.off, over.off);
  }
  return w;
}

template <bool GATEUP, bool SMALL> static int pf_allow_lds() {
  static std::atomic<int> allowed{0};   // host threads may race to set the attribute; setting it twice is harmless
  if (allowed.load(std::memory_order_acquire)) return MIMO_OK;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&prefill_gemm_kernel<GATEUP, SMALL>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, PfKind<SMALL>::LDS);
  if (e != hipSuccess) return set_error(MIMO_ERR_HIP, "prefill LDS attribute: %s", hipGetErrorString(e));
  allowed.store(1, std::memory_order_release);
  return MIMO_OK;
}

// stage (optional): a second bank whose slots follow the bank's (slot ids bank->n_slots ...).  zero_status: the status
// word has not been cleared yet in this call (the dispatch's first kernel clears it before it may flag bad slots)
static int run_prefill(const uint16_t* x, int T, const int32_t* slot_inds, const float* wts, int k, const mimo_bank* bank,
                       const mimo_bank* stage, uint16_t* y, const PrefillWs& ws, hipStream_t st, bool zero_status,
                       const uint16_t* resid = nullptr) {
  const int H = bank->hidden, I = bank->inter, S = bank->n_slots + (stage ? stage->n_slots : 0);
  const int P = T * k;
  // the GEMM kernels address activation and h rows with 32-bit byte offsets
  MIMO_REQUIRE((int64_t)T * H < (int64_t)1 << 31 && (int64_t)P * I < (int64_t)1 << 31, MIMO_ERR_SHAPE,
               "moe_prefill: T * hidden and T * k * inter must stay below 2^31");
  int err;
  const uint16_t* sig = sigtab_device(&err);
  if (!sig) return err;
  const PfTiling tl = pf_tiling(P, S, I);
  const TileSpec spec{PF_NARROW_MAX, tl.rows, tl.wcap};
  int rc = launch_dispatch(slot_inds, P, S, ws.hist, ws.perm, ws.offsets, ws.inv, &spec, ws.tiles, ws.status,
                           zero_status, st);
  if (rc) return rc;
  PrefillArgs a{};
  a.x = x; a.perm = ws.perm; a.tiles = ws.tiles; a.wcap = tl.wcap; a.k = k; a.H = H; a.I = I;
  a.S0 = bank->n_slots;
  const mimo_bank* pools[2] = {bank, stage ? stage : bank};
  for (int i = 0; i < 2; ++i) {
    a.gate_w[i] = pools[i]->gate_w; a.up_w[i] = pools[i]->up_w; a.down_w[i] = pools[i]->down_w;
    a.gate_s[i] = pools[i]->gate_s; a.up_s[i] = pools[i]->up_s; a.down_s[i] = pools[i]->down_s;
  }
  a.sigtab = sig; a.h = ws.h; a.Y = ws.Y;
  rc = pf_allow_lds<true, true>();
  if (!rc) rc = pf_allow_lds<false, true>();
  if (!rc) rc = pf_allow_lds<true, false>();
  if (!rc) rc = pf_allow_lds<false, false>();
  if (rc) return rc;
  // 1-D grids with an index on every XCD for each of its (tile, output block) pairs of either kind; blocks past the
  // used pairs exit at once.  A wide tile costs at least kTileCost + 1, all of them at most `cost`, and a share holds an
  // eighth of the cost and less than one tile more.
  const int64_t cost = (int64_t)(kTileCost + 1) * tl.wcap + P / PF_UNIT;
  auto grid_of = [&](int obn) {
    const int64_t wide = (cost / 8 + 1 + kTileCost + tl.rows / PF_UNIT) * obn / (kTileCost + 1) + 2;
    return 8 * (int)(wide + ((int64_t)tl.scap * obn + 7) / 8);
  };
  { ProfScope p(st, "prefill_gateup");
    const int grid = grid_of(I / (PF_ROWS / 2));
    if (tl.small) prefill_gemm_kernel<true, true><<<grid, 256, PfKind<true>::LDS, st>>>(a);
    else prefill_gemm_kernel<true, false><<<grid, 256, PfKind<false>::LDS, st>>>(a); }
  { ProfScope p(st, "prefill_down");
    const int grid = grid_of(H / PF_ROWS);
    if (tl.small) prefill_gemm_kernel<false, true><<<grid, 256, PfKind<true>::LDS, st>>>(a);
    else prefill_gemm_kernel<false, false><<<grid, 256, PfKind<false>::LDS, st>>>(a); }
  { ProfScope p(st, "prefill_combine");
    prefill_combine_kernel<<<dim3((H + 2047) / 2048, T), 256, 0, st>>>(ws.Y, ws.inv, wts, k, H, resid, y); }
  return check_launch("moe prefill");
}

static int check_prefill_bank(const mimo_bank* b) {
  MIMO_REQUIRE(b && b->gate_w && b->gate_s && b->up_w && b->up_s && b->down_w && b->down_s, MIMO_ERR_ARG,
               "bank: null pointer");
  MIMO_REQUIRE(b->n_slots >= 1 && b->n_slots <= 1024 && b->hidden % 256 == 0 && b->hidden >= 256 &&
                   b->inter % 128 == 0 && b->inter >= 128,
               MIMO_ERR_SHAPE, "prefill bank: need hidden a multiple of 256, inter of 128, n_slots <= 1024");
  MIMO_REQUIRE(((reinterpret_cast<uintptr_t>(b->gate_s) | reinterpret_cast<uintptr_t>(b->up_s) |
                 reinterpret_cast<uintptr_t>(b->down_s)) & 3) == 0,
               MIMO_ERR_ALIGN, "bank: scale pools must be 4-byte aligned");
  MIMO_REQUIRE(aligned16(b->gate_w) && aligned16(b->up_w) && aligned16(b->down_w), MIMO_ERR_ALIGN,
               "bank: weight pools must be 16-byte aligned");
  return MIMO_OK;
}

}  // namespace mimo

using namespace mimo;

extern "C" {

size_t mimo_moe_prefill_workspace_size(int T, int k, int n_slots, int H, int I) {
  Carve c(nullptr, 0);
  carve_prefill(c, T, k, n_slots, H, I, 0);
  return c.off;
}

int mimo_moe_prefill(const uint16_t* x, int T, const int32_t* slot_inds, const float* w, int k, const mimo_bank* bank,
                     uint16_t* y, int32_t* status_out, void* ws, size_t ws_bytes, void* stream) {
  ProfChain chain;   // per-kernel timing (when enabled) back to back within this call
  int rc = check_prefill_bank(bank);
  if (rc) return rc;
  MIMO_REQUIRE(x && slot_inds && w && y, MIMO_ERR_ARG, "moe_prefill: null pointer");
  MIMO_REQUIRE(T >= 1 && k >= 1 && (int64_t)T * k < (1 << 30), MIMO_ERR_SHAPE, "moe_prefill: bad T or k");
  MIMO_REQUIRE(aligned16(x) && aligned16(y), MIMO_ERR_ALIGN, "moe_prefill: 16-byte alignment");
  Carve c(ws, ws_bytes);
  PrefillWs pw = carve_prefill(c, T, k, bank->n_slots, bank->hidden, bank->inter, 0);
  MIMO_REQUIRE(ws && c.fits(), MIMO_ERR_WORKSPACE, "moe_prefill: workspace too small (need %zu)", c.off);
  if (status_out) pw.status = status_out;
  return run_prefill(x, T, slot_inds, w, k, bank, nullptr, y, pw, as_stream(stream), true);
}

int mimo_moe_prefill_staged(const uint16_t* x, int T, const int32_t* slot_inds, const float* w, int k,
                            const mimo_bank* bank, const mimo_bank* stage, uint16_t* y, int32_t* status_out, void* ws,
                            size_t ws_bytes, void* stream) {
  ProfChain chain;
  int rc = check_prefill_bank(bank);
  if (rc) return rc;
  rc = check_prefill_bank(stage);
  if (rc) return rc;
  MIMO_REQUIRE(stage->hidden == bank->hidden && stage->inter == bank->inter, MIMO_ERR_SHAPE,
               "moe_prefill_staged: staging bank of another expert shape");
  MIMO_REQUIRE(bank->n_slots + stage->n_slots <= 1024, MIMO_ERR_SHAPE,
               "moe_prefill_staged: at most 1024 slots in the bank and the staging bank together");
  MIMO_REQUIRE(x && slot_inds && w && y, MIMO_ERR_ARG, "moe_prefill_staged: null pointer");
  MIMO_REQUIRE(T >= 1 && k >= 1 && (int64_t)T * k < (1 << 30), MIMO_ERR_SHAPE, "moe_prefill_staged: bad T or k");
  MIMO_REQUIRE(aligned16(x) && aligned16(y), MIMO_ERR_ALIGN, "moe_prefill_staged: 16-byte alignment");
  Carve c(ws, ws_bytes);
  PrefillWs pw = carve_prefill(c, T, k, bank->n_slots + stage->n_slots, bank->hidden, bank->inter, 0);
  MIMO_REQUIRE(ws && c.fits(), MIMO_ERR_WORKSPACE, "moe_prefill_staged: workspace too small (need %zu)", c.off);
  if (status_out) pw.status = status_out;
  return run_prefill(x, T, slot_inds, w, k, bank, stage, y, pw, as_stream(stream), true);
}

size_t mimo_moe_prefill_block_workspace_size(int T, int E, int k, int n_slots, int H, int I) {
  Carve c(nullptr, 0);
  carve_prefill(c, T, k, n_slots, H, I, E);
  return c.off;
}

}  // extern "C"

namespace mimo {
// Router + grouped GEMMs + combine on rows x; resid: optional residual stream added in the combine.
static int prefill_block_impl(const uint16_t* x, int T, const uint16_t* Wg, const float* bias, const int32_t* slot_of,
                              int E, int k, const mimo_bank* bank, uint16_t* y, int32_t* inds_out, float* w_out,
                              const uint16_t* resid, int32_t* status_out, void* ws, size_t ws_bytes, hipStream_t st) {
  int rc = check_prefill_bank(bank);
  if (rc) return rc;
  MIMO_REQUIRE(x && Wg && bias && y, MIMO_ERR_ARG, "moe_prefill_block: null pointer");
  MIMO_REQUIRE(T >= 1 && k >= 1 && k <= 16 && E >= k && E <= 1024 && bank->hidden % 64 == 0, MIMO_ERR_SHAPE,
               "moe_prefill_block: need 1 <= k <= min(16, E), E <= 1024");
  MIMO_REQUIRE(aligned16(x) && aligned16(Wg) && aligned16(y), MIMO_ERR_ALIGN, "moe_prefill_block: alignment");
  Carve c(ws, ws_bytes);
  PrefillWs pw = carve_prefill(c, T, k, bank->n_slots, bank->hidden, bank->inter, E);
  MIMO_REQUIRE(ws && c.fits(), MIMO_ERR_WORKSPACE, "moe_prefill_block: workspace too small (need %zu)", c.off);
  int32_t* inds = inds_out ? inds_out : pw.inds;
  float* wts = w_out ? w_out : pw.w;
  if (status_out) pw.status = status_out;
  const bool parts = router_logits_parts(x, Wg, T, bank->hidden);
  rc = parts ? launch_router_logits_parts(x, Wg, T, bank->hidden, E, pw.logits, st, pw.status)
             : launch_router_logits(x, Wg, T, bank->hidden, E, pw.logits, st, pw.status);   // clears the status word
  if (rc) return rc;
  rc = launch_router_select(pw.logits, bias, T, E, k, 1.0f, inds, wts, slot_of, pw.slot_inds, bank->n_slots, pw.status,
                            st, parts);
  if (rc) return rc;
  return run_prefill(x, T, pw.slot_inds, wts, k, bank, nullptr, y, pw, st, false, resid);
}
}  // namespace mimo

extern "C" {

int mimo_moe_prefill_block(const uint16_t* x, int T, const uint16_t* Wg, const float* bias, const int32_t* slot_of,
                           int E, int k, const mimo_bank* bank, uint16_t* y, int32_t* inds_out, float* w_out,
                           int32_t* status_out, void* ws, size_t ws_bytes, void* stream) {
  ProfChain chain;   // per-kernel timing (when enabled) back to back within this call
  return prefill_block_impl(x, T, Wg, bias, slot_of, E, k, bank, y, inds_out, w_out, nullptr, status_out, ws, ws_bytes,
                            as_stream(stream));
}

// The normalised rows r (T x H bf16) go first in the layer workspace, 256-byte aligned.
static size_t prefill_rows_bytes(int T, int H) { return ((size_t)T * H * 2 + 255) / 256 * 256; }

size_t mimo_moe_layer_prefill_workspace_size(int T, int E, int k, int n_slots, int H, int I) {
  return prefill_rows_bytes(T, H) + mimo_moe_prefill_block_workspace_size(T, E, k, n_slots, H, I);
}

int mimo_moe_layer_prefill(const uint16_t* x, int T, const uint16_t* norm_w, float eps, const uint16_t* Wg,
                           const float* bias, const int32_t* slot_of, int E, int k, const mimo_bank* bank, uint16_t* h,
                           uint16_t* r_out, int32_t* inds_out, float* w_out, int32_t* status_out, void* ws,
                           size_t ws_bytes, void* stream) {
  ProfChain chain;
  MIMO_REQUIRE(x && norm_w && h && bank, MIMO_ERR_ARG, "moe_layer_prefill: null pointer");
  MIMO_REQUIRE(T >= 1, MIMO_ERR_SHAPE, "moe_layer_prefill: need T >= 1");
  MIMO_REQUIRE(aligned16(x) && aligned16(h) && (!r_out || aligned16(r_out)), MIMO_ERR_ALIGN,
               "moe_layer_prefill: 16-byte alignment");
  MIMO_REQUIRE(r_out != x && r_out != h, MIMO_ERR_ARG, "moe_layer_prefill: r_out may not alias x or h");
  const int H = bank->hidden;
  const size_t rb = prefill_rows_bytes(T, H);
  MIMO_REQUIRE(ws && ws_bytes >= rb, MIMO_ERR_WORKSPACE, "moe_layer_prefill: workspace too small (need %zu)",
               mimo_moe_layer_prefill_workspace_size(T, E, k, bank->n_slots, H, bank->inter));
  hipStream_t st = as_stream(stream);
  uint16_t* r = r_out ? r_out : static_cast<uint16_t*>(ws);
  int rc = launch_rmsnorm(x, T, H, norm_w, eps, r, st);
  if (rc) return rc;
  return prefill_block_impl(r, T, Wg, bias, slot_of, E, k, bank, h, inds_out, w_out, x, status_out,
                            static_cast<uint8_t*>(ws) + rb, ws_bytes - rb, st);
}

}  // extern "C"
