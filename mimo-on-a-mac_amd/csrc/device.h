// Device helpers shared by the MoE kernels (gfx950 / CDNA4, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mimo {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// ------------------------------------------------------------------ bf16
__device__ __forceinline__ float bf16_to_f32(uint16_t b) { return __uint_as_float((uint32_t)b << 16); }

// round-to-nearest-even float -> bf16 bits; NaN stays a quiet NaN with its high payload bits, i.e.
// ((u + 0x7FFF + ((u >> 16) & 1)) >> 16 for numbers, (u >> 16) | 0x40 for NaN.  The hardware conversion
// (v_cvt_pk_bf16_f32) gives exactly these bits for every one of the 2^32 inputs (checked on MI355X).
__device__ __forceinline__ uint16_t f32_to_bf16(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
__device__ __forceinline__ float round_bf16(float f) { return bf16_to_f32(f32_to_bf16(f)); }

// ------------------------------------------------------------------ E2M1 / E8M0
// E2M1 magnitude code for y >= 0 already divided by the block scale: nearest-even on
// {0, .5, 1, 1.5, 2, 3, 4, 6}, saturating at 6 (OCP MX v1.0).
__device__ __forceinline__ uint32_t e2m1_mag_code(float y) {
  float v;
  if (y < 2.0f) v = rintf(y * 2.0f) * 0.5f;
  else if (y < 4.0f) v = rintf(y);
  else v = rintf(y * 0.5f) * 2.0f;
  // v in {0,.5,1,1.5,2,3,4,6,8}
  if (v >= 6.0f) return 7u;
  if (v >= 4.0f) return 6u;
  if (v >= 3.0f) return 5u;
  if (v >= 2.0f) return 4u;
  return (uint32_t)(v * 2.0f);  // 0, 1, 2, 3
}

// Eight E2M1 codes (low nibble first) times the power of two of `scale`: exact in bf16 for every scale byte up to 252
// (checked on MI355X for every code; the conversion reads the scale's exponent field alone, so byte 0 is 2^-127 and
// byte 255 gives NaN).  Bytes 253 and 254 make weights of 2^128 and more, which bf16 cannot hold.
__device__ __forceinline__ bf16x8 fp4_bf16x8(uint32_t w, float scale) {
  const bf16x2 a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale, 0);
  const bf16x2 b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale, 1);
  const bf16x2 c = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale, 2);
  const bf16x2 d = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w, scale, 3);
  return bf16x8{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
}
__device__ __forceinline__ float e8m0_f32(uint32_t byte) { return __uint_as_float(byte << 23); }
// Scale bytes 253 and 254: sums that meet one are taken again in two parts, first these scale blocks alone at a quarter of
// their scale (then their weights fit), and on four times those sums all other blocks, exactly as they are.  part_codes
// clears the codes of the blocks that do not belong to a part.
__device__ __forceinline__ bool huge_scale(uint32_t byte) { return byte - 253u <= 1u; }
__device__ __forceinline__ uint4 part_codes(uint4 w, uint32_t byte, bool huge) {
  const uint32_t keep = huge_scale(byte) == huge ? 0xFFFFFFFFu : 0u;
  return make_uint4(w.x & keep, w.y & keep, w.z & keep, w.w & keep);
}
__device__ __forceinline__ float part_scale(uint32_t byte, bool huge) { return e8m0_f32(byte) * (huge ? 0.25f : 1.0f); }

// ------------------------------------------------------------------ E4M3 (activation hi/lo split)
// E8M0 exponent X for an E4M3 block with maximum magnitude amax: amax / 2^X in (224, 448].
__device__ __forceinline__ int fp8_block_exp(float amax) {
  if (amax == 0.0f) return 0;
  uint32_t u = __float_as_uint(amax);
  int E = (int)((u >> 23) & 0xFF);
  int e = E == 0 ? -127 : E - 127;
  int X = (u & 0x7FFFFFu) > 0x600000u ? e - 7 : e - 8;
  return X < -127 ? -127 : (X > 127 ? 127 : X);
}
__device__ __forceinline__ float exp2i(int X) {   // 2^X for -127 <= X <= 127, exact
  return X >= -126 ? __uint_as_float((uint32_t)(X + 127) << 23) : __uint_as_float(0x00400000u);
}
// Two E4M3 codes (bits 0-7 and 8-15) of values already divided by their block scale (|y| <= 448) from the
// hardware conversion (OCP E4M3, round to nearest even, checked against the oracle on every bf16 input; a NaN or an
// infinity gives the E4M3 NaN), with the sign of zero codes cleared.
__device__ __forceinline__ uint32_t e4m3_pack2(float y0, float y1) {
  const uint32_t w = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(y0, y1, 0, false) & 0xFFFFu;
  const uint32_t t = w & 0x7F7Fu;
  return t | (w & ((t + 0x7F7Fu) & 0x8080u));   // bit 7 of each byte kept only where the magnitude is nonzero
}
typedef float v2f __attribute__((ext_vector_type(2)));
__device__ __forceinline__ v2f e4m3_unpack2(uint32_t w) { return __builtin_amdgcn_cvt_pk_f32_fp8((int)w, false); }

// ------------------------------------------------------------------ the specified sigmoid
// exp(x) for |x| <= 200: Cody-Waite reduction by ln 2 (fdlibm split) and a degree-13 Taylor polynomial in
// Horner form, every step one correctly rounded IEEE double operation (no contraction), so the result is
// reproducible bit for bit on any IEEE platform that evaluates the same sequence.
__device__ __forceinline__ double exp_spec(double x) {
#pragma clang fp contract(off)
  const double LN2_HI = 0x1.62e42feep-1;
  const double LN2_LO = 0x1.a39ef35793c76p-33;
  const double INV_LN2 = 0x1.71547652b82fep+0;
  double n = __builtin_rint(x * INV_LN2);
  double r = (x - n * LN2_HI) - n * LN2_LO;
  double p = 1.0 / 6227020800.0;             // 1/13!
  p = p * r + 1.0 / 479001600.0;             // 1/12!
  p = p * r + 1.0 / 39916800.0;
  p = p * r + 1.0 / 3628800.0;
  p = p * r + 1.0 / 362880.0;
  p = p * r + 1.0 / 40320.0;
  p = p * r + 1.0 / 5040.0;
  p = p * r + 1.0 / 720.0;
  p = p * r + 1.0 / 120.0;
  p = p * r + 1.0 / 24.0;
  p = p * r + 1.0 / 6.0;
  p = p * r + 0.5;
  p = p * r + 1.0;
  p = p * r + 1.0;
  return __builtin_ldexp(p, (int)n);
}
// fp32 sigmoid = fp32(1 / (1 + exp_spec(-x))), input clamped to [-200, 200]; NaN -> canonical quiet NaN.
// Branch-free, so that independent evaluations interleave.
__device__ __forceinline__ float sigmoid_spec(float xf) {
#pragma clang fp contract(off)
  const bool nan = xf != xf;
  double x = nan ? 0.0 : (double)xf;
  x = x < -200.0 ? -200.0 : x;
  x = x > 200.0 ? 200.0 : x;
  const double e = exp_spec(-x);
  float s = (float)(1.0 / (1.0 + e));
  asm volatile("" : "+v"(s));   // evaluated for every lane: keeps the compiler from branching around it
  return nan ? __uint_as_float(0x7FC00000u) : s;
}

// round_bf16(sigmoid_spec(x)) for a bf16 x, through the hardware exponential and reciprocal: their fp32 result is within
// 8 units of its last place (x log2 e split so that its fraction is exact to the last bits; 1 ulp each from v_exp_f32,
// the addition and v_rcp_f32), so it rounds to the same bf16 unless it lies that close to the middle between two; those,
// and arguments past 80, take the specified evaluation (some 1,000 cycles of dependent fp64).
__device__ __forceinline__ float sigmoid_bf16(float x) {
#pragma clang fp contract(off)
  constexpr float kHi = 0x1.714p+0f, kLo = 0x1.47652b8p-12f;   // log2 e: 13 bits (times 8 of x: exact), the rest
  const float t = -x * kHi;
  const float n = __builtin_rintf(t);
  const float f = (t - n) - x * kLo;
  const float e = __builtin_ldexpf(__builtin_amdgcn_exp2f(f), (int)n);
  const float s = __builtin_amdgcn_rcpf(1.0f + e);
  const int off = (int)(__float_as_uint(s) & 0xFFFFu) - 0x8000;
  const bool sure = fabsf(x) <= 80.0f && (off > 32 || off < -32);
  if (sure) return round_bf16(s);
  return round_bf16(sigmoid_spec(x));
}

// 32 bf16-valued floats -> hi / lo E4M3 words (4 codes per word, element order) and E8M0 bytes: hi = E4M3 block
// quantisation of v, lo = the same of the exact residual v - hi.  Codes from the hardware conversion
// (v_cvt_pk_fp8_f32: OCP E4M3, round to nearest even, checked against the oracle on every bf16 input;
// e4m3_pack2 clears the sign of zero codes); the scalings by 2^-X and 2^-Y are exact, and the residual is one
// fused multiply-add (exact, with no overflow of the product for the largest blocks).
__device__ __forceinline__ void quant_block_fp8_hilo(const float* v, uint32_t* hw, uint32_t* lw, uint8_t* hsb,
                                                        uint8_t* lsb) {
  float amax = 0.0f;
#pragma unroll
  for (int j = 0; j < 32; ++j) amax = fmaxf(amax, fabsf(v[j]));
  const int X = fp8_block_exp(amax);
  const float sx = exp2i(-X), dx = exp2i(X);
  float r[32];
  float ramax = 0.0f;
#pragma unroll
  for (int w = 0; w < 8; ++w) {
    const uint32_t c01 = e4m3_pack2(v[4 * w] * sx, v[4 * w + 1] * sx);
    const uint32_t c23 = e4m3_pack2(v[4 * w + 2] * sx, v[4 * w + 3] * sx);
    hw[w] = c01 | (c23 << 16);
    const v2f d01 = e4m3_unpack2(c01), d23 = e4m3_unpack2(c23);
    r[4 * w] = __builtin_fmaf(-d01.x, dx, v[4 * w]);          // exact residuals, no overflow of the product
    r[4 * w + 1] = __builtin_fmaf(-d01.y, dx, v[4 * w + 1]);
    r[4 * w + 2] = __builtin_fmaf(-d23.x, dx, v[4 * w + 2]);
    r[4 * w + 3] = __builtin_fmaf(-d23.y, dx, v[4 * w + 3]);
#pragma unroll
    for (int j = 0; j < 4; ++j) ramax = fmaxf(ramax, fabsf(r[4 * w + j]));
  }
  const int Y = fp8_block_exp(ramax);
  const float sy = exp2i(-Y);
#pragma unroll
  for (int w = 0; w < 8; ++w)
    lw[w] = e4m3_pack2(r[4 * w] * sy, r[4 * w + 1] * sy) | (e4m3_pack2(r[4 * w + 2] * sy, r[4 * w + 3] * sy) << 16);
  *hsb = (uint8_t)(X + 127);
  *lsb = (uint8_t)(Y + 127);
}

// ------------------------------------------------------------------ wave reductions (wave64)
// wave64 sum through DPP row operations (xor 1, xor 2, half-row and row mirrors, then row_bcast15 / 31 into
// rows 1-3); the total is read from lane 63 and returned to every lane
__device__ __forceinline__ float dpp_sum_f32(float v) {
  v = v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, false));
  v = v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, false));
  v = v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xF, 0xF, false));
  v = v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xF, 0xF, false));
  v = v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x142, 0xA, 0xF, false));
  v = v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x143, 0xC, 0xF, false));
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

// wave64 max / min of a uint32 through DPP row operations (xor 1, xor 2, half-row and row mirrors, then the
// row_bcast15 / row_bcast31 steps across rows); every lane receives the result read from lane 63.
__device__ __forceinline__ uint32_t dpp_max_u32(uint32_t v) {
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0xB1, 0xF, 0xF, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x4E, 0xF, 0xF, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x141, 0xF, 0xF, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x140, 0xF, 0xF, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x142, 0xA, 0xF, false));
  v = max(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x143, 0xC, 0xF, false));
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
__device__ __forceinline__ uint32_t dpp_min_u32(uint32_t v) {
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0xB1, 0xF, 0xF, false));
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x4E, 0xF, 0xF, false));
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x141, 0xF, 0xF, false));
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x140, 0xF, 0xF, false));
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x142, 0xA, 0xF, false));
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp((int)v, (int)v, 0x143, 0xC, 0xF, false));
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// order-preserving map of an fp32 key to uint32 (NaN lowest, -0 treated as +0)
__device__ __forceinline__ uint32_t key_to_ordered(float k) {
  const uint32_t u = __float_as_uint(k == 0.0f ? 0.0f : k);
  const uint32_t o = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
  return k != k ? 0u : o;
}

// ------------------------------------------------------------------ global -> LDS copies
// global_load_lds: lane l's 16 (or 4) bytes at gbase + voff land at lds_dst + 16 l (or 4 l), without passing
// through registers.  gbase and lds_dst must be wave-uniform (they go to SGPRs and M0).  Issued from inline
// assembly so that the compiler's wait-counter bookkeeping does not pin the address registers (it would wait
// for every outstanding load before reusing them); the caller waits with wait_vm_all() before any wave reads
// the data.  M0 is only a launch-time scratch register on gfx950 (ordinary LDS instructions do not use it).
__device__ __forceinline__ uint64_t uniform_u64(uint64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return ((uint64_t)hi << 32) | lo;
}
// The LDS byte offset of a pointer into LDS: the low 32 bits of its generic address (the LDS aperture puts the
// offset there).  No address-space cast: its null check, folded against the aperture base in divergent code,
// made the gfx950 backend emit an invalid compare.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
  return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)p);
}
// The base address operands of these copies are SGPRs that are often written by v_readfirstlane just before
// the asm; a VMEM instruction reading an SGPR that a VALU instruction wrote needs 5 wait states, which the
// compiler does not supply inside inline assembly: each asm starts with them (s_nop 4 = 5 wait states).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"     // M0 is declared clobbered on purpose
__device__ __forceinline__ void lds_copy16(const void* gbase, uint32_t voff, const void* lds_dst) {
  const uint64_t b = uniform_u64((uint64_t)gbase);
  const uint32_t m = lds_addr(lds_dst);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(b), "s"(m)
               : "memory", "m0");
}
__device__ __forceinline__ void lds_copy4(const void* gbase, uint32_t voff, const void* lds_dst) {
  const uint64_t b = uniform_u64((uint64_t)gbase);
  const uint32_t m = lds_addr(lds_dst);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 4\n\tglobal_load_lds_dword %0, %1" ::"v"(voff), "s"(b), "s"(m)
               : "memory", "m0");
}
#pragma clang diagnostic pop
// s_waitcnt vmcnt(0) (expcnt and lgkmcnt left at their maxima): every global load of the wave has landed,
// including the global -> LDS copies above
__device__ __forceinline__ void wait_vm_all() { __builtin_amdgcn_s_waitcnt(0x0F70); }
// s_waitcnt vmcnt(N): at most the N most recent vector memory loads still in flight (loads, including the LDS
// copies above, complete in issue order, so everything issued before them has landed)
__host__ __device__ constexpr int vm_keep(int n) { return (n & 15) | (7 << 4) | (15 << 8) | (((n >> 4) & 3) << 14); }
template <int N>
__device__ __forceinline__ void wait_vm_keep() {
  static_assert(N >= 0 && N < 64, "vmcnt holds 6 bits");
  __builtin_amdgcn_s_waitcnt(vm_keep(N));
}

}  // namespace mimo
