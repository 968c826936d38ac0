// libosmos MI355X - the f16 matmul's weight decode straight from global memory into the matrix cores' A operand (mm.hip's
// direct kernels), for Q4_0, Q3_K, Q4_K, IQ1_S, IQ1_M, IQ2_XXS and IQ3_XXS.
//
// A wave decodes a 16-row tile's 256-value block: lane l holds row l % 16, and lane group q = l / 16 the chunks
// (8 values) 4 g + q of the block's 32-value groups g - v_mfma_f32_16x16x32_f16's A slots, one group a step. Raw<T>::load
// only loads: 16 bytes a lane where the type allows, a row's four lane groups side by side, so that a load instruction
// touches each row's line once (8-byte pieces, five instructions a Q4_K block, streamed 4.2 TB/s; 16-byte pieces and a
// 4-byte header word 6.1). head() hands the words round between the lane groups (v_permlane16_swap, v_permlane32_swap)
// and decodes the block's fields; step() gives the 8 f16 of one step.
//
// The values are decode.h's, rounded to f16 (nearest even): exact F32 scales and products, then one conversion. (A group's
// scale is d times an odd whole number, 2 s + 1, never s d + d / 2, which is no number where d is infinite and s is 0.) What an
// instruction costs chose the forms (measured, cycles a wave64 instruction): v_fma_mixlo/hi_f16 9, permlane swaps 8.3,
// fma, conversions, perm, bfi and packed f16 4.5, F32 mul / add, shifts and logic 2.6. No asm holds an instruction: the
// compiler does not see into asm, and a VALU write needs idle states before a matrix instruction reads it.
#pragma once
#include <type_traits>

#include "decode.h"

namespace osm {
namespace mm {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// words at the blocks' 2-byte alignment
struct __attribute__((packed, aligned(2))) W1 { uint32_t x; };
struct __attribute__((packed, aligned(2))) W2 { uint32_t x, y; };
struct __attribute__((packed, aligned(2))) W4 { uint32_t x, y, z, w; };

// exchanges between the lane groups q = 2 b1 + b0: swap1 trades lane bit b1 for the slot (a: slot 0, b: slot 1), swap0
// lane bit b0
__device__ inline void swap1(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0], b = r[1];
}
__device__ inline void swap0(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0], b = r[1];
}
// lane group s's x to every lane group, as o[s]
__device__ inline void spread4(uint32_t x, uint32_t* o) {
  uint32_t e = x, f = x;
  swap0(e, f);  // e: (x0 x0 x2 x2), f: (x1 x1 x3 x3)
  o[0] = e, o[2] = e, o[1] = f, o[3] = f;
  swap1(o[0], o[2]), swap1(o[1], o[3]);
}
// lane group s's t[q] to lane group q's t[s]
__device__ inline void turn4(uint32_t* t) { swap1(t[0], t[2]), swap1(t[1], t[3]), swap0(t[0], t[1]), swap0(t[2], t[3]); }

__device__ inline uint32_t pk16(float a, float b) {  // (the two conversions one instruction)
  const half2v h = {(_Float16) a, (_Float16) b};
  return __builtin_bit_cast(uint32_t, h);
}
__device__ inline uint32_t pk16x2(float a) {
  asm("" : "+v"(a));
  return pk16(a, a);
}
// byte codes 0, 1 (hi: 2, 3) of w as an f16 pair plus c: 0x6400 | code is 1024 + code
__device__ inline half2v code_pair(uint32_t w, int hi, half2v c) {
  return __builtin_bit_cast(half2v, __builtin_amdgcn_perm(0x64646464u, w, hi ? 0x07030602u : 0x05010400u)) + c;
}
// 4 f16 pairs times an F32 scale, the products exact in F32, rounded once: the mixed fma to F32 (plus -0, so that a -0
// product stays -0) and the packed conversion, or (Mixed) the mixed fma to f16
template <bool Mixed = false>
__device__ inline half8 scaled8(float s, const uint32_t* w) {
  float z = -0.0f;
  asm("" : "+s"(z));
  half8 o;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const half2v g = __builtin_bit_cast(half2v, w[i]);
    float a = __builtin_fmaf(s, (float) g[0], z), b = __builtin_fmaf(s, (float) g[1], z);
    if constexpr (!Mixed) asm("" : "+v"(a), "+v"(b));  // (held in F32: the f16 mixed fma is the slower)
    o[2 * i] = (_Float16) a, o[2 * i + 1] = (_Float16) b;
  }
  return o;
}
__device__ inline half8 cat4(half2v a, half2v b, half2v c, half2v d) { return half8{a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1]}; }
// 8 f16 of three (v01: two, v2: the third) by a codebook entry's byte selectors
__device__ inline half8 pick8(uint32_t v01, uint32_t v2, uint4 sel) {
  return __builtin_bit_cast(half8, u32x4{__builtin_amdgcn_perm(v2, v01, sel.x), __builtin_amdgcn_perm(v2, v01, sel.y),
                                         __builtin_amdgcn_perm(v2, v01, sel.z), __builtin_amdgcn_perm(v2, v01, sel.w)});
}
// a 7-bit sign index's 8 signs (the eighth their parity) at bits 0 .. 7 and at 15 .. 22: values 2i and 2i + 1's 16 apart
__device__ inline uint32_t sign_word(uint32_t s7) {
  const uint32_t s8 = (uint32_t) __builtin_popcount(s7) << 7 | s7;  // (the bits past 7 meet no other)
  return s8 << 15 | s8;
}
// values 2i and 2i + 1's signs on a pair of non-negative f16
__device__ inline uint32_t signed_pair(uint32_t sw, int i, uint32_t g) {
  return ((sw << (15 - 2 * i)) & 0x80008000u) | (g & 0x7FFF7FFFu);
}

// ---- the codebooks as the steps read them, copied to LDS: IQ3_XXS's entries as f16; IQ2_XXS's and IQ1's as pick8's
// selectors, two bytes a value (2 c, 2 c + 1 for the value's place c among the three) ----
constexpr uint16_t half_bits(uint32_t n) {  // a small positive integer's f16 bits
  int e = 0;
  while ((n >> (e + 1)) != 0) e++;
  return (uint16_t) ((15 + e) << 10 | ((n << (10 - e)) & 0x3FFu));
}
constexpr uint32_t selectors(uint64_t entry, int pair, uint32_t m0, uint32_t m1) {
  uint32_t r = 0;
  for (int v = 0; v < 2; v++) {
    const uint32_t b = (uint32_t) (entry >> (8 * (2 * pair + v))) & 0xFF, c = b == m0 ? 0 : b == m1 ? 1 : 2;
    r |= (2 * c | (2 * c + 1) << 8) << (16 * v);
  }
  return r;
}
struct alignas(16) StepTabs {
  uint32_t iq2xxs[256][4], iq1[2048][4];
  uint16_t iq3xxs[256][4];
};
constexpr StepTabs make_step_tabs() {
  const Grids g = make_grids();
  StepTabs t{};
  for (int i = 0; i < 256; i++)
    for (int j = 0; j < 4; j++) {
      t.iq2xxs[i][j] = selectors(g.iq2xxs[i], j, 0x08, 0x19);
      t.iq3xxs[i][j] = half_bits((g.iq3xxs[i] >> (8 * j)) & 0xFF);
    }
  for (int i = 0; i < 2048; i++)
    for (int j = 0; j < 4; j++) t.iq1[i][j] = selectors(g.iq1s[i], j, 0xFF, 0x00);
  return t;
}
__constant__ StepTabs kStepTabs = make_step_tabs();

template <uint32_t T> struct Tab { static constexpr bool kSome = false; };
template <> struct Tab<kIQ2_XXS> { static constexpr bool kSome = true; uint4 g[256]; };
template <> struct Tab<kIQ3_XXS> { static constexpr bool kSome = true; uint2 g[256]; };
template <> struct Tab<kIQ1_S> { static constexpr bool kSome = true; uint4 g[2048]; };
template <> struct Tab<kIQ1_M> { static constexpr bool kSome = true; uint4 g[2048]; };
template <uint32_t T>
__device__ inline void fill_step_tab(Tab<T>& t) {  // every thread of the workgroup
  if constexpr (Tab<T>::kSome) {
    const void* src = T == kIQ2_XXS ? (const void*) kStepTabs.iq2xxs : T == kIQ3_XXS ? (const void*) kStepTabs.iq3xxs
                                                                                      : (const void*) kStepTabs.iq1;
    for (uint32_t i = threadIdx.x; i < sizeof t.g / 16; i += blockDim.x) ((u32x4*) t.g)[i] = ((const u32x4*) src)[i];
  }
}

// ---- per type: SL, W the K split (mm.hip's), NP = 256 / SL the partitions of a block; R a lane's loaded words, H its
// decoded fields, for NPW of the block's partitions from pw (kPart: those alone; else the whole block whatever NPW).
// step's j: the partition - kPart: of the wave's, else of the block - and s its step of 32 values ----
template <uint32_t T> struct Raw;
// Q4_K: lane group q loads header word q and, of a whole block, group pair q's 32 bytes (four 8-byte units: unit u is what
// lane group u decodes); of half a block 16 bytes
template <> struct Raw<kQ4_K> {
  static constexpr int SL = 32, W = 16, NP = 8;
  static constexpr bool kPart = true;
  template <int NPW> struct R { uint32_t h; uint32_t n[NPW]; };
  template <int NPW> __device__ static void load(R<NPW>& r, const uint8_t* b, int pw, int q) {
    r.h = gload<W1>(b + 4 * q).x;
    if constexpr (NPW == 8) {
      const W4 u = gload<W4>(b + 16 + 32 * q), v = gload<W4>(b + 32 + 32 * q);
      r.n[0] = u.x, r.n[1] = u.y, r.n[2] = u.z, r.n[3] = u.w, r.n[4] = v.x, r.n[5] = v.y, r.n[6] = v.z, r.n[7] = v.w;
    } else {
      static_assert(NPW == 4, "a whole block or half of one");
      const W4 u = gload<W4>(b + 16 + 16 * pw + 32 * (q & 1) + 16 * (q >> 1));
      r.n[0] = u.x, r.n[1] = u.y, r.n[2] = u.z, r.n[3] = u.w;
    }
  }
  template <int NPW> struct H { uint32_t sc[2], mn[2]; float d, m; uint32_t n[NPW]; };
  template <int NPW> __device__ static void head(H<NPW>& h, const R<NPW>& r, int pw, int q) {
    uint32_t hd[4];
    spread4(r.h, hd);
#pragma unroll
    for (int i = 0; i < NPW; i++) h.n[i] = r.n[i];
    if constexpr (NPW == 8) {  // lane: pair q, slots the four 8-byte units -> lane: unit q, slots the pairs
      swap1(h.n[0], h.n[4]), swap1(h.n[1], h.n[5]), swap1(h.n[2], h.n[6]), swap1(h.n[3], h.n[7]);
      swap0(h.n[0], h.n[2]), swap0(h.n[1], h.n[3]), swap0(h.n[4], h.n[6]), swap0(h.n[5], h.n[7]);
    } else {
      swap0(h.n[0], h.n[2]), swap0(h.n[1], h.n[3]);
    }
    h.sc[0] = hd[1] & 0x3F3F3F3Fu, h.mn[0] = hd[2] & 0x3F3F3F3Fu;
    h.sc[1] = (hd[3] & 0x0F0F0F0Fu) | ((hd[1] >> 2) & 0x30303030u);
    h.mn[1] = ((hd[3] >> 4) & 0x0F0F0F0Fu) | ((hd[2] >> 2) & 0x30303030u);
    h.d = f16(hd[0] & 0xFFFF), h.m = f16(hd[0] >> 16);
    if constexpr (NPW < 8) {  // (uniform) the wave's groups to the low bytes
      const int sel = pw >> 2, sh = 8 * (pw & 3);
      h.sc[0] = (sel ? h.sc[1] : h.sc[0]) >> sh, h.mn[0] = (sel ? h.mn[1] : h.mn[0]) >> sh;
    }
  }
  template <int NPW> __device__ static half8 step(const H<NPW>& h, const Tab<kQ4_K>&, int j, int s, int q) {
    const float S = mul(h.d, (float) ((h.sc[j / 4] >> (8 * (j % 4))) & 0xFF)), M = mul(h.m, (float) ((h.mn[j / 4] >> (8 * (j % 4))) & 0xFF));
    const uint32_t nx = h.n[2 * (j / 2)], ny = h.n[2 * (j / 2) + 1];
    uint32_t a = (j & 1 ? nx >> 4 : nx) & 0x0F0F0F0Fu, c = (j & 1 ? ny >> 4 : ny) & 0x0F0F0F0Fu;
    asm("" : "+v"(a), "+v"(c));  // (masked bytes: v_cvt_f32_ubyte each)
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
      v[i] = __builtin_fmaf(S, (float) (((i < 4 ? a : c) >> (8 * (i % 4))) & 0xFF), -M);
      asm("" : "+v"(v[i]));  // (rounded to f32 before its f16: not one mixed fma)
    }
    return __builtin_bit_cast(half8, u32x4{pk16(v[0], v[1]), pk16(v[2], v[3]), pk16(v[4], v[5]), pk16(v[6], v[7])});
  }
};
// Q4_0, 8 blocks of 18 bytes: lane group q loads blocks 2q and 2q + 1 (36 bytes). d (q - 8) in packed f16: the code less 8
// and its product with d are exact before the one rounding
template <> struct Raw<kQ4_0> {
  static constexpr int SL = 64, W = 4, NP = 4;
  static constexpr bool kPart = false;
  template <int NPW> struct R { uint32_t n[9]; };
  template <int NPW> __device__ static void load(R<NPW>& r, const uint8_t* b, int pw, int q) {
    const W4 u = gload<W4>(b + 36 * q), v = gload<W4>(b + 36 * q + 16);
    r.n[0] = u.x, r.n[1] = u.y, r.n[2] = u.z, r.n[3] = u.w, r.n[4] = v.x, r.n[5] = v.y, r.n[6] = v.z, r.n[7] = v.w;
    r.n[8] = gload<W1>(b + 36 * q + 32).x;
  }
  template <int NPW> struct H { uint32_t n[16], d[4]; };
  template <int NPW> __device__ static void head(H<NPW>& h, const R<NPW>& r, int pw, int q) {
    auto al = [](uint32_t hi, uint32_t lo) { return __builtin_amdgcn_alignbit(hi, lo, 16); };
    uint32_t u0[4] = {al(r.n[1], r.n[0]), al(r.n[2], r.n[1]), r.n[5], r.n[6]};  // unit 0 of the lane's two blocks
    uint32_t u1[4] = {al(r.n[3], r.n[2]), al(r.n[4], r.n[3]), r.n[7], r.n[8]};
#pragma unroll
    for (int i = 0; i < 4; i++) swap0(u0[i], u1[i]);  // lane (s1, unit), slots s0
#pragma unroll
    for (int i = 0; i < 4; i++) {
      uint32_t a = u0[i], b = u0[i], c = u1[i], d = u1[i];
      swap1(a, b), swap1(c, d);  // a: s = 0, c: s = 1, b: s = 2, d: s = 3
      h.n[i] = a, h.n[4 + i] = c, h.n[8 + i] = b, h.n[12 + i] = d;
    }
    spread4((r.n[0] & 0xFFFFu) | (r.n[4] & 0xFFFF0000u), h.d);
  }
  template <int NPW> __device__ static half8 step(const H<NPW>& h, const Tab<kQ4_0>&, int j, int s, int q) {
    const int g = 2 * j + s, sh = 4 * (q >> 1);
    const uint32_t a = (h.n[2 * g] >> sh) & 0x0F0F0F0Fu, c = (h.n[2 * g + 1] >> sh) & 0x0F0F0F0Fu;
    const uint32_t dp = __builtin_amdgcn_perm(h.d[g / 2], h.d[g / 2], g & 1 ? 0x03020302u : 0x01000100u);
    const half2v d = __builtin_bit_cast(half2v, dp), off = {(_Float16) -1032.0f, (_Float16) -1032.0f};
    return cat4(code_pair(a, 0, off) * d, code_pair(a, 1, off) * d, code_pair(c, 0, off) * d, code_pair(c, 1, off) * d);
  }
};
// Q3_K: lane group q = 2 b1 + b0 loads unit b1's pair of the codes' half b0, its own high bits, and word q of the scales
// (word 3: the last two bytes' d)
template <> struct Raw<kQ3_K> {
  static constexpr int SL = 64, W = 8, NP = 4;
  static constexpr bool kPart = false;
  template <int NPW> struct R { uint32_t n[4], hm[2], t; };
  template <int NPW> __device__ static void load(R<NPW>& r, const uint8_t* b, int pw, int q) {
    const W4 u = gload<W4>(b + 32 + 32 * (q & 1) + 16 * (q >> 1));
    const W2 v = gload<W2>(b + 8 * q);
    r.n[0] = u.x, r.n[1] = u.y, r.n[2] = u.z, r.n[3] = u.w, r.hm[0] = v.x, r.hm[1] = v.y;
    r.t = gload<W1>(b + 96 + 4 * q - (q == 3 ? 2 : 0)).x;  // (group 3: the last scale bytes again and d)
  }
  template <int NPW> struct H { uint32_t n[4], hm[2], t[3]; float d; };
  template <int NPW> __device__ static void head(H<NPW>& h, const R<NPW>& r, int pw, int q) {
#pragma unroll
    for (int i = 0; i < 4; i++) h.n[i] = r.n[i];
    swap0(h.n[0], h.n[2]), swap0(h.n[1], h.n[3]);
    h.hm[0] = r.hm[0], h.hm[1] = r.hm[1];
    uint32_t t[4];
    spread4(r.t, t);
    const int sh = 8 * (q >> 1);
    h.t[0] = t[0] >> sh, h.t[1] = t[1] >> sh, h.t[2] = t[2] >> sh, h.d = f16(t[3] >> 16);
  }
  template <int NPW> __device__ static half8 step(const H<NPW>& h, const Tab<kQ3_K>&, int j, int s, int q) {
    const int g = 2 * j + s;
    const uint32_t lo = (h.t[(g & 3) >> 1] >> (16 * (g & 1) + 4 * (g >> 2))) & 15u, hi = (h.t[2] >> (16 * (g & 1) + 2 * (g >> 1))) & 3u;
    const float S = mul(h.d, (float) ((int) (lo | hi << 4) - 32));
    const half2v off = {(_Float16) -1028.0f, (_Float16) -1028.0f};
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const uint32_t c = ((h.n[2 * (g >> 2) + i] >> (2 * (g & 3))) & 0x03030303u) | ((h.hm[i] >> g) & 0x01010101u) << 2;
      o[2 * i] = __builtin_bit_cast(uint32_t, code_pair(c, 0, off)), o[2 * i + 1] = __builtin_bit_cast(uint32_t, code_pair(c, 1, off));
    }
    return scaled8(S, o);
  }
};
// IQ2_XXS: lane group q loads groups 2q and 2q + 1 (16 bytes); the index bytes go to the groups that read them, the sign
// and scale words to all. an f16 value is one of the group's three magnitudes with its sign
template <> struct Raw<kIQ2_XXS> {
  static constexpr int SL = 128, W = 4, NP = 2;
  static constexpr bool kPart = false;
  template <int NPW> struct R { uint32_t n[4]; uint16_t d; };
  template <int NPW> __device__ static void load(R<NPW>& r, const uint8_t* b, int pw, int q) {
    const W4 u = gload<W4>(b + 2 + 16 * q);
    r.n[0] = u.x, r.n[1] = u.y, r.n[2] = u.z, r.n[3] = u.w, r.d = gload<uint16_t>(b);
  }
  template <int NPW> struct H { uint32_t t[4], a[8]; float d; };
  template <int NPW> __device__ static void head(H<NPW>& h, const R<NPW>& r, int pw, int q) {
    constexpr uint32_t sel[4] = {0x0C0C0400u, 0x0C0C0501u, 0x0C0C0602u, 0x0C0C0703u};
#pragma unroll
    for (int i = 0; i < 4; i++) h.t[i] = __builtin_amdgcn_perm(r.n[2], r.n[0], sel[i]);
    turn4(h.t);
    const uint32_t flip = r.d & 0x8000u ? 0x0FFFFFFFu : 0u;  // (a negative scale: every sign the other way, |d| below)
    uint32_t x[4], y[4];
    spread4(r.n[1] ^ flip, x), spread4(r.n[3] ^ flip, y);
#pragma unroll
    for (int i = 0; i < 4; i++) h.a[2 * i] = x[i], h.a[2 * i + 1] = y[i];
    h.d = 0.125f * f16(r.d & 0x7FFFu);
  }
  template <int NPW> __device__ static half8 step(const H<NPW>& h, const Tab<kIQ2_XXS>& tab, int j, int s, int q) {
    const int g = 4 * j + s;
    const uint4 v = tab.g[(h.t[g / 2] >> (8 * (g & 1))) & 255u];
    const float S = mul(h.d, (float) (h.a[g] >> 27 | 1u));  // (2 s + 1: the top four bits over a one)
    const uint32_t sw = sign_word(__builtin_amdgcn_ubfe(h.a[g], 7 * q, 7));
    // the group's three magnitudes, picked by the entry's selectors
    const uint32_t v01 = pk16(mul(S, 8.0f), mul(S, 25.0f)), v2 = pk16x2(mul(S, 43.0f));
    const u32x4 p = __builtin_bit_cast(u32x4, pick8(v01, v2, v));
    return __builtin_bit_cast(half8, u32x4{signed_pair(sw, 0, p[0]), signed_pair(sw, 1, p[1]), signed_pair(sw, 2, p[2]),
                                           signed_pair(sw, 3, p[3])});
  }
};
// IQ3_XXS: as IQ2_XXS with two index bytes a chunk; the f16 grid entries times the F32 scale
template <> struct Raw<kIQ3_XXS> {
  static constexpr int SL = 128, W = 8, NP = 2;
  static constexpr bool kPart = false;
  template <int NPW> struct R { uint32_t n[4], a[2]; uint16_t d; };
  template <int NPW> __device__ static void load(R<NPW>& r, const uint8_t* b, int pw, int q) {
    const W4 u = gload<W4>(b + 2 + 16 * q);
    const W2 v = gload<W2>(b + 66 + 8 * q);
    r.n[0] = u.x, r.n[1] = u.y, r.n[2] = u.z, r.n[3] = u.w, r.a[0] = v.x, r.a[1] = v.y, r.d = gload<uint16_t>(b);
  }
  template <int NPW> struct H { uint32_t t[4], a[8]; float d; };
  template <int NPW> __device__ static void head(H<NPW>& h, const R<NPW>& r, int pw, int q) {
    h.t[0] = __builtin_amdgcn_perm(r.n[2], r.n[0], 0x05040100u), h.t[1] = __builtin_amdgcn_perm(r.n[2], r.n[0], 0x07060302u);
    h.t[2] = __builtin_amdgcn_perm(r.n[3], r.n[1], 0x05040100u), h.t[3] = __builtin_amdgcn_perm(r.n[3], r.n[1], 0x07060302u);
    turn4(h.t);
    const uint32_t flip = r.d & 0x8000u ? 0x0FFFFFFFu : 0u;
    uint32_t x[4], y[4];
    spread4(r.a[0] ^ flip, x), spread4(r.a[1] ^ flip, y);
#pragma unroll
    for (int i = 0; i < 4; i++) h.a[2 * i] = x[i], h.a[2 * i + 1] = y[i];
    h.d = 0.25f * f16(r.d & 0x7FFFu);
  }
  template <int NPW> __device__ static half8 step(const H<NPW>& h, const Tab<kIQ3_XXS>& tab, int j, int s, int q) {
    const int g = 4 * j + s;
    const uint2 v0 = tab.g[(h.t[g / 2] >> (16 * (g & 1))) & 255u], v1 = tab.g[(h.t[g / 2] >> (16 * (g & 1) + 8)) & 255u];
    const float S = mul(h.d, (float) (h.a[g] >> 27 | 1u));  // (2 s + 1: the top four bits over a one)
    const uint32_t sw = sign_word(__builtin_amdgcn_ubfe(h.a[g], 7 * q, 7));
    const uint32_t w[4] = {v0.x, v0.y, v1.x, v1.y};
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; i++) o[i] = signed_pair(sw, i, w[i]);
    return scaled8(S, o);
  }
};
// the IQ1 types' three values of a group (the scale times -1, 0, 1 plus the delta), picked by the entry's selectors
__device__ inline half8 iq1_pick(float S, bool neg, uint4 sel) {
  const float v0 = mul(S, neg ? -1.125f : -0.875f), v1 = mul(S, neg ? -0.125f : 0.125f), v2 = mul(S, neg ? 0.875f : 1.125f);
  return pick8(pk16(v0, v1), pk16x2(v2), sel);
}
// IQ1_S: lane group q loads groups 2q and 2q + 1's index bytes and high words
template <> struct Raw<kIQ1_S> {
  static constexpr int SL = 128, W = 4, NP = 2;
  static constexpr bool kPart = false;
  template <int NPW> struct R { uint32_t n[2], h; uint16_t d; };
  template <int NPW> __device__ static void load(R<NPW>& r, const uint8_t* b, int pw, int q) {
    const W2 u = gload<W2>(b + 2 + 8 * q);
    r.n[0] = u.x, r.n[1] = u.y, r.h = gload<W1>(b + 34 + 4 * q).x, r.d = gload<uint16_t>(b);
  }
  template <int NPW> struct H { uint32_t t[4], h[4]; float d; };
  template <int NPW> __device__ static void head(H<NPW>& h, const R<NPW>& r, int pw, int q) {
    constexpr uint32_t sel[4] = {0x0C0C0400u, 0x0C0C0501u, 0x0C0C0602u, 0x0C0C0703u};
#pragma unroll
    for (int i = 0; i < 4; i++) h.t[i] = __builtin_amdgcn_perm(r.n[1], r.n[0], sel[i]);
    turn4(h.t);
    spread4(r.h, h.h);
    h.d = f16(r.d);
  }
  template <int NPW> __device__ static half8 step(const H<NPW>& h, const Tab<kIQ1_S>& tab, int j, int s, int q) {
    const int g = 4 * j + s, o = 16 * (g & 1);
    const uint32_t qh = h.h[g / 2];
    const uint32_t idx = ((h.t[g / 2] >> (8 * (g & 1))) & 255u) | __builtin_amdgcn_ubfe(qh, o + 3 * q, 3) << 8;
    const float S = mul(h.d, (float) (((qh >> (o + 11)) & 14u) | 1u));
    return iq1_pick(S, (qh >> (o + 15)) & 1u, tab.g[idx]);
  }
};
// IQ1_M: as IQ1_S with a nibble a chunk, and the scale words' (0, 1) or (2, 3) by the lane group's low bit
template <> struct Raw<kIQ1_M> {
  static constexpr int SL = 128, W = 4, NP = 2;
  static constexpr bool kPart = false;
  template <int NPW> struct R { uint32_t n[2], h, s; };
  template <int NPW> __device__ static void load(R<NPW>& r, const uint8_t* b, int pw, int q) {
    const W2 u = gload<W2>(b + 8 * q);
    r.n[0] = u.x, r.n[1] = u.y, r.h = gload<W1>(b + 32 + 4 * q).x, r.s = gload<W1>(b + 48 + 4 * (q & 1)).x;
  }
  template <int NPW> struct H { uint32_t t[4], h[4], s[2]; float d; };
  template <int NPW> __device__ static void head(H<NPW>& h, const R<NPW>& r, int pw, int q) {
    constexpr uint32_t sel[4] = {0x0C0C0400u, 0x0C0C0501u, 0x0C0C0602u, 0x0C0C0703u};
#pragma unroll
    for (int i = 0; i < 4; i++) h.t[i] = __builtin_amdgcn_perm(r.n[1], r.n[0], sel[i]);
    turn4(h.t);
    spread4(r.h, h.h);
    uint32_t e = r.s, f = r.s;
    swap0(e, f);
    h.d = f16(((e >> 12) & 15u) | ((e >> 28) << 4) | ((f >> 12) & 15u) << 8 | (f >> 28) << 12);
    const int sh = 3 * (q >> 1);  // (doubled: 2 s + 1 is what the steps read)
    h.s[0] = (e << 1) >> sh, h.s[1] = (f << 1) >> sh;
  }
  template <int NPW> __device__ static half8 step(const H<NPW>& h, const Tab<kIQ1_M>& tab, int j, int s, int q) {
    const int g = 4 * j + s;
    const uint32_t nib = __builtin_amdgcn_ubfe(h.h[g / 2], 16 * (g & 1) + 4 * q, 4);
    const uint32_t idx = ((h.t[g / 2] >> (8 * (g & 1))) & 255u) | (nib & 7u) << 8;
    const uint32_t sc = ((h.s[g >> 2] >> (16 * ((g >> 1) & 1) + 6 * (g & 1))) & 14u) | 1u;
    const float S = mul(h.d, (float) sc);
    return iq1_pick(S, nib & 8u, tab.g[idx]);
  }
};

}  // namespace mm
}  // namespace osm
