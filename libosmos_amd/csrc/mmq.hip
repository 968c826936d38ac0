// libosmos MI355X - the experts' matmul on the int8 matrix cores (include/osmos/gpu/mmq.h): mmq_x8_rows, mmq_group,
// mmq_known.
//
// contract (reference include/osmos/gpu/mmq.h:37-55, kernels/mmq.hip:33-151): activations int8 a 32-value group
// (dx = amax / 127, q = clamp(rint(x / dx)), sx = dx * sum q) in 16-slot tiles; Q4_K's 32-value group g of a weight row
// contributes (d sc) dx I - (dmin m) sx with I the group's exact integer dot, applied as v = (d sc) * dx;
// acc = fmaf(v, I, acc); acc = fmaf(dmin m, -sx, acc); K split into 4 partitions by 256-value block (partition p its
// blocks p, p + 4, ...), each its groups in order, then the partitions summed in order. every output the reference's
// bits, whatever the batch.
//
// CDNA4 mapping: one v_mfma_i32_16x16x32_i8 is exactly one group's 16 tokens x 16 rows of integer dots (K = 32 = the
// contract's group), so the epilogue applies per MFMA with no reassociation. a wave owns 16 rows and keeps the 4 K
// partitions' sums side by side in registers, for CT tiles of 16 tokens at a time; a workgroup is 4 such waves (64 rows)
// of one expert.
// the tokens are the A operand and the rows B: lane l is weight row l % 16, with the row's (d sc), (dmin m) of the group
// in its own registers, and its results are tokens 4 (l / 16) + i. so a lane needs 4 tokens' dx and sx a group, and they
// reach it as DPP operands (row_newbcast: a value of a lane of its row of 16) with no LDS read: the lane holds a
// float a tile and 64 slots of dx, and one of sx. what bounds it is the epilogue - mul, fma, fma and a conversion a
// result and group, 16 results an MFMA's 8 cycles - so a pass of at most 8 tokens spends it only on the results i that hold
// a token (the tokens of a tile are laid out over the lanes as 4 i + l / 16, so that 5 tokens are 2 results of 4).
#include "mmraw.h"

extern "C" {
#include "../../include/osmos/gpu/mmq.h"
}

namespace osm {
namespace mmq {

using mm::u32x4;
constexpr int kWaves = 4, kThreads = kWave * kWaves, kTile = 16, kBlockBytes = 144;
constexpr uint32_t kXWords = 256, kDWords = 32;  // 16-byte words of a tile's block: its x8, its dx (or sx)
typedef int v4i __attribute__((ext_vector_type(4)));
struct __attribute__((packed, aligned(4))) F4 { uint32_t x, y, z, w; };  // (dx and sx at a float's alignment)

// a half-wave a group: its 32 values' max |x| and the codes' sum by the half-wave's tree (reference kernels/mmq.hip:33-52)
__global__ __launch_bounds__(256) void x8_rows_kernel(const float* __restrict__ x, uint32_t xs,
                                                      const int32_t* __restrict__ idx, uint32_t slots, uint32_t cols,
                                                      int8_t* __restrict__ x8, float* __restrict__ dx,
                                                      float* __restrict__ sx) {
  const uint64_t i = (uint64_t) blockIdx.x * 256 + threadIdx.x;
  if (i >= (uint64_t) slots * cols) return;  // whole groups: slots * cols a multiple of 32, a half-wave's
  const uint32_t s = (uint32_t) (i / cols), c = (uint32_t) (i % cols);
  const int32_t r = idx[s];
  const float v = r >= 0 ? x[(uint64_t) r * xs + c] : 0.0f;
  float a = fabsf(v);
#pragma unroll
  for (int o = 16; o > 0; o >>= 1) a = fmaxf(a, __shfl_xor(a, o, 32));
  const float d = __fdiv_rn(a, 127.0f);
  const int q = a == 0.0f ? 0 : (int) fminf(fmaxf(rintf(__fdiv_rn(v, d)), -127.0f), 127.0f);
  int sum = q;
#pragma unroll
  for (int o = 16; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 32);
  x8[mmq_x8_at(s, c, cols)] = (int8_t) q;
  if (c % MMQ_GROUP == 0) {
    const uint64_t g = mmq_dx_at(s, c / MMQ_GROUP, cols / MMQ_GROUP);
    const float dd = a == 0.0f ? 0.0f : d;
    dx[g] = dd;
    sx[g] = __fmul_rn(dd, (float) sum);
  }
}

// the same with 4 lanes a group, 8 values a lane (two 16-byte loads of the token's row, one 8-byte store): for x rows
// 16-aligned. each value's code and the group's dx / sx exactly as above (max and the integer sum in any order)
__global__ __launch_bounds__(256) void x8_rows8_kernel(const float* __restrict__ x, uint32_t xs,
                                                       const int32_t* __restrict__ idx, uint32_t slots, uint32_t cols,
                                                       int8_t* __restrict__ x8, float* __restrict__ dx,
                                                       float* __restrict__ sx) {
  const uint32_t groups = cols / MMQ_GROUP;
  const uint64_t gi = ((uint64_t) blockIdx.x * 256 + threadIdx.x) / 4, ng = (uint64_t) slots * groups;
  const uint32_t c8 = 8 * (threadIdx.x % 4);
  const uint64_t gc = gi < ng ? gi : ng - 1;  // (past the end: the last group again, nothing stored)
  const uint32_t s = (uint32_t) (gc / groups), g = (uint32_t) (gc % groups);
  const int32_t r = idx[s];
  float v[8];
  if (r >= 0) {
    const float4* src = (const float4*) (x + (uint64_t) r * xs + (uint64_t) g * MMQ_GROUP + c8);
    const float4 lo = src[0], hi = src[1];
    v[0] = lo.x, v[1] = lo.y, v[2] = lo.z, v[3] = lo.w, v[4] = hi.x, v[5] = hi.y, v[6] = hi.z, v[7] = hi.w;
  } else {
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = 0.0f;
  }
  float a = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; i++) a = fmaxf(a, fabsf(v[i]));
  a = fmaxf(a, __shfl_xor(a, 1, 4));
  a = fmaxf(a, __shfl_xor(a, 2, 4));
  const float dd = __fdiv_rn(a, 127.0f);
  int sum = 0;
  uint64_t w = 0;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const int qv = a == 0.0f ? 0 : (int) fminf(fmaxf(rintf(__fdiv_rn(v[i], dd)), -127.0f), 127.0f);
    sum += qv;
    w |= (uint64_t) (uint8_t) (int8_t) qv << (8 * i);
  }
  sum += __shfl_xor(sum, 1, 4);
  sum += __shfl_xor(sum, 2, 4);
  if (gi < ng) {
    *(uint64_t*) (x8 + mmq_x8_at(s, g * MMQ_GROUP + c8, cols)) = w;
    if (c8 == 0) {
      const uint64_t at = mmq_dx_at(s, g, groups);
      const float d0 = a == 0.0f ? 0.0f : dd;
      dx[at] = d0;
      sx[at] = __fmul_rn(d0, (float) sum);
    }
  }
}

// a group's step for the first NI (1, 2 or 4) of a lane's 4 results: acc = fma(S dx, I, acc), acc = fma(-sx, M, acc) with result i's
// dx and sx from lane 4 B + i of the lane's row of 16. every F32 operation rounds on its own (fma, mul: the contract's).
// the waits that asm takes on itself: a DPP source needs two idle states after a VALU write (s_nop 1); the integer
// results are converted outside, where the compiler waits for the MFMA; and they stay an operand here to the end (I),
// also those with no token, so that no temporary of this asm gets a register that an MFMA in flight still writes
#define OSM_Q_MUL(i, lane) "v_mul_f32_dpp %[t" #i "], %[dv], %[S] row_newbcast:" lane " row_mask:0xf bank_mask:0xf\n\t"
#define OSM_Q_DOT(i) "v_fmac_f32 %[a" #i "], %[t" #i "], %[f" #i "]\n\t"
#define OSM_Q_SUM(i, lane) \
  "v_fmac_f32_dpp %[a" #i "], -%[sv], %[M] row_newbcast:" lane " row_mask:0xf bank_mask:0xf\n\t"
#define OSM_Q_OUT(i) [a##i] "+v"(acc[i]), [t##i] "=&v"(t[i])
#define OSM_Q_IN [dv] "v"(dv), [sv] "v"(sv), [S] "v"(S), [M] "v"(M), [I] "v"(I)
#define OSM_Q_STEP(l0, l1, l2, l3)                                                                                      \
  if constexpr (NI == 4)                                                                                                \
    asm("s_nop 1\n\t" OSM_Q_MUL(0, l0) OSM_Q_MUL(1, l1) OSM_Q_MUL(2, l2) OSM_Q_MUL(3, l3) OSM_Q_DOT(0) OSM_Q_DOT(1)     \
            OSM_Q_DOT(2) OSM_Q_DOT(3) OSM_Q_SUM(0, l0) OSM_Q_SUM(1, l1) OSM_Q_SUM(2, l2) OSM_Q_SUM(3, l3)               \
        : OSM_Q_OUT(0), OSM_Q_OUT(1), OSM_Q_OUT(2), OSM_Q_OUT(3)                                                        \
        : OSM_Q_IN, [f0] "v"(f[0]), [f1] "v"(f[1]), [f2] "v"(f[2]), [f3] "v"(f[3]));                                    \
  else if constexpr (NI == 2)                                                                                           \
    asm("s_nop 1\n\t" OSM_Q_MUL(0, l0) OSM_Q_MUL(1, l1) OSM_Q_DOT(0) OSM_Q_DOT(1) OSM_Q_SUM(0, l0) OSM_Q_SUM(1, l1)     \
        : OSM_Q_OUT(0), OSM_Q_OUT(1)                                                                                    \
        : OSM_Q_IN, [f0] "v"(f[0]), [f1] "v"(f[1]));                                                                    \
  else                                                                                                                  \
    asm("s_nop 1\n\t" OSM_Q_MUL(0, l0) OSM_Q_DOT(0) OSM_Q_SUM(0, l0) : OSM_Q_OUT(0) : OSM_Q_IN, [f0] "v"(f[0]));
template <int NI, int B>
__device__ inline void qstep(float* acc, v4i I, float dv, float sv, float S, float M) {
#if __HIP_DEVICE_COMPILE__
  float t[4];
  const float f[4] = {(float) I[0], (float) I[1], (float) I[2], (float) I[3]};
  if constexpr (B == 0) { OSM_Q_STEP("0", "1", "2", "3") }
  else if constexpr (B == 1) { OSM_Q_STEP("4", "5", "6", "7") }
  else if constexpr (B == 2) { OSM_Q_STEP("8", "9", "10", "11") }
  else { OSM_Q_STEP("12", "13", "14", "15") }
#endif
}
#undef OSM_Q_STEP
#undef OSM_Q_IN
#undef OSM_Q_OUT
#undef OSM_Q_SUM
#undef OSM_Q_DOT
#undef OSM_Q_MUL

struct QArgs {
  const uint8_t* const* wt;
  const int32_t* cnt;
  uint32_t rows, cols;
  const int8_t* x8;
  const float *dx, *sx;
  const uint32_t* soff;
  float* ya;
  const uint32_t* yoff;
  uint32_t ys;
};

// a workgroup: 64 rows (a wave 16) of matrix blockIdx.y over its cnt tokens, CT tiles of 16 at a time, a pass in every
// gridDim.z. partition p sums the 256-blocks b with b % 4 == p, its groups in ascending order; then the 4 sums are added
// in order. a block's activations for the tiles (x8 4 KB a tile, dx and sx 512 B a tile, contiguous in the slot
// layout) go through one of two LDS buffers, the next block's loads in flight during this one's MFMAs and stored behind
// them: one barrier a block. the weights' codes and header words come straight from global memory (mmraw.h's Q4_K).
// with the rows as A (their scales and the tokens' dx, sx through LDS, two barriers a block) and so, us, x8_rows
// included: 256 experts of 7168 x 2048, 512 tokens x 8: 875, 795; 128 of 2048 x 768: 148, 124; one expert of 17 tokens
// 22.5, 15.5, of 512 53.6, 52.2; 64 of 1040 x 1024 at 40 tokens 21.6, 19.0. slower, by up to 9 % (kernel alone, weights from
// HBM), are short rows in launches of about one round of the chip, where 149 VGPRs hold 3 waves a SIMD and 4 were held: 16 of
// 2048 x 768 at 40 / 64 / 100 / 200 tokens 13.5 / 16.3 / 23.4 / 36.3, 14.4 / 16.7 / 23.0 / 38.6. (held to 128 VGPRs, 5 spilled:
// 13.6 / 17.3 / 23.2 / 38.0, but 240 of 383 launches slower, by 8 % in the mean.)
// the kernel alone about 745, of which about 470 are left without the MFMAs and 555 without the loads: the epilogue's
// VALU work, then its waits on the MFMAs
template <int CT>
__global__ __launch_bounds__(kThreads) void q4k_kernel(QArgs a) {
  using X = mm::Raw<kQ4_K>;
  __shared__ u32x4 xs[2][CT * kXWords];
  __shared__ u32x4 ds[2][2 * CT * kDWords];  // dx of the tiles, then sx
  const uint32_t m = blockIdx.y, n = (uint32_t) a.cnt[m];
  if (n <= blockIdx.z * kTile * CT) return;  // (the whole workgroup: no pass of its own)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, q = lane / 16, c = lane % 16;
  const uint32_t row0 = (blockIdx.x * kWaves + wave) * kTile, nb = a.cols / 256, groups = a.cols / MMQ_GROUP;
  // (a wave past the rows computes the last row again, meets the barriers and stores nothing)
  const uint8_t* wr = table_at(a.wt, m) + (uint64_t) min(row0 + c, a.rows - 1) * nb * kBlockBytes;
  float* y = a.ya + a.yoff[m];
  const uint32_t soff = a.soff[m];
  auto pass = [&](auto tiles, auto results, uint32_t c0) __attribute__((always_inline)) {
    constexpr int C = decltype(tiles)::value, NI = decltype(results)::value;  // tiles; a tile's results with tokens
    constexpr uint32_t XW = C * kXWords, DW = C * kDWords, XP = (XW + kThreads - 1) / kThreads, DP = (2 * DW + kThreads - 1) / kThreads;
    const uint32_t s0 = soff + c0;  // the pass's first slot: a multiple of 16
    u32x4 xr[XP];
    F4 dr[DP];
    auto load = [&](uint32_t b) __attribute__((always_inline)) {
#pragma unroll
      for (uint32_t u = 0; u < XP; u++) {  // (past the words: the last again, not stored)
        const uint32_t i = min(u * kThreads + threadIdx.x, XW - 1);
        xr[u] = gload<u32x4>(a.x8 + mmq_x8_at(s0 + i / kXWords * kTile, b * 256, a.cols) + i % kXWords * 16);
      }
#pragma unroll
      for (uint32_t u = 0; u < DP; u++) {
        const uint32_t i = min(u * kThreads + threadIdx.x, 2 * DW - 1), f = i % DW;
        dr[u] = gload<F4>((i / DW ? a.sx : a.dx) + mmq_dx_at(s0 + f / kDWords * kTile, b * 8, groups) + f % kDWords * 4);
      }
    };
    auto store = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
      for (uint32_t u = 0; u < XP; u++)
        if (XW % kThreads == 0 || u * kThreads + threadIdx.x < XW) xs[buf][u * kThreads + threadIdx.x] = xr[u];
#pragma unroll
      for (uint32_t u = 0; u < DP; u++)
        if (u * kThreads + threadIdx.x < 2 * DW) ds[buf][u * kThreads + threadIdx.x] = u32x4{dr[u].x, dr[u].y, dr[u].z, dr[u].w};
    };
    X::R<8> raw;
    X::load<8>(raw, wr, 0, q);
    load(0);
    store(0);
    __syncthreads();
    float acc[4][C][4];
#pragma unroll
    for (int p = 0; p < 4; p++)
#pragma unroll
      for (int ct = 0; ct < C; ct++)
#pragma unroll
        for (int i = 0; i < 4; i++) acc[p][ct][i] = 0.0f;
    int buf = 0;
    for (uint32_t b0 = 0; b0 < nb; b0 += 4) {
#pragma unroll
      for (int p = 0; p < 4; p++) {
        const uint32_t b = b0 + (uint32_t) p;
        if (b >= nb) break;  // (uniform)
        const uint32_t next = b + 1 < nb ? b + 1 : b;  // (the last block: itself again)
        load(next);
        X::H<8> h;
        X::head<8>(h, raw, 0, q);
        X::load<8>(raw, wr + (uint64_t) next * kBlockBytes, 0, q);
        // A's lane c is slot 4 (c % 4) + c / 4, so that D's token 4 q + i is slot 4 i + q
        const int8_t* xb = (const int8_t*) xs[buf] + (4 * (c % 4) + c / 4) * MMQ_GROUP + 8 * q;
        // lane 4 g + i of each row of 16 holds slot 4 i + q's dx of groups g and g + 4
        const float* db = (const float*) ds[buf] + c / 4 * MMQ_SLOTS + 4 * (c % 4) + q;
        float dv[C][2], sv[C][2];
#pragma unroll
        for (int ct = 0; ct < C; ct++)
#pragma unroll
          for (int i = 0; i < 2; i++) dv[ct][i] = db[ct * 128 + 64 * i], sv[ct][i] = db[C * 128 + ct * 128 + 64 * i];
        // (the loads above and the stores below stay outside the groups: 848 us where the compiler mixes them, 746)
        __builtin_amdgcn_sched_barrier(0);
        auto group = [&](auto gc) __attribute__((always_inline)) {
          constexpr int g = decltype(gc)::value;
          const float S = __fmul_rn(h.d, (float) ((h.sc[g / 4] >> (8 * (g % 4))) & 0xFF));
          const float M = __fmul_rn(h.m, (float) ((h.mn[g / 4] >> (8 * (g % 4))) & 0xFF));
          const uint32_t w0 = (h.n[2 * (g / 2)] >> (4 * (g & 1))) & 0x0F0F0F0Fu, w1 = (h.n[2 * (g / 2) + 1] >> (4 * (g & 1))) & 0x0F0F0F0Fu;
          const long wv = (long) ((uint64_t) w1 << 32 | w0);
#pragma unroll
          for (int ct = 0; ct < C; ct++) {
            const long xv = *(const long*) (xb + ct * (int) kXWords * 16 + g * (MMQ_SLOTS * MMQ_GROUP));
            const v4i I = __builtin_amdgcn_mfma_i32_16x16x32_i8(xv, wv, v4i{0, 0, 0, 0}, 0, 0, 0);
            qstep<NI, g % 4>(acc[p][ct], I, dv[ct][g / 4], sv[ct][g / 4], S, M);
          }
        };
        group(std::integral_constant<int, 0>{}), group(std::integral_constant<int, 1>{});
        group(std::integral_constant<int, 2>{}), group(std::integral_constant<int, 3>{});
        group(std::integral_constant<int, 4>{}), group(std::integral_constant<int, 5>{});
        group(std::integral_constant<int, 6>{}), group(std::integral_constant<int, 7>{});
        store(buf ^ 1);  // (read a block ago, behind the last barrier)
        __syncthreads();
        buf ^= 1;
      }
    }
    const uint32_t r = row0 + c;
#pragma unroll
    for (int ct = 0; ct < C; ct++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const uint32_t t = c0 + ct * kTile + 4 * i + q;
        const float s = __fadd_rn(__fadd_rn(__fadd_rn(acc[0][ct][i], acc[1][ct][i]), acc[2][ct][i]), acc[3][ct][i]);
        if (t < n && r < a.rows) y[(uint64_t) t * a.ys + r] = s;
      }
  };
  for (uint32_t c0 = blockIdx.z * kTile * CT; c0 < n; c0 += gridDim.z * kTile * CT) {
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I4 = std::integral_constant<int, 4>;
    const uint32_t live = n - c0;  // (uniform; a tile's tokens 1 .. 4 are one result a lane, 5 .. 8 two, ...)
    if (live <= 4) pass(I1{}, I1{}, c0);
    else if (live <= 8) pass(I1{}, I2{}, c0);
    else if (CT == 1 || live <= 16) pass(I1{}, I4{}, c0);
    else if constexpr (CT == 2) pass(I2{}, I4{}, c0);
    __syncthreads();  // (the pass's buffers read before the next one's first store)
  }
}

// the token passes of a matrix spread over blockIdx.z: enough workgroups for the chip when few matrices hold many
// tokens (one expert at 512 tokens: 112 row blocks x 8), each workgroup a pass in every Z
template <int CT>
bool q4k_launch(const void* const* w, const int32_t* cnt, uint32_t n_mat, uint32_t max_cnt, uint32_t rows,
                uint32_t cols, const int8_t* x8, const float* dx, const float* sx, const uint32_t* soff, float* y,
                const uint32_t* yoff, uint32_t ys, hipStream_t s) {
  const uint32_t per = kTile * kWaves, bx = (rows + per - 1) / per, passes = (max_cnt + kTile * CT - 1) / (kTile * CT);
  uint32_t z = 1;
  while (z < passes && (uint64_t) bx * n_mat * z < 2048) z *= 2;  // (about 8 workgroups a CU at most)
  const QArgs a{(const uint8_t* const*) w, cnt, rows, cols, x8, dx, sx, soff, y, yoff, ys};
  q4k_kernel<CT><<<dim3(bx, n_mat, min(z, passes)), kThreads, 0, s>>>(a);
  return hipGetLastError() == hipSuccess;
}

}  // namespace mmq
}  // namespace osm

using namespace osm;

extern "C" OSM_API bool mmq_known(uint32_t type) { return type == kQ4_K; }

extern "C" OSM_API bool mmq_x8_rows(const float* x, uint32_t xs, const int32_t* idx, uint32_t slots, uint32_t cols,
                                    int8_t* x8, float* dx, float* sx, void* stream) {
  if (!x || !idx || !x8 || !dx || !sx || !slots || !cols || cols % MMQ_GROUP || xs < cols) return false;
  const uint64_t work = (uint64_t) slots * cols;
  if ((uintptr_t) x % 16 == 0 && xs % 4 == 0 && (uintptr_t) x8 % 8 == 0) {  // (the vector form where it is aligned)
    mmq::x8_rows8_kernel<<<(unsigned) ((work / 8 + 255) / 256), 256, 0, (hipStream_t) stream>>>(x, xs, idx, slots, cols,
                                                                                                x8, dx, sx);
    return hipGetLastError() == hipSuccess;
  }
  mmq::x8_rows_kernel<<<(unsigned) ((work + 255) / 256), 256, 0, (hipStream_t) stream>>>(x, xs, idx, slots, cols, x8,
                                                                                          dx, sx);
  return hipGetLastError() == hipSuccess;
}

extern "C" OSM_API bool mmq_group(uint32_t type, const void* const* w, const int32_t* cnt, uint32_t n_mat,
                                  uint32_t max_cnt, uint32_t rows, uint32_t cols, const int8_t* x8, const float* dx,
                                  const float* sx, const uint32_t* soff, float* y, const uint32_t* yoff, uint32_t ys,
                                  void* stream) {
  if (!mmq_known(type) || !w || !cnt || !x8 || !dx || !sx || !soff || !y || !yoff || !n_mat || !max_cnt || !rows ||
      rows % mmq::kTile || !cols || cols % 256 || ys < rows)
    return false;
  const hipStream_t s = (hipStream_t) stream;
  // (2 tiles a pass, 149 VGPRs, 3 waves a SIMD: a weight block decoded once for both; one tile's 112 VGPRs lose at 512
  // tokens x 8, 833 us for 745, and at the dense 512 tokens, 58 for 51. 4 would hold 2 waves)
  if (max_cnt <= mmq::kTile)
    return mmq::q4k_launch<1>(w, cnt, n_mat, max_cnt, rows, cols, x8, dx, sx, soff, y, yoff, ys, s);
  return mmq::q4k_launch<2>(w, cnt, n_mat, max_cnt, rows, cols, x8, dx, sx, soff, y, yoff, ys, s);
}
