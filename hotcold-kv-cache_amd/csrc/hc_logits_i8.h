// Window logits of f16/bf16 keys on the int8 matrix cores, bit-equal to the
// fp64 MFMA kernel (hc_snapkv.hip logits_kernel) that defines them.
//
// The 16 key rows of a tile are written as 31-bit fixed point under one power
// of two and that as four balanced base-256 digits (int8); a group-mean query
// row likewise, under its own.  The 16 digit products run on
// v_mfma_i32_16x16x64_i8, summed by weight into seven int32 accumulators (at
// most 4 * 128 * 2^14 = 2^23 each), so the 62-bit integer dot product is exact.
// It differs from the defining fp64 fma chain only by
//   * the chain's own roundings: 2^-53 of every partial sum, which together are
//     at most 2^-53 * ||q'|| * ||k|| with q'_d = (D - d) q_d (a product is in
//     D - d partial sums), about 0.58 D * ||q|| for even elements;
//   * query digits below the window: at most (sum of the residuals) * ||k||.
// With delta the sum of these, a logit whose dot product -delta and +delta
// round to one float is that float; a 16 x 16 tile with any other logit is
// recomputed by the fp64 chain itself (chain_tiles): 0.7 to 0.8% of the tiles of
// N(0,1) prompts, a count over 12000.  (Not under a scale that is a power of two:
// the exact products then fall on midpoints of floats, and the host takes the
// fp64 kernel.)
//
// Keys with bits below the window (f16 tiles of wide channels, a bf16 tile in
// some hundred) take a fifth digit, four more products (KDigits::low).  What
// has no digits goes to the chain without them: tiles beyond five digits,
// infinities and NaN, and every tile of a workgroup whose query rows have
// residuals that would leave most of its tiles open (kOpenRatio).
//
// What it buys: the fp64 matrix rate is 32 flop per cycle and SIMD, 1/64 of
// int8's, so 16 products cost a quarter of the one fp64 product.  Kernel times
// (fp64 form -> this one, 8 KV heads of 128): window 64, 32k keys x 16 rows
// f16 1243 -> 685 us, 64k x 4 bf16 with outlier channels 650 -> 400; window
// 32, 32 layers of 8k keys 343 -> 207, one layer 20.8 -> 16.5 (bound by
// latency); 32 heads of 5003 x 5003 (H2O) 1977 -> 1100.  What bounds it:
// vector issue (per 16 keys x 64 rows about 270 instructions make the key
// digits and 350 the logits, beside 128 matrix instructions of 16 cycles that
// hide two vector instructions each) and the logits' stores, which are 14% of
// the 32k launch and 27% of the H2O one.  Measured no faster: two key tiles
// per wave, a row block's products interleaved with the logits of the one
// before, and the keys' digits made once for all row blocks.
//
// Off the common path (f16, 8 KV heads, the whole score call, fp64 form -> this
// one; 32k keys x 4 rows, window 64 | 8k x 32, window 32): four channels 100
// times wider 411 -> 343 us, 400 times 412 -> 384 | 459 -> 446; a query channel
// 100 times wider 409 -> 415 | 450 -> 399, 1000 times 409 -> 463 | 451 -> 430;
// exponents over 24 binades 415 -> 461 | 453 -> 432; logits that cancel exactly
// 409 -> 577.  So where all tiles are known to be the chain's it is from 5% faster
// to 13% slower than the fp64 kernel (the same products, from a smaller LDS
// block); where only the digits show it, they come on top.
#pragma once
#include <type_traits>

#include "hc_common.h"

namespace hc {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef double doublex2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

constexpr int kDigitChunk = 64;              // keys per workgroup and step: 4 waves x 16
constexpr int kDigits = 4;
constexpr uint32_t kBalance = 0x80808080u;   // digits of u: the bytes of (u + kBalance) ^ kBalance
constexpr uint32_t kFixMax = 0x7f7f7f7fu;    // the largest value that four balanced digits hold

// Per window row, beside its digits: the scale 2^-sh of its fixed point, and
// upper bounds of 2^53 times the roundings' share of delta against a key of
// 2-norm 1 (||q'|| and kEvalUlps ||q|| for the evaluation's own) and of the sum
// of its residuals.
struct QDigitRow {
  double scale;
  float norm, resid;
};
constexpr int kEvalUlps = 16;
// A row whose residuals are r of its norm leaves about 2^34 r of its logits
// open (delta over half an ulp of a logit of typical size, head dim 128).  From
// this sum of r over a row block on, the mean over a workgroup's, all its tiles
// go to the chain.  Measured with one query channel 60 to 1000 times wider (f16,
// 8k keys x 32 rows, window 32): 371, 390, 432, 435, 426 us where a bound of
// 2^-39 gives 413, 441, 505, 488, 458; at 32k x 4, window 64, the two differ by
// at most 6% either way.
constexpr float kOpenRatio = 0x1p-41f;

// Reductions over a wave's lanes: rows (col, col + 16, col + 32, col + 48) by
// gfx950's row swaps, the 16 lanes of a row by rotations.
template <int N>
__device__ __forceinline__ uint32_t row_ror(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x120 + N, 0xf, 0xf, false);
}
template <typename F>
__device__ __forceinline__ uint32_t reduce_rows(uint32_t x, F&& f) {   // over the four rows
  const auto a = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  x = f(a[0], a[1]);
  const auto c = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  return f(c[0], c[1]);
}
template <typename F>
__device__ __forceinline__ uint32_t reduce_cols(uint32_t x, F&& f) {   // over the 16 lanes of a row
  x = f(x, row_ror<8>(x));
  x = f(x, row_ror<4>(x));
  x = f(x, row_ror<2>(x));
  return f(x, row_ror<1>(x));
}
struct MaxU16x2 {
  __device__ uint32_t operator()(uint32_t p, uint32_t q) const {
    return __builtin_bit_cast(uint32_t,
                              __builtin_elementwise_max(__builtin_bit_cast(u16x2, p), __builtin_bit_cast(u16x2, q)));
  }
};
struct MaxU32 {
  __device__ uint32_t operator()(uint32_t p, uint32_t q) const { return p > q ? p : q; }
};
struct MaxF32 {
  __device__ uint32_t operator()(uint32_t p, uint32_t q) const {
    return __float_as_uint(fmaxf(__uint_as_float(p), __uint_as_float(q)));
  }
};
struct SumF32 {
  __device__ uint32_t operator()(uint32_t p, uint32_t q) const {
    return __float_as_uint(__uint_as_float(p) + __uint_as_float(q));
  }
};

// The group-mean queries with their digits, and qmean_kernel's resets of the
// row maxima, the NaN flag and the padding statistics (zero rows past W).
// grid (wpad / RB, Hk, B), block 64 RB, one wave per row; lane l owns dims
// E l .. E l + E - 1.  Both leave in the order that the matrix instructions read
// them, 16 rows to a block, through LDS so that RB rows' 16-byte pieces go out
// together:
//   qf [row block][dims 8u .. 8u + 7][lane][2], lane (kk, row) holding dims
//      8u + kk and 8u + 4 + kk: two k-steps of the fp64 chain;
//   qd [row block][digit][k-step of 64][lane][16], lane (kk, row) holding dims
//      8 * (kk + 4 * t) + r of the pieces t = 2s, 2s + 1 of k-step s.
// Bound by its stores (12 bytes per element): 87 us for 32 heads of 5003 rows at
// RB = 16, 4.2 for 8 heads of 32 at RB = 4.
template <typename T, int D, int RB>
__global__ __launch_bounds__(64 * RB) void qdigit_kernel(const T* __restrict__ q, const T* const* __restrict__ q_rows,
                                                     int64_t q_sb, int64_t q_sh, int64_t q_ss, int64_t q_row0, int Hq,
                                                     int Hk, int W, int wpad, double* __restrict__ qf,
                                                     uint32_t* __restrict__ rmax, RowStat* __restrict__ rstat,
                                                     uint32_t* __restrict__ nan_flag, int8_t* __restrict__ qd,
                                                     QDigitRow* __restrict__ qrow) {
  constexpr int E = D / 64;
  __shared__ double sx[RB][D + 4];
  __shared__ i32x4 sd[RB * D * kDigits / 16];
  const int tid = threadIdx.x, lane = tid & 63, r = tid >> 6;
  const int w = (int)blockIdx.x * RB + r, h = blockIdx.y, b = blockIdx.z;
  const int64_t bh = (int64_t)b * Hk + h, row = bh * wpad;
  const int wst = (int)cdiv(W, kStatPad) * kStatPad;
  if (lane == 0 && w == 0) nan_flag[bh] = 0;
  if (lane == 0 && w < W) rmax[bh * W + w] = order_key(-INFINITY);
  if (lane == 0 && w >= W && w < wst) rstat[bh * wst + w] = RowStat{INFINITY, 0.0};
  double x[E];
#pragma unroll
  for (int e = 0; e < E; ++e) x[e] = 0.0;
  if (w < W) {
    const int G = Hq % Hk == 0 ? Hq / Hk : Hq;          // scoring.py:26: else every query head
    const int g0 = Hq % Hk == 0 ? h * G : 0;
    const T* src = (q_rows ? q_rows[b] : q + b * q_sb) + (q_row0 + w) * q_ss + g0 * q_sh + lane * E;
#pragma unroll
    for (int e = 0; e < E; ++e) x[e] = to_f64(src[e]);
    for (int g = 1; g < G; ++g)
#pragma unroll
      for (int e = 0; e < E; ++e) x[e] = x[e] + to_f64(src[g * q_sh + e]);
#pragma unroll
    for (int e = 0; e < E; ++e) x[e] = x[e] / (double)G;
  }
  uint32_t hi = 0;            // the largest magnitude's high word
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    sx[r][lane * E + e] = x[e];
    hi = max(hi, (uint32_t)__double2hiint(x[e]) & 0x7fffffffu);
    const float xw = (float)x[e] * (float)(D - (lane * E + e) + kEvalUlps);
    ss = fmaf(xw, xw, ss);
  }
  hi = reduce_cols(reduce_rows(hi, MaxU32{}), MaxU32{});
  // |x| < 2^(ex + 1), and below kFixMax / 2^30 * 2^ex if the top mantissa bits allow
  const int ex = (int)(hi >> 20) - 1023;
  static_assert((0x100000ull + 0xfd000ull) << 10 < kFixMax, "the largest value at the full scale");
  const int sh = 30 - ex - ((hi & 0xfffffu) >= 0xfd000u ? 1 : 0);
  const bool use = hi >= (64u << 20) && hi < 0x7ff00000u;    // normal, and no infinity or NaN
  float res = 0.f;
  uint32_t u[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int v = use ? (int)rint(ldexp(x[e], sh)) : 0;
    res += use ? fabsf((float)(x[e] - ldexp((double)v, -sh))) : 0.f;
    u[e] = ((uint32_t)v + kBalance) ^ kBalance;
  }
  const int d = lane * E, t = d >> 5;
  // sd: [digit][k-step][kk][row of RB][16]
  int8_t* dst = reinterpret_cast<int8_t*>(sd) + ((t >> 1) * 4 + ((d >> 3) & 3)) * RB * 16 + r * 16 + (t & 1) * 8 +
                (d & 7);
#pragma unroll
  for (int j = 0; j < kDigits; ++j)
#pragma unroll
    for (int e = 0; e < E; ++e) dst[j * (D / 64) * RB * 64 + e] = (int8_t)(u[e] >> (8 * j));
  ss = __uint_as_float(reduce_cols(reduce_rows(__float_as_uint(ss), SumF32{}), SumF32{}));
  res = __uint_as_float(reduce_cols(reduce_rows(__float_as_uint(res), SumF32{}), SumF32{}));
  if (lane == 0) {
    // rounded up, past what the fp32 sums lose, to underflow too
    const float up = 1.f + 0x1p-14f, tiny = 1e-17f;
    QDigitRow o;
    o.scale = use ? ldexp(1.0, -sh) : 1.0;
    o.norm = hi == 0 ? 0.f : use ? sqrtf(ss) * up + tiny : INFINITY;     // (0: every product is 0)
    o.resid = hi == 0 ? 0.f : res * up + 2e-36f;
    qrow[row + w] = o;
  }
  __syncthreads();
  const int64_t at = (row + (w >> 4) * 16) * D;      // the row block
  const int r0 = (int)blockIdx.x * RB % 16;
  doublex2* of = reinterpret_cast<doublex2*>(qf + at);
  i32x4* od = reinterpret_cast<i32x4*>(qd + at * kDigits);
#pragma unroll
  for (int i = tid; i < RB * D / 2; i += 64 * RB) {  // piece i: dims 8 (i / 4 RB) + (i / RB) % 4, row i % RB
    const int c = i / (4 * RB) * 8 + i / RB % 4;
    of[i / RB * 16 + r0 + i % RB] = doublex2{sx[i % RB][c], sx[i % RB][c + 4]};
  }
  if (tid < RB * D * kDigits / 16) od[tid / RB * 16 + r0 + tid % RB] = sd[tid];
}

// Fixed point of key rows: |x| * 2^(kShift - f) <= kFixMax for every element,
// f from the largest magnitude's bits (its exponent field).  kExactF: up to
// this f no element of the type has bits below the window.  kMinF keeps the
// scale, and the squares of elements that are held exactly, normal floats.
template <typename T>
struct KFix;
template <>
struct KFix<half_t> {
  static constexpr int kMant = 10, kInf = 0x7c00, kShift = 45, kMinF = 1, kExactF = 21;
  __device__ static float get(uint32_t w, int hi) {
    return (float)__builtin_bit_cast(half_t, (uint16_t)(hi ? w >> 16 : w & 0xffffu));
  }
  __device__ static float dot2(uint32_t w, float acc) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, w), __builtin_bit_cast(h2, w), acc, false);
  }
};
template <>
struct KFix<bf16_t> {
  static constexpr int kMant = 7, kInf = 0x7f80, kShift = 157, kMinF = 87, kExactF = 0;
  __device__ static float get(uint32_t w, int hi) { return __uint_as_float(hi ? w & 0xffff0000u : w << 16); }
  __device__ static float dot2(uint32_t w, float acc) {
    typedef __bf16 b2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(b2, w), __builtin_bit_cast(b2, w), acc, false);
  }
};

// The digits of 16 key rows (A operand: lane (kk, col) the same dims of row
// col as q_digit_at), their scale and the largest bound of a row's 2-norm.
template <typename T, int D>
struct KDigits {
  static constexpr int NP = D / 32;   // 16-byte pieces per lane
  static constexpr int NS = D / 64;   // k-steps
  i32x4 d[kDigits][NS];
  i32x4 low[NS];   // the fifth digit, of weight 2^-8
  int f;           // scale 2^(f - kShift)
  int held;        // digits that hold every element exactly: 4, 5, or 0 if no five do
  uint32_t zero;   // bit r: row r is all zero
  float norm;

  __device__ __forceinline__ void scan(const uint32_t (&w)[NP][4]) {
    using F = KFix<T>;
    u16x2 mx = {0, 0};
    float ss = 0.f;
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        mx = __builtin_elementwise_max(mx, __builtin_bit_cast(u16x2, w[p][i] & 0x7fff7fffu));
        ss = F::dot2(w[p][i], ss);
      }
    uint64_t z = __ballot(__builtin_bit_cast(uint32_t, mx) == 0);     // the row's four lanes
    z &= z >> 32;
    zero = (uint32_t)(z & z >> 16) & 0xffffu;
    const uint32_t hi = reduce_cols(reduce_rows(__builtin_bit_cast(uint32_t, mx), MaxU16x2{}), MaxU16x2{});
    const int mb = __builtin_amdgcn_readfirstlane((int)max(hi & 0xffffu, hi >> 16));
    // a mantissa at 2 - 2^-7 or above would pass kFixMax
    f = max((mb + (1 << (F::kMant - 7))) >> F::kMant, F::kMinF);
    held = kDigits;
    if (f > F::kExactF) {       // wave-uniform: the smallest non-zero element decides
      u16x2 mn = {0xffff, 0xffff};
#pragma unroll
      for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const u16x2 a = __builtin_bit_cast(u16x2, w[p][i] & 0x7fff7fffu);
          mn = __builtin_elementwise_min(mn, (u16x2)(a - (u16x2){1, 1}));   // zeros wrap to 0xffff
        }
      const uint32_t lo = reduce_cols(reduce_rows(~__builtin_bit_cast(uint32_t, mn), MaxU16x2{}), MaxU16x2{});
      const int nb = __builtin_amdgcn_readfirstlane(0x10000 - (int)max(lo & 0xffffu, lo >> 16));
      const int below = f - (30 - F::kMant) - max(nb >> F::kMant, 1);   // bits below the four digits
      held = below <= 0 ? 4 : below <= 8 ? 5 : 0;
    }
    if (mb >= F::kInf) held = 0;
    // An fp32 sum of D squares and its root: within 2^-14.  Half subnormals,
    // which the dot product may take as zero, are below sqrt(D) * 2^-14.
    ss = __uint_as_float(reduce_cols(reduce_rows(__float_as_uint(ss), SumF32{}), MaxF32{}));
    norm = sqrtf(ss) * (1.f + 0x1p-14f) + 0x1p-10f;
  }

  // With LOW the four digits hold the nearest integer and the fifth the rest.
  template <bool LOW>
  __device__ __forceinline__ void digits(const uint32_t (&w)[NP][4]) {
    using F = KFix<T>;
    const float mult = __uint_as_float((uint32_t)(127 + F::kShift - f) << 23);
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        uint32_t u[4], rest = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float x = F::get(w[p][2 * h + (i >> 1)], i & 1);
          float v = __builtin_fmaf(x, mult, 0.f);
          if constexpr (LOW) {
            // the nearest integer (a fraction needs |v| < 2^11, so v + 1/2 is
            // exact where it matters) and 256ths of the rest, plus 128
            const float n = __builtin_floorf(v + 0.5f);
            rest = __builtin_amdgcn_cvt_pk_u8_f32(__builtin_fmaf(v - n, 256.f, 128.f), i, rest);
            v = n;
          }
          u[i] = (uint32_t)(int)v + kBalance;
        }
        // bytes of the four elements regrouped by digit
        const uint32_t a0 = __builtin_amdgcn_perm(u[1], u[0], 0x05010400u);
        const uint32_t a1 = __builtin_amdgcn_perm(u[1], u[0], 0x07030602u);
        const uint32_t b0 = __builtin_amdgcn_perm(u[3], u[2], 0x05010400u);
        const uint32_t b1 = __builtin_amdgcn_perm(u[3], u[2], 0x07030602u);
        const int at = 2 * (p & 1) + h;
        d[0][p >> 1][at] = (int)(__builtin_amdgcn_perm(b0, a0, 0x05040100u) ^ kBalance);
        d[1][p >> 1][at] = (int)(__builtin_amdgcn_perm(b0, a0, 0x07060302u) ^ kBalance);
        d[2][p >> 1][at] = (int)(__builtin_amdgcn_perm(b1, a1, 0x05040100u) ^ kBalance);
        d[3][p >> 1][at] = (int)(__builtin_amdgcn_perm(b1, a1, 0x07060302u) ^ kBalance);
        if constexpr (LOW) low[p >> 1][at] = (int)(rest ^ kBalance);
      }
  }
};

// NB 16-key x 16-row tiles by the defining fp64 chain: the keys key0.. that the
// wave holds in w (as the logits kernel loads them), rows wt.. of the
// workgroup's block at window row w0.  Stores the logits and folds the lane's
// maxima of rows wt + 16 t + kk + 4 i into top[t][i].  fetch(row block, pair of
// k-steps) gives a lane its two queries; AHEAD pairs of them are under way.  The
// matrix unit's fp64 products hide few vector instructions, so there are few:
// the addresses are scalar offsets.
template <typename T, int MODE, int D, int NB, int AHEAD, typename F>
__device__ __forceinline__ void chain_tiles(const uint32_t (&w)[D / 32][4], F&& fetch, __amdgpu_buffer_rsrc_t lrs,
                                            int ld, int key0, int w0, int wt, int nw, int qpos0, double scaling,
                                            float (&top)[NB][4]) {
  typedef double doublex4 __attribute__((ext_vector_type(4)));
  constexpr int NU = D / 8;
  int lane = threadIdx.x & 63;
  // what follows from the lane is worked out here: hoisted out of the caller's
  // chunk loop, it would hold registers (or scratch) in the common path too
  __asm__ volatile("" : "+v"(lane));
  const int col = lane & 15, kk = lane >> 4, key = key0 + col;
  doublex4 acc[NB];
  doublex2 q[AHEAD][NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) acc[i] = doublex4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int u = 0; u < AHEAD; ++u)
#pragma unroll
    for (int i = 0; i < NB; ++i) q[u][i] = fetch(i, u);
  static_assert(4 % AHEAD == 0, "whole turns of the ring in a piece");
#pragma unroll
  for (int u0 = 0; u0 < NU; u0 += 4) {
    const uint32_t(&wp)[4] = w[u0 / 4];
    // A lane holds 8 consecutive dims of its key, the key's four lanes 32; a
    // k-step wants dim 4t + kk in lane kk.  Dims kk and kk + 4 of a lane are
    // packed for lane kk, and the four packed words go their ways as a 4 x 4
    // transpose over the rows of 16 lanes: x[g] then holds lane kk's dims of
    // k-steps 2 (u0 + g) and 2 (u0 + g) + 1.
    uint32_t x[4];
    x[0] = __builtin_amdgcn_perm(wp[2], wp[0], 0x05040100u);
    x[1] = __builtin_amdgcn_perm(wp[2], wp[0], 0x07060302u);
    x[2] = __builtin_amdgcn_perm(wp[3], wp[1], 0x05040100u);
    x[3] = __builtin_amdgcn_perm(wp[3], wp[1], 0x07060302u);
#pragma unroll
    for (int i = 0; i < 4; i += 2) {
      const auto s = __builtin_amdgcn_permlane16_swap(x[i], x[i + 1], false, false);
      x[i] = s[0];
      x[i + 1] = s[1];
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const auto s = __builtin_amdgcn_permlane32_swap(x[i], x[i + 2], false, false);
      x[i] = s[0];
      x[i + 2] = s[1];
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const double kd = (double)KFix<T>::get(x[g], s);
#pragma unroll
        for (int i = 0; i < NB; ++i)
          acc[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(q[g % AHEAD][i][s], kd, acc[i], 0, 0, 0);
      }
      if (u0 + g + AHEAD < NU)
#pragma unroll
        for (int i = 0; i < NB; ++i) q[g % AHEAD][i] = fetch(i, u0 + g + AHEAD);
    }
  }
  // Lane (kk, col): rows kk + 4i of the tiles, key col.
  const uint32_t off = key < ld ? (uint32_t)((w0 + wt + kk) * ld + key) * 4u : kOob;
  auto finish = [&](auto plain_c) {
    constexpr bool PLAIN = decltype(plain_c)::value;
#pragma unroll
    for (int t = 0; t < NB; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 16 * t + 4 * i;
        float L;
        if constexpr (MODE == HC_SCORE_SNAPKV) L = (float)(acc[t][i] * scaling);
        else L = (float)(acc[t][i] / scaling);
        uint32_t o = off;
        if constexpr (!PLAIN) {
          if constexpr (MODE == HC_SCORE_SNAPKV) L = key > qpos0 + wt + kk + r ? -INFINITY : L;
          o = wt + kk + r < nw ? off : kOob;
        }
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(L), lrs, (int)o, (int)((uint32_t)(r * ld) * 4u), 0);
        if constexpr (MODE == HC_SCORE_SNAPKV) top[t][i] = fmaxf(top[t][i], L);
      }
  };
  // wave-uniform: every key at or before every row's position, every row real
  if ((MODE != HC_SCORE_SNAPKV || key0 + 15 <= qpos0 + wt) && wt + 16 * NB <= nw) finish(std::true_type{});
  else finish(std::false_type{});
}

// The logits kernel.  grid (ceil(S / (64 * cpw)), Hk * ceil(W / (16 * NRB)),
// B), block 256; workgroup order, causal skips and stores' extent as
// logits_kernel's.  Each wave owns 16 keys of a chunk: their digits stay
// in registers while the row blocks' digits come from LDS, 16 rows at a time.
// Keys are the A operand, so a lane's four results are consecutive keys of one
// row: one 16-byte store.  The next chunk's keys are loaded while this one is
// multiplied.  Chunks that take more than four digits are left for two loops of
// their own, the chain's with the queries in LDS for the whole workgroup: each
// form keeps its registers, and the chain's tiles their matrix rate (the same
// tiles redone one by one in place, the queries read from memory, took five
// times the fp64 kernel).  Up to 32 rows four waves fit a SIMD, and one 8k
// layer's 1024 workgroups the chip at once (19.3 us with three).
template <typename T, int MODE, int D, int NRB>
__global__ __launch_bounds__(256, MODE == HC_SCORE_SNAPKV && NRB < 4 ? 4 : 3) void logits_i8_kernel(
    const T* __restrict__ k, const T* const* __restrict__ k_rows, int64_t k_sb, int64_t k_sh, int64_t k_ss,
    uint32_t k_bytes, const double* __restrict__ qf, const int8_t* __restrict__ qd,
    const QDigitRow* __restrict__ qrow, int Hk, int S, int W, int wpad, double scaling, int cpw, int ld,
    float* __restrict__ logits, uint32_t* __restrict__ rmax) {
  constexpr int ROWS = 16 * NRB, NS = D / 64, NP = D / 32, CHUNK = kDigitChunk;
  constexpr int PB = NRB < 2 ? NRB : 2;       // row blocks per pass over the hard chunks
  constexpr int SQ_DIGITS = NRB * kDigits * NS * 64, SQ_CHAIN = PB * 8 * D;
  __shared__ i32x4 sq[SQ_DIGITS > SQ_CHAIN ? SQ_DIGITS : SQ_CHAIN];
  __shared__ doublex2 srow[ROWS];    // row scale times the logit scale; a key of 2-norm 1's delta against the row
  __shared__ uint32_t redk[ROWS];
  __shared__ int open_s;             // the rows' residuals leave most tiles open
  __shared__ int hard_s;             // a wave has hard chunks
  const int nrb = (W + ROWS - 1) / ROWS, nx = (int)gridDim.x;
  const int fl = (int)blockIdx.x + nx * (int)blockIdx.y;
  const int rb = nrb - 1 - fl % nrb;
  const int xr = nx - 1 - (fl / nrb) % nx;
  const int h = fl / (nrb * nx);
  const int b = blockIdx.z, tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, kk = lane >> 4;
  const int w0 = rb * ROWS;
  const int nw = min(ROWS, W - w0);
  const int64_t bh = (int64_t)b * Hk + h;
  const T* krow = k_rows ? k_rows[b] : k + b * k_sb;
  const __amdgpu_buffer_rsrc_t krs = make_rsrc(krow + h * k_sh, k_bytes);
  const uint32_t rowb = (uint32_t)(k_ss * (int64_t)sizeof(T));
  const int qpos0 = S - W + w0;
  const __amdgpu_buffer_rsrc_t lrs = make_rsrc(logits + bh * W * ld, (uint32_t)((int64_t)W * ld * 4));
  const int wg_key0 = xr * (CHUNK * cpw);
  if constexpr (MODE == HC_SCORE_SNAPKV)
    if (wg_key0 > qpos0 + nw - 1 + kNeverRead) return;   // workgroup-uniform
  const bool stage = MODE != HC_SCORE_SNAPKV || wg_key0 <= qpos0 + nw - 1;

  int key0 = wg_key0 + wave * 16;
  uint32_t raw[NP][4];
  auto load_keys = [&](uint32_t (&dst)[NP][4], int at) {
    const int key = at + col;
    const uint32_t off = key < S ? (uint32_t)key * rowb + 16u * kk : kOob;
#pragma unroll
    for (int p = 0; p < NP; ++p) bload_so<16>(krs, off, 64u * p, dst[p]);
  };
  auto load = [&](int at) { load_keys(raw, at); };
  load(key0);
  if (tid < ROWS) redk[tid] = order_key(-INFINITY);
  if (tid == 0) open_s = hard_s = 0;
  if (stage) {
    const i32x4* src = reinterpret_cast<const i32x4*>(qd + (bh * wpad + w0) * (int64_t)(D * kDigits));
#pragma unroll
    for (int i = tid; i < NRB * kDigits * NS * 64; i += 256) sq[i] = src[i];
    const double lscale = MODE == HC_SCORE_SNAPKV ? scaling : 1.0 / scaling;
    if (tid < ROWS) {
      const QDigitRow r = qrow[bh * wpad + w0 + tid];
      srow[tid] = doublex2{r.scale * lscale, ((double)r.norm * 0x1p-53 + (double)r.resid) * fabs(lscale) * 1.001};
      float open = r.norm < INFINITY ? (r.norm > 0.f ? r.resid / r.norm : 0.f) : INFINITY;
#pragma unroll
      for (int o = ROWS / 2; o > 0; o >>= 1) open += __shfl_xor(open, o, 64);
      if (tid == 0) open_s = open > NRB * kOpenRatio;
    }
  }
  __syncthreads();
  const bool open_rows = __builtin_amdgcn_readfirstlane(open_s);
  const double* qrows = qf + (bh * wpad + w0) * D;

  const int nch = key0 < S ? min(cpw, (S - key0 + CHUNK - 1) / CHUNK) : 0;
  int nmul = nch;
  if constexpr (MODE == HC_SCORE_SNAPKV) {
    const int last = qpos0 + nw - 1;
    nmul = key0 > last ? 0 : min(nch, (last - key0) / CHUNK + 1);
  }
  float mrow[NRB];
#pragma unroll
  for (int i = 0; i < NRB; ++i) mrow[i] = -INFINITY;
  // chain_tiles' maxima of rows wt .. into redk
  auto fold = [&](const auto& top, int wt) {
    if constexpr (MODE == HC_SCORE_SNAPKV)
#pragma unroll
      for (int t = 0; t < (int)(sizeof(top) / sizeof(top[0])); ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) atomicMax(&redk[wt + 16 * t + kk + 4 * i], order_key(top[t][i]));
  };

  // The products of row block nb against the chunk's keys; with LOW the fifth
  // digits' too, rest of weight 2^-8.
  auto multiply = [&](const KDigits<T, D>& kd, i32x4 (&acc)[2 * kDigits - 1], i32x4& rest, int lane, int nb,
                      auto low_c) {
#pragma unroll
    for (int j = 0; j < kDigits; ++j) {
      i32x4 q[NS];
#pragma unroll
      for (int s = 0; s < NS; ++s) q[s] = sq[((nb * kDigits + j) * NS + s) * 64 + lane];
#pragma unroll
      for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int i = 0; i < kDigits; ++i) {
          const bool first = s == 0 && (j == 0 || i == kDigits - 1);   // of its weight
          acc[i + j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(kd.d[i][s], q[s],
                                                             first ? i32x4{0, 0, 0, 0} : acc[i + j], 0, 0, 0);
        }
      if constexpr (decltype(low_c)::value)
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          i32x4& to = j ? acc[j - 1] : rest;
          to = __builtin_amdgcn_mfma_i32_16x16x64_i8(kd.low[s], q[s], j + s ? to : i32x4{0, 0, 0, 0}, 0, 0, 0);
        }
    }
  };
  // Their logits: stored, or the tile marked for the fp64 chain.  PLAIN: no row
  // before a key's position, no key past the last or all zero (its logits are
  // 0: with a delta of more they would all be redone).
  auto finish = [&](const KDigits<T, D>& kd, const i32x4 (&acc)[2 * kDigits - 1], const i32x4& rest, int key0,
                    uint32_t& redo, int lane, int nb, auto plain_c, auto low_c) {
    const int col = lane & 15, kk = lane >> 4;
    constexpr bool PLAIN = decltype(plain_c)::value, LOW = decltype(low_c)::value;
    const int w = 16 * nb + col;
    const doublex2 row = srow[w];
    const double rs = row[0], dl = row[1];
    const uint64_t live = ((1ull << min(max(nw - 16 * nb, 0), 16)) - 1) * 0x0001000100010001ull;   // real rows' lanes
    const double del = dl * (double)kd.norm;
    const double sc = rs * __hiloint2double((1023 + kd.f - KFix<T>::kShift) << 20, 0);
    const int key = key0 + 4 * kk;
    const uint32_t zero = kd.zero >> 4 * kk;
    float L[4];
    bool open = false;       // a logit that delta does not settle
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t0 = (acc[6][i] << 8) + acc[5][i];
      const int t1 = (acc[4][i] << 8) + acc[3][i];
      const int t2 = (acc[2][i] << 8) + acc[1][i];
      double d = __builtin_fma(__builtin_fma(__builtin_fma((double)t0, 65536.0, (double)t1), 65536.0,
                                             (double)t2), 256.0, (double)acc[0][i]);
      if constexpr (LOW) d = __builtin_fma((double)rest[i], 0x1p-8, d);
      const float lo = (float)__builtin_fma(d, sc, -del);
      L[i] = (float)__builtin_fma(d, sc, del);
      bool bad = !(lo == L[i]);
      if constexpr (!PLAIN) {
        if (zero >> i & 1) {
          L[i] = 0.f;
          bad = false;
        }
        if constexpr (MODE == HC_SCORE_SNAPKV)
          if (key + i > qpos0 + w) {
            L[i] = -INFINITY;
            bad = false;
          }
        bad = bad && key + i < S;
      }
      open |= bad;
    }
    // The stores are issued either way (out of range for an open tile): the
    // wait for the next chunk's keys counts them, and behind a branch it
    // would have to wait for the stores too.
    const bool again = (__ballot(open) & live) != 0;    // wave-uniform
    redo |= again ? 1u << nb : 0u;
    const bool ok = w < nw && !again;
    const uint32_t off = ok ? (uint32_t)((w0 + w) * ld + key) * 4u : kOob;
    const uint32_t bits[4] = {__float_as_uint(L[0]), __float_as_uint(L[1]), __float_as_uint(L[2]),
                              __float_as_uint(L[3])};
    if constexpr (PLAIN) {
      bstore<16>(lrs, off, bits);
      if constexpr (MODE == HC_SCORE_SNAPKV)
        mrow[nb] = fmaxf(mrow[nb], ok ? fmaxf(fmaxf(L[0], L[1]), fmaxf(L[2], L[3])) : -INFINITY);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        bstore<4>(lrs, key + i < ld ? off + 4u * i : kOob, &bits[i]);   // kOob + 12 is out of range too
        if constexpr (MODE == HC_SCORE_SNAPKV) mrow[nb] = fmaxf(mrow[nb], ok && key + i < S ? L[i] : -INFINITY);
      }
    }
  };
  auto row_blocks = [&](const KDigits<T, D>& kd, int key0, int lane, auto plain_c, auto low_c) {
    uint32_t redo = 0;
#pragma unroll
    for (int nb = 0; nb < NRB; ++nb) {
      i32x4 acc[2 * kDigits - 1], rest;
      multiply(kd, acc, rest, lane, nb, low_c);
      finish(kd, acc, rest, key0, redo, lane, nb, plain_c, low_c);
      // side by side, two row blocks with a fifth digit would need more
      // registers than the common form
      if constexpr (decltype(low_c)::value) __builtin_amdgcn_sched_barrier(0);
    }
    return redo;
  };
  auto redo_tiles = [&](uint32_t redo, int key0) {
    if (!redo) return;           // wave-uniform
    uint32_t cur[NP][4];
    load_keys(cur, key0);
    while (redo) {
      const int nb = __ffs(redo) - 1;
      redo &= redo - 1;
      const __amdgpu_buffer_rsrc_t qrs = make_rsrc(qrows + 16 * nb * D, 16 * D * 8);
      float top[1][4] = {{-INFINITY, -INFINITY, -INFINITY, -INFINITY}};
      chain_tiles<T, MODE, D, 1, 4>(cur, [&](int, int u) {
        uint32_t r[4];
        bload_so<16>(qrs, 16u * lane, 1024u * u, r);
        return __builtin_bit_cast(doublex2, u32x4{r[0], r[1], r[2], r[3]});
      }, lrs, ld, key0, w0, 16 * nb, nw, qpos0, scaling, top);
      fold(top, 16 * nb);
    }
  };
  auto chunk = [&](int c) { return wg_key0 + wave * 16 + c * CHUNK; };

  // Chunks whose keys need a fifth digit, and those that only the fp64 chain
  // does, are left for the loops below (bit c of wide and hard).  After two at
  // the start the rest is left unseen: where all are, looking costs a read of
  // the keys.
  const uint32_t all = (1u << nmul) - 1;
  uint32_t wide = 0, hard = open_rows ? all : 0;
  if (!open_rows)
    for (int c = 0; c < nmul; ++c) {
      // the row blocks' LDS reads repeat for every chunk: hoisted, they would
      // hold registers for the kernel's lifetime
      __asm__ volatile("" ::: "memory");
      KDigits<T, D> kd;
      kd.scan(raw);
      if (kd.held != kDigits) {    // wave-uniform
        wide |= 1u << c;
        if (wide == 3) {
          wide = all;
          break;
        }
        load(key0 + CHUNK);
        key0 += CHUNK;
        continue;
      }
      kd.template digits<false>(raw);
      load(key0 + CHUNK);
      const bool plain = key0 + 16 <= S && (MODE != HC_SCORE_SNAPKV || key0 + 16 - 1 <= qpos0) && kd.zero == 0;
      // compiled apart, so that the common form is straight-line code
      const uint32_t redo = plain ? row_blocks(kd, key0, lane, std::true_type{}, std::false_type{})
                                  : row_blocks(kd, key0, lane, std::false_type{}, std::false_type{});
      // (with every row block open, as where logits cancel to a few bits, the
      // chain's loop does them faster)
      if (NRB > 1 && redo == (1u << NRB) - 1) hard |= 1u << c;
      else redo_tiles(redo, key0);
      key0 += CHUNK;
    }
  for (uint32_t left = wide; left;) {
    __asm__ volatile("" ::: "memory");
    const int c = __ffs(left) - 1, at = chunk(c);
    left &= left - 1;
    load(at);                    // (not ahead: the fifth digit takes the registers)
    KDigits<T, D> kd;
    kd.scan(raw);
    if (kd.held) {               // wave-uniform
      kd.template digits<true>(raw);
      int l = lane;              // (as in chain_tiles: nothing hoisted)
      __asm__ volatile("" : "+v"(l));
      redo_tiles(row_blocks(kd, at, l, std::false_type{}, std::true_type{}), at);
      continue;
    }
    hard |= 1u << c;
    if (__popc(hard) == 2 && hard == (wide & ~left)) {
      hard = wide;
      break;
    }
  }

  // The hard chunks, PB row blocks' queries in LDS at a time (in place of the
  // digits).
  if (hard && lane == 0) hard_s = 1;
  __syncthreads();
  if (hard_s) {                  // workgroup-uniform
    const doublex2* sx = reinterpret_cast<const doublex2*>(sq);
    for (int wt = 0; wt < nw; wt += 16 * PB) {
      const i32x4* src = reinterpret_cast<const i32x4*>(qrows + wt * D);
      for (int i = tid; i < SQ_CHAIN; i += 256) sq[i] = src[i];
      __syncthreads();
      uint32_t left = hard;
      float top[PB][4];
#pragma unroll
      for (int t = 0; t < PB; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) top[t][i] = -INFINITY;
      if (left) load(chunk(__ffs(left) - 1));
      while (left) {             // wave-uniform
        const int at = chunk(__ffs(left) - 1);
        left &= left - 1;
        uint32_t cur[NP][4];
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
          for (int i = 0; i < 4; ++i) cur[p][i] = raw[p][i];
        if (left) load(chunk(__ffs(left) - 1));
        chain_tiles<T, MODE, D, PB, 2>(cur, [&](int i, int u) { return sx[(i * (D / 8) + u) * 64 + lane]; }, lrs, ld,
                                       at, w0, wt, nw, qpos0, scaling, top);
      }
      if (hard) fold(top, wt);
      __syncthreads();
    }
  }

  if constexpr (MODE != HC_SCORE_SNAPKV) return;
  key0 = chunk(nmul);
  for (int c = nmul; c < nch && key0 <= qpos0 + nw - 1 + kNeverRead; ++c) {   // wholly masked chunks
    const uint32_t ninf = __float_as_uint(-INFINITY);
#pragma unroll
    for (int nb = 0; nb < NRB; ++nb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int w = 16 * nb + col, key = key0 + 4 * kk + i;
        bstore<4>(lrs, key < ld && w < nw ? (uint32_t)((w0 + w) * ld + key) * 4u : kOob, &ninf);
      }
    key0 += CHUNK;
  }
#pragma unroll
  for (int nb = 0; nb < NRB; ++nb) {
    const float m = __uint_as_float(reduce_rows(__float_as_uint(mrow[nb]), MaxF32{}));
    if (kk == 0) atomicMax(&redk[16 * nb + col], order_key(m));
  }
  __syncthreads();
  if (tid < nw) atomicMax(&rmax[bh * W + w0 + tid], redk[tid]);
}

}  // namespace hc
