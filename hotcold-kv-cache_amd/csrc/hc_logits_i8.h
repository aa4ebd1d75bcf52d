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
//   * query digits below the window: at most (sum of the residuals) * ||k||;
//   * key digits below the window: such a tile's bound is taken as infinite.
// With delta the sum of these, a logit whose dot product -delta and +delta
// round to one float is that float; a 16 x 16 tile with any other logit is
// recomputed by the fp64 chain itself (redo_tile).  Infinities and NaN take
// the same way.  On N(0,1) prompts about 1% of the tiles are redone (22.9k of
// 1.6M in the H2O launch below, before the bound was weighted by q').
//
// What it buys: the fp64 matrix rate is 32 flop per cycle and SIMD, 1/64 of
// int8's, so 16 products cost a quarter of the one fp64 product.  Kernel times
// (fp64 form -> this one, 8 KV heads of 128): window 64, 32k keys x 16 rows
// f16 1243 -> 685 us, 64k x 4 bf16 with outlier channels 650 -> 419; window
// 32, 32 layers of 8k keys 343 -> 207, one layer 21.6 -> 19.9 (bound by
// latency); 32 heads of 5003 x 5003 (H2O) 1977 -> 1172.  What bounds it:
// vector issue (per 16 keys x 64 rows about 270 instructions make the key
// digits and 350 the logits, beside 128 matrix instructions of 16 cycles that
// hide two vector instructions each) and the logits' stores, which are 14% of
// the 32k launch and 27% of the H2O one.  Measured no faster: two key tiles
// per wave, four waves per SIMD (spills), a row block's products interleaved
// with the logits of the one before, and the keys' digits made once for all
// row blocks.
#pragma once
#include <type_traits>

#include "hc_common.h"

namespace hc {

typedef int i32x4 __attribute__((ext_vector_type(4)));
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

// The group-mean queries with their digits: qf[b][h][w][d] as qmean_kernel
// writes it (zero rows past W), and its resets of the row maxima, the NaN flag
// and the padding statistics.  grid (wpad / 4, Hk, B), block 256, one wave per row;
// lane l owns dims E l .. E l + E - 1.  A digit byte of row w lies where the B
// operand reads it: [row block of 16][digit][k-step of 64][lane][16], lane
// (kk, row) holding dims 8 * (kk + 4 * t) + r of the pieces t = 2s, 2s + 1 of
// k-step s.  Bound by its stores (the fp64 means and 4 bytes of digits per
// element): 99 us for 32 heads of 5003 rows, 78 without the digits; a block of
// D threads per row with bounds reduced in fp64 across waves took 170.
template <typename T, int D>
__global__ __launch_bounds__(256) void qdigit_kernel(const T* __restrict__ q, const T* const* __restrict__ q_rows,
                                                     int64_t q_sb, int64_t q_sh, int64_t q_ss, int64_t q_row0, int Hq,
                                                     int Hk, int W, int wpad, double* __restrict__ qf,
                                                     uint32_t* __restrict__ rmax, RowStat* __restrict__ rstat,
                                                     uint32_t* __restrict__ nan_flag, int8_t* __restrict__ qd,
                                                     QDigitRow* __restrict__ qrow) {
  constexpr int E = D / 64;
  const int lane = threadIdx.x & 63, w = (int)blockIdx.x * 4 + (threadIdx.x >> 6), h = blockIdx.y, b = blockIdx.z;
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
    qf[(row + w) * D + lane * E + e] = x[e];
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
  int8_t* dst = qd + row * D * kDigits +
                ((int64_t)(w >> 4) * kDigits * (D / 64) + (t >> 1)) * 1024 + (((d >> 3) & 3) * 16 + (w & 15)) * 16 +
                (t & 1) * 8 + (d & 7);
#pragma unroll
  for (int j = 0; j < kDigits; ++j)
#pragma unroll
    for (int e = 0; e < E; ++e) dst[(int64_t)j * (D / 64) * 1024 + e] = (int8_t)(u[e] >> (8 * j));
  ss = __uint_as_float(reduce_cols(reduce_rows(__float_as_uint(ss), SumF32{}), SumF32{}));
  res = __uint_as_float(reduce_cols(reduce_rows(__float_as_uint(res), SumF32{}), SumF32{}));
  if (lane == 0) {
    // rounded up, past what the fp32 sums lose, to underflow too
    const float up = 1.f + 0x1p-14f, tiny = 1e-17f;
    QDigitRow r;
    r.scale = use ? ldexp(1.0, -sh) : 1.0;
    r.norm = hi == 0 || use ? sqrtf(ss) * up + tiny : INFINITY;
    r.resid = res * up + 2e-36f;
    qrow[row + w] = r;
  }
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
  int f;        // scale 2^(f - kShift)
  float norm;   // +inf if an element is not held exactly

  __device__ __forceinline__ void convert(const uint32_t (&w)[NP][4]) {
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
    const uint32_t hi = reduce_cols(reduce_rows(__builtin_bit_cast(uint32_t, mx), MaxU16x2{}), MaxU16x2{});
    const int mb = __builtin_amdgcn_readfirstlane((int)max(hi & 0xffffu, hi >> 16));
    // a mantissa at 2 - 2^-7 or above would pass kFixMax
    f = max((mb + (1 << (F::kMant - 7))) >> F::kMant, F::kMinF);
    bool exact = mb < F::kInf;
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
      const int nb = 0x10000 - (int)max(lo & 0xffffu, lo >> 16);
      exact = exact && max(nb >> F::kMant, 1) >= f - (30 - F::kMant);
    }
    const float mult = __uint_as_float((uint32_t)(127 + F::kShift - f) << 23);
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        uint32_t u[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          u[i] = (uint32_t)(int)__builtin_fmaf(F::get(w[p][2 * h + (i >> 1)], i & 1), mult, 0.f) + kBalance;
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
      }
    // An fp32 sum of D squares and its root: within 2^-14.  Half subnormals,
    // which the dot product may take as zero, are below sqrt(D) * 2^-14.
    ss = __uint_as_float(reduce_cols(reduce_rows(__float_as_uint(ss), SumF32{}), MaxF32{}));
    const float n = sqrtf(ss) * (1.f + 0x1p-14f) + 0x1p-10f;
    norm = exact ? n : INFINITY;
  }
};

// One 16-key x 16-row tile by the defining fp64 chain (keys key0.., rows wt..
// of the workgroup's block at window row w0; qf at the tile's first row):
// stores its logits and folds its row maxima into redk.
template <typename T, int MODE, int D>
__device__ __forceinline__ void redo_tile(__amdgpu_buffer_rsrc_t krs, uint32_t rowb, const double* qf,
                                       __amdgpu_buffer_rsrc_t lrs, int S, int ld, int key0, int w0, int wt, int nw,
                                       int qpos0, double scaling, uint32_t* redk) {
  typedef double doublex4 __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63, col = lane & 15, kk = lane >> 4;
  const uint32_t koff = key0 + col < S ? (uint32_t)(key0 + col) * rowb + 2u * kk : kOob;
  const double* qr = qf + col * D + kk;   // zero rows past the window
  const int w = wt + col;
  doublex4 acc = {0.0, 0.0, 0.0, 0.0};
  // every operand in flight at once: in four batches the loads' round trips
  // were most of the tile's time (with the tighter norm of QDigitRow 4% of the
  // f16 launches' time and 10% of the bf16 one's)
  uint32_t kw[D / 4];
  double q[D / 4];
#pragma unroll
  for (int t = 0; t < D / 4; ++t) {
    kw[t] = __builtin_amdgcn_raw_buffer_load_b16(krs, (int)koff, t * 8, 0);
    q[t] = qr[t * 4];
  }
#pragma unroll
  for (int t = 0; t < D / 4; ++t)
    acc = __builtin_amdgcn_mfma_f64_16x16x4f64((double)KFix<T>::get(kw[t], 0), q[t], acc, 0, 0, 0);
  float m = -INFINITY;
#pragma unroll
  for (int i = 0; i < 4; ++i) {   // keys kk + 4i, row col
    const int key = key0 + kk + 4 * i;
    float L;
    if constexpr (MODE == HC_SCORE_SNAPKV) L = key > qpos0 + w ? -INFINITY : (float)(acc[i] * scaling);
    else L = (float)(acc[i] / scaling);
    const bool ok = key < ld && w < nw;
    const uint32_t bits = __float_as_uint(L);
    bstore<4>(lrs, ok ? (uint32_t)((w0 + w) * ld + key) * 4u : kOob, &bits);
    m = fmaxf(m, ok ? L : -INFINITY);
  }
  if (w < nw) atomicMax(&redk[w], order_key(m));
}

// The logits kernel.  grid (ceil(S / (64 * cpw)), Hk * ceil(W / (16 * NRB)),
// B), block 256; workgroup order, causal skips and stores' extent as
// logits_kernel's.  Each wave owns 16 keys of a chunk: their digits stay
// in registers while the row blocks' digits come from LDS, 16 rows at a time.
// Keys are the A operand, so a lane's four results are consecutive keys of one
// row: one 16-byte store.  The next chunk's keys are loaded while this one is
// multiplied.
template <typename T, int MODE, int D, int NRB>
__global__ __launch_bounds__(256, 3) void logits_i8_kernel(
    const T* __restrict__ k, const T* const* __restrict__ k_rows, int64_t k_sb, int64_t k_sh, int64_t k_ss,
    uint32_t k_bytes, const double* __restrict__ qf, const int8_t* __restrict__ qd,
    const QDigitRow* __restrict__ qrow, int Hk, int S, int W, int wpad, double scaling, int cpw, int ld,
    float* __restrict__ logits, uint32_t* __restrict__ rmax) {
  constexpr int ROWS = 16 * NRB, NS = D / 64, NP = D / 32, CHUNK = kDigitChunk;
  __shared__ i32x4 sq[NRB * kDigits * NS * 64];
  __shared__ double ssc[ROWS];       // row scale times the logit scale
  __shared__ double sdel[NRB];       // a key of 2-norm 1's delta against the row block
  __shared__ uint32_t redk[ROWS];
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
  auto load = [&](int at) {
    const int key = at + col;
    const uint32_t off = key < S ? (uint32_t)key * rowb + 16u * kk : kOob;
#pragma unroll
    for (int p = 0; p < NP; ++p) bload_so<16>(krs, off, 64u * p, raw[p]);
  };
  load(key0);
  if (tid < ROWS) redk[tid] = order_key(-INFINITY);
  if (stage) {
    const i32x4* src = reinterpret_cast<const i32x4*>(qd + (bh * wpad + w0) * (int64_t)(D * kDigits));
#pragma unroll
    for (int i = tid; i < NRB * kDigits * NS * 64; i += 256) sq[i] = src[i];
    const double lscale = MODE == HC_SCORE_SNAPKV ? scaling : 1.0 / scaling;
    if (tid < ROWS) {
      const QDigitRow r = qrow[bh * wpad + w0 + tid];
      ssc[tid] = r.scale * lscale;
      double dl = (double)r.norm * 0x1p-53 + (double)r.resid;
#pragma unroll
      for (int o = 8; o > 0; o >>= 1) dl = fmax(dl, __shfl_xor(dl, o, 64));
      if (col == 0) sdel[tid >> 4] = dl * fabs(lscale) * 1.001;
    }
  }
  __syncthreads();

  const int nch = key0 < S ? min(cpw, (S - key0 + CHUNK - 1) / CHUNK) : 0;
  int nmul = nch;
  if constexpr (MODE == HC_SCORE_SNAPKV) {
    const int last = qpos0 + nw - 1;
    nmul = key0 > last ? 0 : min(nch, (last - key0) / CHUNK + 1);
  }
  float mrow[NRB];
#pragma unroll
  for (int i = 0; i < NRB; ++i) mrow[i] = -INFINITY;

  for (int c = 0; c < nmul; ++c) {
    // the row blocks' LDS reads repeat for every chunk: hoisted, they would
    // hold registers for the kernel's lifetime
    __asm__ volatile("" ::: "memory");
    KDigits<T, D> kd;
    kd.convert(raw);
    load(key0 + CHUNK);
    // every key at or before every row's position, none past S
    const bool plain = key0 + 16 <= S && (MODE != HC_SCORE_SNAPKV || key0 + 16 - 1 <= qpos0);
    uint32_t redo = 0;
    // The products of row block nb against the chunk's keys.
    auto multiply = [&](i32x4 (&acc)[2 * kDigits - 1], int nb) {
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
      }
    };
    // Their logits: stored, or the tile marked for redo_tile.
    auto finish = [&](const i32x4 (&acc)[2 * kDigits - 1], int nb, auto plain_c) {
      constexpr bool PLAIN = decltype(plain_c)::value;
      const int w = 16 * nb + col;
      const double rs = ssc[w], dl = sdel[nb];
      const uint64_t live = ((1ull << min(max(nw - 16 * nb, 0), 16)) - 1) * 0x0001000100010001ull;   // real rows' lanes
      const double del = dl * (double)kd.norm;
      const double sc = rs * __hiloint2double((1023 + kd.f - KFix<T>::kShift) << 20, 0);
      const int key = key0 + 4 * kk;
      float L[4];
      bool open = false;       // a logit that delta does not settle
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t0 = (acc[6][i] << 8) + acc[5][i];
        const int t1 = (acc[4][i] << 8) + acc[3][i];
        const int t2 = (acc[2][i] << 8) + acc[1][i];
        const double d = __builtin_fma(__builtin_fma(__builtin_fma((double)t0, 65536.0, (double)t1), 65536.0,
                                                     (double)t2), 256.0, (double)acc[0][i]);
        const float lo = (float)__builtin_fma(d, sc, -del);
        L[i] = (float)__builtin_fma(d, sc, del);
        bool bad = !(lo == L[i]);
        if constexpr (!PLAIN) {
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
    auto row_blocks = [&](auto plain_c) {
#pragma unroll
      for (int nb = 0; nb < NRB; ++nb) {
        i32x4 acc[2 * kDigits - 1];
        multiply(acc, nb);
        finish(acc, nb, plain_c);
      }
    };
    // compiled apart, so that the common form is straight-line code
    if (plain) row_blocks(std::true_type{});
    else row_blocks(std::false_type{});
    while (redo) {               // wave-uniform
      const int nb = __ffs(redo) - 1;
      redo &= redo - 1;
      redo_tile<T, MODE, D>(krs, rowb, qf + (bh * wpad + w0 + 16 * nb) * D, lrs, S, ld, key0, w0,
                            16 * nb, nw, qpos0, scaling, redk);
    }
    key0 += CHUNK;
  }

  if constexpr (MODE != HC_SCORE_SNAPKV) return;
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
