// fp32-accurate matrix products on the fp16 matrix cores, and the wave-level
// Polar-Express built on them (fp32 compute mode).
//
// An fp32 operand x, scaled by a power of two into fp16's range, is held as
// two fp16 numbers, hi = fp16(s x) and lo = fp16(s x - hi): together 22 to 23
// significant bits while s x is above 2^-3 (lo ends at fp16's 2^-24), one less
// for each power of two below that, none under 2^-25.  With the largest at 2^12
// to 2^15 that is about 2^-16 of it.  So the columns (the longer side) of
// Polar-Express and its VJP carry scales of their own, at any size down to 2^-60
// of the largest; rows share their matrix's scale: a row's result keeps fp32's
// relative accuracy while the row is above about 2^-20 of the largest (the steps
// lift it), and is accurate relative to the matrix below that.
// A product takes three MFMAs with fp32 accumulation,
// lo hi + hi lo + hi hi (the dropped lo lo is below 2^-24 of the operands'
// product).  Each v_mfma_f32_32x32x16_f16 adds 16 exact products to the fp32
// accumulator where v_mfma_f32_32x32x2f32 rounds after every two, so the sums
// carry fewer roundings; measured against 64 bits the errors of Polar-Express
// are smaller than with fp32 operands (figures at PESplit).  Rate: 16 of the
// contraction in 3 x 32 cycles against 8 x 64.
#pragma once

#include "atlas_common.hpp"

namespace atlas {

// hi and lo of the eight elements of K-block kb of a C-layout tile times s (a
// power of two: exact).
struct SFrag {
  f16x8 hi, lo;
};
__device__ __forceinline__ int opaque_lane() {
  int l = lane_id();
  asm volatile("" : "+v"(l));
  return l;
}
// (The pair is opaque between the conversion and the subtraction: formed
// twice, by two different instructions, a hi on a rounding boundary could
// differ from the one that lo completes.)
__device__ __forceinline__ void split2(float x0, float x1, float s, f16x2& hi, f16x2& lo) {
  hi = f16x2{(_Float16)(x0 * s), (_Float16)(x1 * s)};
  asm("" : "+v"(hi));
  lo = f16x2{(_Float16)fmaf(x0, s, -(float)hi[0]), (_Float16)fmaf(x1, s, -(float)hi[1])};
}
__device__ __forceinline__ SFrag split_c(const f32x16& t, int kb, float s) {
  SFrag f;
#pragma unroll
  for (int v = 0; v < 8; v += 2) {
    f16x2 hi, lo;
    split2(t[8 * kb + v], t[8 * kb + v + 1], s, hi, lo);
    f.hi[v] = hi[0]; f.hi[v + 1] = hi[1];
    f.lo[v] = lo[0]; f.lo[v + 1] = lo[1];
  }
  return f;
}
// c += a b to fp32 accuracy, the small terms first
__device__ __forceinline__ f32x16 mma_split(const SFrag& a, const SFrag& b, f32x16 c) {
  c = ModeF16::mma(a.lo, b.hi, c);
  c = ModeF16::mma(a.hi, b.lo, c);
  return ModeF16::mma(a.hi, b.hi, c);
}

// k with 2^k times the largest entry of this lane's column (TI C-layout tiles)
// in [2^(top - 1), 2^top), at most 100 + top (a column of zeros: top).
template <int TI>
__device__ __forceinline__ int column_exponent(const f32x16 (&t)[TI], int top) {
  float m = 0.f;
#pragma unroll
  for (int I = 0; I < TI; ++I)
#pragma unroll
    for (int r = 0; r < 16; ++r) m = fmaxf(m, fabsf(t[I][r]));
  float m0, m1;
  swap32(m, m0, m1);   // the other rows lie in the other half
  return top + min(-__builtin_amdgcn_frexp_expf(fmaxf(m0, m1)), 100);
}

// Per-step factors of the split Polar-Express.  The iterate is carried as
// X_s = mu X, mu_0 = 2^30, mu <- mu / a each step (so the step needs no a X
// multiply, as in polar_express_wave_t).  Its operand is x = sx X_s, the Gram
// accumulates nu^2 G (nu = sx mu), its operand is g = sg nu^2 G = gamma G; then
//   R = gamma^2 (G^2 + (b/c) G)   accumulated onto kappa (nu^2 G),
//   r = rho R = 2^15 (B / a)      an operand of the update X_s <- X_s + r (2^-15 X_s).
// All scales are powers of two chosen so that every operand's largest entry
// (|X|, |G|^(1/2) <= 2, |B / a| <= 1 over the iteration) stays below 2^15 (r: at
// most 2^15).  Each column of X_s is carried times a power of two 2^k of its own
// (its largest entry 2^26 to 2^27 at first, so that its norm, which the steps do not
// increase, stays below 2^30): the update works on columns, so a column far below
// the others keeps its bits; only the Gram's operands are scaled back by 2^-k.
struct PEScale {
  float sx, sg, kappa, rho;
};
constexpr float PE_XU = 1.f / 32768.f;   // X_s as the update's operand
constexpr double kPEd64[5][3] = {
    {8.156554524902461, -22.48329292557795, 15.878769915207462},
    {4.042929935166739, -2.808917465908714, 0.5000178451051316},
    {3.8916678022926607, -2.772484153217685, 0.5060648178503393},
    {3.285753657755655, -2.3681294933425376, 0.46449024233003106},
    {2.3465413258596377, -1.7097828382687081, 0.42323551169305323},
};
constexpr double pe_pow2(int e) { return e == 0 ? 1.0 : e > 0 ? 2.0 * pe_pow2(e - 1) : 0.5 * pe_pow2(e + 1); }
constexpr double pe_mu(int st) { return st == 0 ? pe_pow2(30) : pe_mu(st - 1) / kPEd64[st - 1][0]; }
constexpr PEScale pe_scale(int st) {
  const double sx = pe_pow2(-15 + st), nu = sx * pe_mu(st);   // nu: 2^15, 2^13, 2^12, 2^11, 2^10 (rounded up)
  double sg = 1.0;
  while (sg * nu * nu > 4096.0) sg *= 0.5;                    // gamma in (2^11, 2^12]
  const double gamma = sg * nu * nu, a = kPEd64[st][0], b = kPEd64[st][1], c = kPEd64[st][2];
  return {(float)sx, (float)sg, (float)(b / c * gamma * gamma / (nu * nu)), (float)(32768.0 * c / (a * gamma * gamma))};
}
__constant__ static const PEScale kPEsplit[5] = {pe_scale(0), pe_scale(1), pe_scale(2), pe_scale(3), pe_scale(4)};
__constant__ static const float kPEmu[6] = {(float)(1.0 / pe_mu(0)), (float)(1.0 / pe_mu(1)), (float)(1.0 / pe_mu(2)),
                                            (float)(1.0 / pe_mu(3)), (float)(1.0 / pe_mu(4)), (float)(1.0 / pe_mu(5))};

// The pieces of one wave's split Polar-Express on a D x E matrix (D <= E) in
// C-layout tiles.  Per step at 64 x 128, 204 products of 32 cycles and about
// 1100 VALU instructions (the splits) against 80 x 512 cycles with fp32
// operands: 4 096 matrices, 5 steps, 546 -> 147 us (two waves per SIMD), 64 x
// 64 (16 384 matrices) 1166 -> 315 us.  Bound by the products at the clock the
// power limit leaves and by the latency between the dependent ones.  Relative
// error against 64 bits, fp32 operands -> split: random 64 x 128 3.05e-6 ->
// 2.60e-6, momentum-like (singular values over 2^-60) 3.73e-5 -> 2.48e-5; 32 x
// 32 2.37e-6 -> 1.79e-6, 2.13e-5 -> 1.53e-5.  xs: ELEMS halves of LDS per wave, one 32-column block of X
// as fp16 rows e of D halves, hi and lo, unpadded: the 8-byte units of row e
// are permuted by the row so that the staging writes (32 rows, one unit each)
// and the transposing reads (4 rows x 16 columns per 16 lanes) touch every
// bank once.
template <int D, int E>
struct PESplit {
  static constexpr int TI = D / 32, TJ = E / 32;
  static constexpr int BLOCK = 32 * D;
  static constexpr int ELEMS = 2 * BLOCK;
  static_assert(D == 32 || D == 64 || D == 96 || D == 128, "units per row");

  // 8-byte unit u of row r lies at u ^ g(r).  The low three bits of g are r / 4
  // (eight different units of a write to rows that share their banks); where
  // the four rows of a transposing read share banks too (two rows span them at
  // D 64, one at D 128), the bits above separate those.
  __device__ __forceinline__ static int at(int r, int u) {
    const int g = (r >> 2 & 7) | (D == 64 ? (r >> 1 & 1) << 3 : D == 128 ? (r & 3) << 3 : 0);
    return r * D + 4 * (u ^ g);
  }
  __device__ __forceinline__ static void put4(const f32x16& t, int q, float s, _Float16* p) {
    f16x2 h0, l0, h1, l1;
    split2(t[4 * q], t[4 * q + 1], s, h0, l0);
    split2(t[4 * q + 2], t[4 * q + 3], s, h1, l1);
    const f16x4 hi{h0[0], h0[1], h1[0], h1[1]}, lo{l0[0], l0[1], l1[0], l1[1]};
    *reinterpret_cast<f16x4*>(p) = hi;
    *reinterpret_cast<f16x4*>(p + BLOCK) = lo;
  }
  // column block J of X: lane (c, h) writes d = 32I + 8q + 4h + 0..3 of row c
  // (ln: the lane, which a caller may pass through an opaque value so that the
  // offsets are formed where they are used instead of held across its loops)
  __device__ __forceinline__ static void put_block(const f32x16 (&X)[TI][TJ], int J, float s, _Float16* xs,
                                                   int ln = lane_id()) {
    const int c = ln & 31, h = ln >> 5;
#pragma unroll
    for (int I = 0; I < TI; ++I)
#pragma unroll
      for (int q = 0; q < 4; ++q) put4(X[I][J], q, s, xs + at(c, 8 * I + 2 * q + h));
  }
  __device__ __forceinline__ static f16x8 tr2(const _Float16* lo_p, const _Float16* hi_p) {
    const f16x4 a = lds_read_tr16(lo_p), b = lds_read_tr16(hi_p);
    return f16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
  }
  // Gram fragment: lane l holds X[32I + l % 32][columns 16 kb + 8 (l / 32) + v of the block]
  __device__ __forceinline__ static SFrag get(const _Float16* xs, int I, int kb, int l = lane_id()) {
    const int j = l & 15, r = 16 * kb + 8 * (l >> 5) + (j >> 2), u = 8 * I + 4 * ((l >> 4) & 1) + (j & 3);
    const _Float16 *p = xs + at(r, u), *p4 = xs + at(r + 4, u);
    return {tr2(p, p4), tr2(p + BLOCK, p4 + BLOCK)};
  }
  // A 32 x 32 C-layout tile times s, transposed: fragments with k in C-layout order
  __device__ __forceinline__ static void put_tile(const f32x16& t, float s, _Float16* xs, int ln = lane_id()) {
    const int c = ln & 31, h = ln >> 5;
#pragma unroll
    for (int q = 0; q < 4; ++q) put4(t, q, s, xs + at(c, 2 * q + h));
  }
  __device__ __forceinline__ static SFrag get_tile(const _Float16* xs, int kb, int l = lane_id()) {
    const int j = l & 15, r = 16 * kb + 4 * (l >> 5) + (j >> 2), u = 4 * ((l >> 4) & 1) + (j & 3);
    const _Float16 *p = xs + at(r, u), *p8 = xs + at(r + 8, u);
    return {tr2(p, p8), tr2(p + BLOCK, p8 + BLOCK)};
  }

  // exponent k of this lane's column of block J (ke: four signed bytes)
  __device__ __forceinline__ static int column_exp(int ke, int J) { return (ke << (24 - 8 * J)) >> 24; }

  // nu^2 G, upper tiles (I, I2 >= I)
  __device__ __forceinline__ static void gram(const f32x16 (&X)[TI][TJ], f32x16 (&A)[TI][TI], float sx, int ke, _Float16* xs) {
#pragma unroll
    for (int J = 0; J < TJ; ++J) {
      put_block(X, J, __builtin_amdgcn_ldexpf(sx, -column_exp(ke, J)), xs);
      SFrag th[TI][2];
#pragma unroll
      for (int I = 0; I < TI; ++I)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) th[I][kb] = get(xs, I, kb);
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int I = 0; I < TI; ++I)
#pragma unroll
          for (int I2 = I; I2 < TI; ++I2)
            A[I][I2] = mma_split(th[I][kb], th[I2][kb], (J == 0 && kb == 0) ? zero16() : A[I][I2]);
    }
  }

  // operand fragments of a symmetric matrix from its upper C tiles times s
  // (tile (1, 0) as the transpose of (0, 1) through xs)
  __device__ __forceinline__ static void sym_frags(const f32x16 (&A)[TI][TI], float s, SFrag (&f)[TI][TI][2], _Float16* xs) {
    if constexpr (TI == 2) put_tile(A[0][1], s, xs);
#pragma unroll
    for (int I = 0; I < TI; ++I)
#pragma unroll
      for (int I2 = I; I2 < TI; ++I2)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) f[I][I2][kb] = split_c(A[I][I2], kb, s);
    if constexpr (TI == 2) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) f[1][0][kb] = get_tile(xs, kb);
    }
  }

  // X_s <- X_s + r x for step st from the Gram's upper tiles (consumed)
  __device__ __forceinline__ static void apply(f32x16 (&X)[TI][TJ], f32x16 (&A)[TI][TI], const PEScale& k, _Float16* xs) {
    SFrag f[TI][TI][2];
    sym_frags(A, k.sg, f, xs);
#pragma unroll
    for (int I = 0; I < TI; ++I)
#pragma unroll
      for (int I2 = I; I2 < TI; ++I2) A[I][I2] *= k.kappa;
    // (G^2)[I][I2] = sum_K G[I][K] G[K][I2]: tile (K, I) is the A operand G[I][K], tile (K, I2) the B operand
#pragma unroll
    for (int K = 0; K < TI; ++K)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int I = 0; I < TI; ++I)
#pragma unroll
          for (int I2 = I; I2 < TI; ++I2) A[I][I2] = mma_split(f[K][I][kb], f[K][I2][kb], A[I][I2]);
    sym_frags(A, k.rho, f, xs);
#pragma unroll
    for (int J = 0; J < TJ; ++J) {
      SFrag xf[TI][2];
#pragma unroll
      for (int K = 0; K < TI; ++K) {
        asm volatile("" : "+v"(X[K][J]));   // split again rather than kept from the Gram's staging (registers)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) xf[K][kb] = split_c(X[K][J], kb, PE_XU);
      }
#pragma unroll
      for (int K = 0; K < TI; ++K)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int I = 0; I < TI; ++I) X[I][J] = mma_split(f[K][I][kb], xf[K][kb], X[I][J]);
    }
  }
};

// One matrix per wave, fp32 accuracy: X <- PolarExpress(X).
template <int D, int E>
__device__ __forceinline__ void polar_express_wave_split(f32x16 (&X)[D / 32][E / 32], int ns, float norm_eps, _Float16* xs) {
  using P = PESplit<D, E>;
  static_assert(D <= 64 && E <= 128, "column norms, packed exponents");
  float ss = 0.f;
#pragma unroll
  for (int I = 0; I < P::TI; ++I)
#pragma unroll
    for (int J = 0; J < P::TJ; ++J)
#pragma unroll
      for (int r = 0; r < 16; ++r) ss += X[I][J][r] * X[I][J][r];
  ss = wave_sum(ss);
  const float s = 1.f / (sqrtf(ss + norm_eps) * 1.01f + 1e-6f);
  int ke = 0;
#pragma unroll
  for (int J = 0; J < P::TJ; ++J) {
    float m = 0.f;
#pragma unroll
    for (int I = 0; I < P::TI; ++I)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        X[I][J][r] *= s;
        m = fmaxf(m, fabsf(X[I][J][r]));
      }
    float m0, m1;
    swap32(m, m0, m1);   // the column's other rows
    // 2^k m in [2^-4, 2^-3): the column's norm is below sqrt(D) / 8 <= 1 (a column of zeros: k = -3)
    const int k = min(-3 - __builtin_amdgcn_frexp_expf(fmaxf(m0, m1)), 90);
    ke |= (k & 255) << (8 * J);
#pragma unroll
    for (int I = 0; I < P::TI; ++I)
#pragma unroll
      for (int r = 0; r < 16; ++r) X[I][J][r] = __builtin_amdgcn_ldexpf(X[I][J][r], 30 + k);   // mu_0 = 2^30
  }
  for (int st = 0; st < ns; ++st) {
    const PEScale k = kPEsplit[st];
    f32x16 A[P::TI][P::TI];
    P::gram(X, A, k.sx, ke, xs);
    P::apply(X, A, k, xs);
  }
#pragma unroll
  for (int J = 0; J < P::TJ; ++J) {
    const float ps = __builtin_amdgcn_ldexpf(kPEmu[ns], -P::column_exp(ke, J));
#pragma unroll
    for (int I = 0; I < P::TI; ++I) X[I][J] *= ps;
  }
}

}  // namespace atlas
