// VJP of Polar-Express in fp32 accuracy on the fp16 matrix cores: operands as
// two fp16 numbers (atlas_pe_split.hpp), one workgroup of four waves per matrix
// (persistent over the batch).
//
// Wave w holds the 32-column blocks J = w, w + 4, .. of the iterate Y and of
// the cotangent G as fp32 C-layout tiles.  One step Y' = a Y + (b A + c A^2) Y,
// A = Y Y^T, backwards, for the cotangent G of Y':
//   G_Y = a G + B G + C Y,  B = b A + c A^2,  C = b Gs + c (Gs A + A Gs),
//   Gs = G Y^T + Y G^T,
// in three phases between barriers:
//   1  every wave's blocks of Y and G staged in LDS as split rows; wave 0 forms
//      the upper tiles of A, waves 1-3 one upper tile of Gs each (A and Gs are
//      symmetric), over all blocks;
//   2  A and Gs shared through LDS as operand fragments (every lane writes the
//      16 bytes that the same lane of another wave reads); wave 0 forms B,
//      waves 1-3 their tile of C;
//   3  B and C shared the same way; every wave updates its own blocks, whose
//      C tiles are the B operands as they are.
// The forward recompute has the same phases with one upper tile of A and B per
// wave.  G is brought to a largest entry in [1, 2) by a power of two before the
// first step and back after the normalisation (cotangents of any size, subnormal
// ones included).  As operands, Y and G staged for the Gram-like products and A
// and B have fixed scales (|Y| <= 2, |A| <= 4, |B| <= 8; G's is set again for each
// step), Gs and C the ones that the largest entry of Gs allows, and the columns of
// Y and G that B and C act on one each, so that columns far below the others keep
// their bits (rows down to about 2^-20 of the largest do).
// Y_1 .. Y_{ns-3} go to the workgroup's global scratch, Y_{ns-2} stays in
// registers, Y_0 is X / nrm again.
//
// 4 096 matrices of 64 x 128, 5 steps: 2908 -> 650 us against fp32 MFMA on
// element-wise LDS operands (one workgroup per CU; the split tiles leave room
// for two), 2 048 of 64 x 256: 7.2 -> 0.85 ms (one scale for all columns and
// fixed ones for Gs and C: 640 us, 0.79 ms, with the small columns' bits lost).  About 1000 products of 32
// cycles per SIMD and matrix; the barriers between the phases, with waves idle
// where a phase has fewer tiles than waves, bound it.  Addresses and fragments
// are kept from being hoisted (opaque lanes, fences): hoisted, 244 registers
// spilled and it took twice as long.  Error against 64 bits 1.29e-5 -> 9.1e-6
// (random X), 1.09e-6 -> 6.7e-7 (momentum-like).
#pragma once

#include "atlas_pe_split.hpp"

// keeps later fragments' loads from being hoisted over the products (registers)
#define PE_FENCE() __builtin_amdgcn_sched_barrier(0)

namespace atlas {

template <int D, int E>
struct VjpSplit {
  static constexpr int TI = D / 32, NB = E / 32;
  static constexpr int BPW = NB > 4 ? NB / 4 : 1;          // column blocks per wave
  static constexpr int BLK = PESplit<D, 32>::ELEMS;        // halves of a staged block (hi and lo)
  static constexpr int FR = TI * TI * 2 * 2 * 512;         // halves of a D x D matrix as fragments
  static constexpr int TSC = PESplit<32, 32>::ELEMS;       // transposing scratch of one tile
  static constexpr int STG = 2 * NB * BLK;
  static constexpr int MAIN = STG > 4 * FR ? STG : 4 * FR;
  static constexpr int NRED = 16;
  static constexpr size_t bytes() { return (size_t)(MAIN + 2 * TSC) * 2 + NRED * sizeof(float); }
  static constexpr int PER_CU = 2 * bytes() <= 160 * 1024 ? 2 : 1;
  // scratch floats of one workgroup
  static constexpr size_t scratch_floats(int ns) { return ns > 3 ? (size_t)(ns - 3) * D * E : 0; }
};

// e with 2^e m in [1, 2) (0 for 0, infinities and NaN)
__device__ __forceinline__ int vjp_exponent(float m) { return m > 0.f && m < INFINITY ? -ilogbf(m) : 0; }

template <int D, int E>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(VjpSplit<D, E>::PER_CU)))
pe_vjp_split_kernel(long long n, int ns, int tall, const float* X, float* G, float* scratch) {
  using V = VjpSplit<D, E>;
  using P = PESplit<D, 32>;
  using T32 = PESplit<32, 32>;
  constexpr int TI = V::TI, NB = V::NB, BPW = V::BPW;
  constexpr float YS = 4096.f, GS = 2048.f;   // scales of Y and of G with its largest entry in [1, 2)
  constexpr float AS = 2048.f;                // A (entries <= 4) as an operand: 2^11
  constexpr float BS = 4096.f;                // B (<= 8): 2^12
  extern __shared__ __attribute__((aligned(16))) _Float16 lds[];
  _Float16* yst = lds;                        // staged Y blocks
  _Float16* gst = lds + NB * V::BLK;          // staged G blocks
  _Float16 *fA = lds, *fG = lds + V::FR, *fB = lds + 2 * V::FR, *fC = lds + 3 * V::FR;
  float* red = reinterpret_cast<float*>(lds + V::MAIN + 2 * V::TSC);
  const int w = __builtin_amdgcn_readfirstlane(wave_id()), lane = lane_id();
  _Float16* tsc = lds + V::MAIN + (w == 0 ? 0 : V::TSC);   // (two waves at a time transpose a tile)
  float* scr = scratch + (long long)blockIdx.x * V::scratch_floats(ns);

  auto put_frag = [&](_Float16* m, int K, int I, int kb, const SFrag& f) {
    _Float16* p = m + ((K * TI + I) * 2 + kb) * 1024 + lane * 8;
    *reinterpret_cast<f16x8*>(p) = f.hi;
    *reinterpret_cast<f16x8*>(p + 512) = f.lo;
  };
  auto get_frag = [&](const _Float16* m, int K, int I, int kb) {
    const _Float16* p = m + ((K * TI + I) * 2 + kb) * 1024 + lane * 8;
    return SFrag{*reinterpret_cast<const f16x8*>(p), *reinterpret_cast<const f16x8*>(p + 512)};
  };
  // upper tile (I, I2) of a symmetric matrix times s as fragments, (1, 0) transposed from (0, 1)
  auto share = [&](_Float16* m, const f32x16& t, int I, int I2, float s) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) put_frag(m, I, I2, kb, split_c(t, kb, s));
    if (I != I2) {
      const int l = opaque_lane();
      T32::put_tile(t, s, tsc, l);
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) put_frag(m, I2, I, kb, T32::get_tile(tsc, kb, l));
    }
  };
  // the upper tiles first .. first + N - 1 of sum_e y_I y_I2^T over all staged blocks
  auto gram_tiles = [&](auto& A, int first) {
    constexpr int N = sizeof(A) / sizeof(f32x16);
    const int l = opaque_lane();
#pragma unroll
    for (int j = 0; j < N; ++j) A[j] = zero16();
#pragma unroll 1
    for (int J = 0; J < NB; ++J) {
      const _Float16* ys = yst + J * V::BLK;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        SFrag y[TI];
#pragma unroll
        for (int I = 0; I < TI; ++I) y[I] = P::get(ys, I, kb, l);
#pragma unroll
        for (int j = 0; j < N; ++j) {
          const int t = N > 1 ? j : first;
          if (t == 0) A[j] = mma_split(y[0], y[0], A[j]);
          else if (t == 1) A[j] = mma_split(y[0], y[TI - 1], A[j]);
          else A[j] = mma_split(y[TI - 1], y[TI - 1], A[j]);
        }
      }
    }
  };
  // tile (I, I2) of G Y^T + Y G^T over all staged blocks
  auto gs_tile = [&](int I, int I2) {
    const int l = opaque_lane();
    f32x16 S = zero16();
#pragma unroll 1
    for (int J = 0; J < NB; ++J) {
      const _Float16 *ys = yst + J * V::BLK, *gs = gst + J * V::BLK;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        S = mma_split(P::get(gs, I, kb, l), P::get(ys, I2, kb, l), S);
        S = mma_split(P::get(ys, I, kb, l), P::get(gs, I2, kb, l), S);
      }
    }
    return S;
  };
  // sum_K x[I][K] y[K][I2] of two shared symmetric matrices
  auto dd_tile = [&](const _Float16* x, const _Float16* y, int I, int I2, f32x16 acc) {
#pragma unroll
    for (int K = 0; K < TI; ++K)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        acc = mma_split(get_frag(x, K, I, kb), get_frag(y, K, I2, kb), acc);
        PE_FENCE();
      }
    return acc;
  };
  // upper tile number of wave job j: 0 (0,0), 1 (0,1), 2 (1,1)
  auto tI = [](int j) { return j == 2 ? 1 : 0; };
  auto tI2 = [](int j) { return j == 0 ? 0 : 1; };
  constexpr int NT = TI == 2 ? 3 : 1;   // upper tiles

  typedef f32x16 Tiles[BPW][TI];
  auto own = [&](int q) { return w + 4 * q < NB; };
  auto load = [&](Tiles& t, const float* x) {   // this wave's blocks of a D x E matrix (`tall`: stored E x D)
    const int l = opaque_lane(), c = l & 31, h = l >> 5;
#pragma unroll
    for (int q = 0; q < BPW; ++q)
#pragma unroll
      for (int I = 0; I < TI; ++I) {
        const int e = own(q) ? 32 * (w + 4 * q) + c : c;
        if (tall) {
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(x + e * D + 32 * I + 8 * g + 4 * h);
#pragma unroll
            for (int u = 0; u < 4; ++u) t[q][I][4 * g + u] = v[u];
          }
        } else {
#pragma unroll
          for (int r = 0; r < 16; ++r) t[q][I][r] = x[(32 * I + crow(r, h)) * E + e];
        }
      }
  };
  auto stage = [&](_Float16* st, const Tiles& t, float s) {
    const int l = opaque_lane();
#pragma unroll
    for (int q = 0; q < BPW; ++q)
      if (own(q)) {
        f32x16 b[TI][1];
#pragma unroll
        for (int I = 0; I < TI; ++I) b[I][0] = t[q][I];
        P::put_block(b, 0, s, st + (w + 4 * q) * V::BLK, l);
      }
  };
  auto scale2 = [&](Tiles& t, int e) {   // times 2^e
#pragma unroll
    for (int q = 0; q < BPW; ++q)
#pragma unroll
      for (int I = 0; I < TI; ++I)
#pragma unroll
        for (int r = 0; r < 16; ++r) t[q][I][r] = __builtin_amdgcn_ldexpf(t[q][I][r], e);
  };
  // the block's largest |t|, through red[8 ..] (a barrier: every wave's earlier LDS accesses are done)
  auto block_max4 = [&](const Tiles& t) {
    float mx = 0.f;
#pragma unroll
    for (int q = 0; q < BPW; ++q)
#pragma unroll
      for (int I = 0; I < TI; ++I)
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, own(q) ? fabsf(t[q][I][r]) : 0.f);
    mx = wave_max(mx);
    if (lane == 0) red[8 + w] = mx;
    __syncthreads();
    return fmaxf(fmaxf(red[8], red[9]), fmaxf(red[10], red[11]));
  };
  auto block_sum4 = [&](float x, int slot) {   // fixed order; slot: 4 floats of red
    x = wave_sum(x);
    if (lane == 0) red[slot + w] = x;
    __syncthreads();
    return (red[slot] + red[slot + 1]) + (red[slot + 2] + red[slot + 3]);
  };

  for (long long mi = blockIdx.x; mi < n; mi += gridDim.x) {
    const float* Xm = X + mi * (D * E);
    float* Gm = G + mi * (D * E);
    Tiles Y, Yp, Gb;
    load(Y, Xm);
    float ss = 0.f;
#pragma unroll
    for (int q = 0; q < BPW; ++q)
#pragma unroll
      for (int I = 0; I < TI; ++I)
#pragma unroll
        for (int r = 0; r < 16; ++r) ss += own(q) ? Y[q][I][r] * Y[q][I][r] : 0.f;
    const float nn = sqrtf(block_sum4(ss, 0) + 1e-12f);
    const float nrm = nn * 1.01f + 1e-6f, inv = 1.f / nrm;
#pragma unroll
    for (int q = 0; q < BPW; ++q)
#pragma unroll
      for (int I = 0; I < TI; ++I) Yp[q][I] = Y[q][I] *= inv;

    // ---- forward recompute: Y_0 .. Y_{ns-1}
    for (int k = 0; k + 1 < ns; ++k) {
      if (k >= 1 && k <= ns - 3) {
        f32x4* o = reinterpret_cast<f32x4*>(scr + (size_t)(k - 1) * D * E);
#pragma unroll
        for (int q = 0; q < BPW; ++q)
          if (own(q))
#pragma unroll
            for (int I = 0; I < TI; ++I)
#pragma unroll
              for (int g = 0; g < 4; ++g)
                o[(((w + 4 * q) * TI + I) * 4 + g) * WAVE + lane] =
                    f32x4{Y[q][I][4 * g], Y[q][I][4 * g + 1], Y[q][I][4 * g + 2], Y[q][I][4 * g + 3]};
      }
#pragma unroll
      for (int q = 0; q < BPW; ++q)
#pragma unroll
        for (int I = 0; I < TI; ++I) Yp[q][I] = Y[q][I];   // Y_k: Y_{ns-2} after the last step
      const float ka = kPE[k][0], kb_ = kPE[k][1], kc = kPE[k][2];
      stage(yst, Y, YS);
      __syncthreads();
      f32x16 A[1];
      if (w < NT) gram_tiles(A, w);
      __syncthreads();   // the staged blocks have been read
      if (w < NT) {
        A[0] *= 1.f / (YS * YS);
        share(fA, A[0], tI(w), tI2(w), AS);
      }
      __syncthreads();
      if (w < NT) {
        const f32x16 A2 = dd_tile(fA, fA, tI(w), tI2(w), zero16());
        A[0] = kb_ * A[0] + (kc / (AS * AS)) * A2;
        share(fB, A[0], tI(w), tI2(w), BS);
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < BPW; ++q)
        if (own(q)) {
          f32x16 acc[TI];
#pragma unroll
          for (int I = 0; I < TI; ++I) acc[I] = zero16();
          const int ey = column_exponent<TI>(Yp[q], 12);
          const float ys = __builtin_amdgcn_ldexpf(1.f, ey);
#pragma unroll
          for (int K = 0; K < TI; ++K)
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
              const SFrag y = split_c(Yp[q][K], kb, ys);
#pragma unroll
              for (int I = 0; I < TI; ++I) acc[I] = mma_split(get_frag(fB, K, I, kb), y, acc[I]);
              PE_FENCE();
            }
#pragma unroll
          for (int I = 0; I < TI; ++I) Y[q][I] = ka * Yp[q][I] + acc[I] * __builtin_amdgcn_ldexpf(1.f / BS, -ey);
        }
      __syncthreads();   // B has been read: the blocks may be staged over it
    }

    // ---- backward through the steps
    // G is brought to a largest entry in [1, 2) before the first step and back
    // after the normalisation: its own size may be any, subnormal included.
    load(Gb, Gm);
    const int eg = vjp_exponent(block_max4(Gb));
    scale2(Gb, eg);
    __syncthreads();   // red is written again
    for (int k = ns - 1; k >= 0; --k) {
      if (k + 1 < ns) {
        if (k == 0) {
          load(Y, Xm);
#pragma unroll
          for (int q = 0; q < BPW; ++q)
#pragma unroll
            for (int I = 0; I < TI; ++I) Y[q][I] *= inv;
        } else if (k == ns - 2) {
#pragma unroll
          for (int q = 0; q < BPW; ++q)
#pragma unroll
            for (int I = 0; I < TI; ++I) Y[q][I] = Yp[q][I];
        } else {
          const f32x4* o = reinterpret_cast<const f32x4*>(scr + (size_t)(k - 1) * D * E);
#pragma unroll
          for (int q = 0; q < BPW; ++q)
            if (own(q))
#pragma unroll
              for (int I = 0; I < TI; ++I)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                  const f32x4 v = o[(((w + 4 * q) * TI + I) * 4 + g) * WAVE + lane];
#pragma unroll
                  for (int u = 0; u < 4; ++u) Y[q][I][4 * g + u] = v[u];
                }
        }
      }
      const float sg = pow2_scale(block_max4(Gb)), isg = 1.f / sg;   // (its barrier: the previous step's B and C have been read)
      const float ka = kPE[k][0], kb_ = kPE[k][1], kc = kPE[k][2];
      stage(yst, Y, YS);
      stage(gst, Gb, sg * GS);
      __syncthreads();
      f32x16 A[NT], S;
      if (w == 0) {
        gram_tiles(A, 0);
      } else if (w <= NT) {
        S = gs_tile(tI(w - 1), tI2(w - 1));
        S *= 1.f / (GS * YS);   // Gs of sg G
      }
      {
        float gm = 0.f;
        if (w != 0 && w <= NT) {
#pragma unroll
          for (int r = 0; r < 16; ++r) gm = fmaxf(gm, fabsf(S[r]));
        }
        gm = wave_max(gm);
        if (lane == 0) red[12 + w] = gm;
      }
      __syncthreads();   // the staged blocks have been read
      // Gs as an operand: its largest entry to [2^13, 2^14); C at most 2^9 (first
      // step: |A| <= 1, |b| + 2 |c| sqrt(D) |A| < 2^9) or 2^6 times that of Gs
      const float SS = __builtin_amdgcn_ldexpf(
          1.f, min(14 - __builtin_amdgcn_frexp_expf(fmaxf(fmaxf(red[12], red[13]), fmaxf(red[14], red[15]))), 24));
      const float CS = SS * (k == 0 ? 1.f / 256.f : 1.f / 32.f);
      if (w == 0) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          A[j] *= 1.f / (YS * YS);
          share(fA, A[j], tI(j), tI2(j), AS);
        }
      } else if (w <= NT) {
        share(fG, S, tI(w - 1), tI2(w - 1), SS);
      }
      __syncthreads();
      if (w == 0) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
          const f32x16 A2 = dd_tile(fA, fA, tI(j), tI2(j), zero16());
          A[j] = kb_ * A[j] + (kc / (AS * AS)) * A2;
          share(fB, A[j], tI(j), tI2(j), BS);
        }
      } else if (w <= NT) {
        f32x16 t = dd_tile(fG, fA, tI(w - 1), tI2(w - 1), zero16());
        t = dd_tile(fA, fG, tI(w - 1), tI2(w - 1), t);
        S = kb_ * S + kc / (AS * SS) * t;
        share(fC, S, tI(w - 1), tI2(w - 1), CS);
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < BPW; ++q)
        if (own(q)) {
          f32x16 acc[TI];
#pragma unroll
          for (int I = 0; I < TI; ++I) acc[I] = zero16();
          // (exponents of columns 60 or more powers of two down are held there: the factor between the sums stays finite)
          const int eg_ = min(column_exponent<TI>(Gb[q], 12), 72), ey = min(column_exponent<TI>(Y[q], 12), 72);
          const float gs = __builtin_amdgcn_ldexpf(1.f, eg_), ys = __builtin_amdgcn_ldexpf(1.f, ey);
#pragma unroll
          for (int K = 0; K < TI; ++K)
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
              const SFrag g = split_c(Gb[q][K], kb, gs);
#pragma unroll
              for (int I = 0; I < TI; ++I) acc[I] = mma_split(get_frag(fB, K, I, kb), g, acc[I]);
              PE_FENCE();
            }
          const float bc = __builtin_amdgcn_ldexpf(sg * CS * (1.f / BS), ey - eg_);   // B G and C Y on one scale
#pragma unroll
          for (int I = 0; I < TI; ++I) acc[I] *= bc;
#pragma unroll
          for (int K = 0; K < TI; ++K)
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
              const SFrag y = split_c(Y[q][K], kb, ys);
#pragma unroll
              for (int I = 0; I < TI; ++I) acc[I] = mma_split(get_frag(fC, K, I, kb), y, acc[I]);
              PE_FENCE();
            }
          const float ss_ = __builtin_amdgcn_ldexpf(isg / CS, -ey);
#pragma unroll
          for (int I = 0; I < TI; ++I) Gb[q][I] = ka * Gb[q][I] + acc[I] * ss_;
        }
    }

    // ---- normalisation
    load(Y, Xm);
    float dot = 0.f;
#pragma unroll
    for (int q = 0; q < BPW; ++q)
#pragma unroll
      for (int I = 0; I < TI; ++I)
#pragma unroll
        for (int r = 0; r < 16; ++r) dot += own(q) ? Gb[q][I][r] * Y[q][I][r] : 0.f;
    const float coef = block_sum4(dot, 4) * 1.01f / (nrm * nrm * nn);
    const int ln = opaque_lane(), c = ln & 31, h = ln >> 5;
#pragma unroll
    for (int q = 0; q < BPW; ++q)
      if (own(q)) {
        const int e = 32 * (w + 4 * q) + c;
#pragma unroll
        for (int I = 0; I < TI; ++I) {
          f32x16 d = Gb[q][I] * inv - coef * Y[q][I];
#pragma unroll
          for (int r = 0; r < 16; ++r) d[r] = __builtin_amdgcn_ldexpf(d[r], -eg);
          if (tall) {
#pragma unroll
            for (int g = 0; g < 4; ++g)
              *reinterpret_cast<f32x4*>(Gm + e * D + 32 * I + 8 * g + 4 * h) =
                  f32x4{d[4 * g], d[4 * g + 1], d[4 * g + 2], d[4 * g + 3]};
          } else {
#pragma unroll
            for (int r = 0; r < 16; ++r) Gm[(32 * I + crow(r, h)) * E + e] = d[r];
          }
        }
      }
    __syncthreads();   // red and the fragments are free for the next matrix
  }
}

}  // namespace atlas
