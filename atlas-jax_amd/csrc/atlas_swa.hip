// Sliding-window causal attention with rotary embeddings: the attention of
// the MAG blocks (atlas_jax/model.py:83-133, SlidingWindowAttention.__call__
// between the qkv projection and to_out; used by MAGBlock,
// atlas_jax/mag_transformer.py:63-79).
//
// Per (b, h) and query t, with q', k' the half-split rotary rotation of q, k
// (model.py:64-73) and the mask of model.py:123-127 (causal, t - s <= window):
//   out_t = sum_s softmax_s(q'_t . k'_s / sqrt(D)) v_s.
//
// One workgroup per (b, h, block of 128 or 512 queries).  Keys and values of
// the window are streamed through LDS in blocks of 64.
// The score tile is formed transposed, S^T = K Q^T (keys along the C-layout
// rows, queries along the lanes), so that after the online softmax the
// probabilities are already the B operand of O^T = V^T P^T (the contraction
// index -- the key -- runs along the rows).  fp16 matrix-core operands, fp32
// accumulation, scores, softmax statistics and output scaling.
#include <hip/hip_runtime.h>

#include <math.h>

#include "atlas_common.hpp"
#include "atlas_scan.h"
#include "atlas_status.hpp"

namespace atlas {
namespace {

constexpr int SWA_D = 64;           // head dim
constexpr int SWA_BK = 64;          // keys per LDS block

struct SwaArgs {
  int B, T, H, window, io_dtype;
  long long sb, st, sh;             // q/k/v element strides
  const void *q, *k, *v;
  void* out;                        // (B, T, H, D) contiguous
  const float *cos_tab, *sin_tab;   // (T, D/2)
  float scale;
  float* lse;                       // (B, H, T) softmax log-normalisers of the scaled scores, or NULL
};

// ---- operand tiles: 64 tokens x 64 halves in LDS, unpadded -------------------
// Rows ([token][d], 128 bytes) serve two kinds of reads: contiguous 16-byte
// fragments along d (32 rows at once), and transposing reads of 4 rows x 16
// columns per 16-lane group.  Unpadded rows put every second row on the same
// banks, so 16-byte piece p of row r lies at p ^ f(r): f takes all eight
// values over the even (and the odd) rows of any 16, which keeps the
// contiguous reads free of conflicts, and its bit 2 differs between rows r and
// r + 2, which does the same for the transposing ones.
constexpr int SWA_TILE = SWA_BK * SWA_D;   // halves

__device__ __forceinline__ int row_piece(int r, int p) {
  return r * SWA_D + ((p ^ (((r >> 1 & 1) << 2) | (r >> 2 & 3))) << 3);
}
// This lane's offsets in the transposing reads of columns 32 I .. 32 I + 31:
// rows 4h + j / 4 and the same + 8, columns 32 I + 16 (lane / 16 % 2) + 4 (j % 4)
// (16 more rows leave the pieces' places alone).
struct TrOff {
  int lo[2], hi[2];
  __device__ __forceinline__ TrOff() {
    const int l = lane_id(), j = l & 15, r = 4 * (l >> 5) + (j >> 2);
#pragma unroll
    for (int I = 0; I < 2; ++I) {
      const int p = 4 * I + 2 * ((l >> 4) & 1) + ((j & 3) >> 1), u = 4 * (j & 1);
      lo[I] = row_piece(r, p) + u;
      hi[I] = row_piece(r + 8, p) + u;
    }
  }
};
// Fragment (lane = column 32 I + lane % 32, k = rows 32 kt + 16 kb .. in C-layout order)
__device__ __forceinline__ f16x8 ld_tr(const _Float16* tile, const TrOff& o, int I, int kt, int kb) {
  const _Float16* p = tile + (32 * kt + 16 * kb) * SWA_D;
  const f16x4 lo = lds_read_tr16(p + o.lo[I]), hi = lds_read_tr16(p + o.hi[I]);
  return f16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
}
// Fragment (lane = row 32 kt + c, k = d in 16 kb + 8 h + 0..7)
__device__ __forceinline__ f16x8 ld_row(const _Float16* tile, int kt, int kb, int c, int h) {
  return *reinterpret_cast<const f16x8*>(tile + row_piece(32 * kt + c, 2 * kb + h));
}
__device__ __forceinline__ void st_rows(_Float16* tile, int r, int p, f16x8 x1, f16x8 x2) {
  *reinterpret_cast<f16x8*>(tile + row_piece(r, p)) = x1;
  *reinterpret_cast<f16x8*>(tile + row_piece(r, p + 4)) = x2;
}

// 8 consecutive fp32 of a caller's table (any 4-byte alignment)
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ void ldtab8(const float* t, float (&r)[8]) {
  const f32x4u a = *reinterpret_cast<const f32x4u*>(t), b = *reinterpret_cast<const f32x4u*>(t + 4);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    r[u] = a[u];
    r[4 + u] = b[u];
  }
}

template <bool BF>
__device__ __forceinline__ void unpack8(const uint4& w, float (&r)[8]) {
  if constexpr (BF) {
    const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      r[2 * k] = __uint_as_float(ws[k] << 16);
      r[2 * k + 1] = __uint_as_float(ws[k] & 0xffff0000u);
    }
  } else {
    const f16x8 f = __builtin_bit_cast(f16x8, w);
#pragma unroll
    for (int k = 0; k < 8; ++k) r[k] = (float)f[k];
  }
}
__device__ __forceinline__ f16x8 pack8(const float (&x)[8]) {
  f16x8 f;
#pragma unroll
  for (int u = 0; u < 8; ++u) f[u] = (_Float16)x[u];
  return f;
}

// Four consecutive values as fp32 (DT 0), bf16 (1) or fp16 (2), rounded to nearest
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
template <int DT>
__device__ __forceinline__ void st4(void* p, long long i, f32x4 v) {
  if constexpr (DT == 0)
    *reinterpret_cast<f32x4*>(static_cast<float*>(p) + i) = v;
  else if constexpr (DT == 1)
    *reinterpret_cast<bf16x4*>(static_cast<__bf16*>(p) + i) =
        bf16x4{(__bf16)v[0], (__bf16)v[1], (__bf16)v[2], (__bf16)v[3]};
  else
    *reinterpret_cast<f16x4*>(static_cast<_Float16*>(p) + i) =
        f16x4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
}

// One 64-row operand block on its way from global memory to LDS: this thread's
// piece (row tid/4 of the block, d in [8p, 8p+8) and [8p+32, 8p+40)) and, for
// a rotated operand, its cosines and sines.
template <bool BF, bool ROT>
struct SwaPiece {
  uint4 lo, hi;
  float cs[ROT ? 8 : 1], sn[ROT ? 8 : 1];

  __device__ __forceinline__ void load(const void* x, long long row, int d0, int j, const SwaArgs& a) {
    constexpr int HD = SWA_D / 2;
    const bool ok = j < a.T;
    lo = hi = uint4{0, 0, 0, 0};
    if (ok) {
      const uint16_t* s = static_cast<const uint16_t*>(x) + row + d0;
      lo = *reinterpret_cast<const uint4*>(s);
      hi = *reinterpret_cast<const uint4*>(s + HD);
    }
    if constexpr (ROT) {
      const long long t = (long long)(ok ? j : 0) * HD + d0;
      ldtab8(a.cos_tab + t, cs);
      ldtab8(a.sin_tab + t, sn);
    }
  }
  __device__ __forceinline__ void rows(f16x8& x1, f16x8& x2) const {
    float r1[8], r2[8];
    unpack8<BF>(lo, r1);
    unpack8<BF>(hi, r2);
    if constexpr (ROT) {
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const float y1 = r1[u], y2 = r2[u];
        r1[u] = y1 * cs[u] - y2 * sn[u];
        r2[u] = y2 * cs[u] + y1 * sn[u];
      }
    }
    x1 = pack8(r1);
    x2 = pack8(r2);
  }
};

// Query fragments of 32 queries (B operands, contraction over d): lane (c, h)
// holds x[t][16 kb + 8 h + v], rotated when ROT.
template <bool BF, bool ROT>
__device__ __forceinline__ void load_frags(const SwaArgs& a, const void* x, long long row, int t, int h, f16x8 (&f)[4]) {
#pragma unroll
  for (int kb = 0; kb < 2; ++kb) {
    SwaPiece<BF, ROT> p;
    p.load(x, row, 16 * kb + 8 * h, t, a);
    p.rows(f[kb], f[kb + 2]);
  }
}

// Forward, NW waves of QT x 32 queries per workgroup.  Key blocks of 64 go
// through two LDS buffers: the next block's loads are issued before the
// current block's products and written to the other buffer after them, one
// barrier per block.  A wave's QT query tiles share every K and V fragment
// read.  The online softmax runs on 64 keys at a time in base 2 (the score
// scale and log2 e folded into one multiply-add); a query tile's accumulators
// are rescaled only when some query's maximum grew by more than a factor 2^8
// (until then its probabilities may exceed 1, at the same relative precision
// in fp16 and fp32).  Only blocks on the band's edges are masked.
//
// Bound by the VALU: per 32 queries x 64 keys and wave about 200 instructions
// (four per score: multiply-add, exp, sum, half a conversion and half a
// maximum; 32 exps at a quarter of the rate; the rotation and conversion of the
// staged keys) against 16 products, and by the latency between the two kinds:
// 47 % VALU-busy and 24 % MFMA-busy at a clock of 1.95 GHz (power).  B4 T16384
// H12, window 2048, bf16: 650 us, 0.63 PFLOP/s; 1853 us when every block was loaded, rotated, transposed with 2-byte
// LDS writes and used between two barriers, 128 queries to a workgroup.  A
// wave per SIMD more (four, spilling 19-35 registers) takes 905-1320 us, 32
// keys to a softmax update 742 us.
template <int NW, int QT, bool BF>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(QT == 1 ? 3 : 2))) swa_fwd_kernel(SwaArgs a) {
  using M = ModeF16;
  using frag = M::frag;
  constexpr int BQ = 32 * NW * QT, NT = 64 * NW;
  constexpr int NP = NT < 512 ? 512 / NT : 1;   // staged pieces per thread: 256 of K, 256 of V
  __shared__ __attribute__((aligned(16))) _Float16 Ks[2][SWA_TILE], Vs[2][SWA_TILE];

  const int nqb = (a.T + BQ - 1) / BQ;
  const int lb = xcd_block();
  const int bh = lb / nqb, qb = lb % nqb;
  const int b = bh / a.H, hh = bh % a.H;
  const int tid = threadIdx.x, lane = lane_id(), c = lane & 31, h = lane >> 5, w = wave_id();
  const int q0 = qb * BQ, qw = q0 + 32 * QT * w, qs = __builtin_amdgcn_readfirstlane(qw);
  const long long base_bh = (long long)b * a.sb + (long long)hh * a.sh;

  frag qf[QT][4];
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    const int tq = qw + 32 * t + c;
    load_frags<BF, true>(a, a.q, base_bh + (long long)tq * a.st, tq, h, qf[t]);
  }

  // pieces of this thread: with NW = 8 waves 0-3 stage K and waves 4-7 V
  SwaPiece<BF, true> pk[NP > 1 ? NP / 2 : 1];
  SwaPiece<BF, false> pv[NP > 1 ? NP / 2 : 1];
  const bool isk = NP > 1 || w < 4, isv = NP > 1 || (w >= 4 && w < 8);
  auto fetch = [&](int kb0) {
#pragma unroll
    for (int i = 0; i < (NP > 1 ? NP / 2 : 1); ++i) {
      const int it = (tid + NT * i) & 255, j = kb0 + (it >> 2), d0 = 8 * (it & 3);
      const long long row = base_bh + (long long)j * a.st;
      if (isk) pk[i].load(a.k, row, d0, j, a);
      if (isv) pv[i].load(a.v, row, d0, j, a);
    }
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int i = 0; i < (NP > 1 ? NP / 2 : 1); ++i) {
      const int it = (tid + NT * i) & 255, jj = it >> 2, p = it & 3;
      f16x8 x1, x2;
      if (isk) {
        pk[i].rows(x1, x2);
        st_rows(Ks[buf], jj, p, x1, x2);
      }
      if (isv) {
        pv[i].rows(x1, x2);
        st_rows(Vs[buf], jj, p, x1, x2);
      }
    }
  };

  const float sc = a.scale * 1.4426950408889634f;   // scores in base-2 units
  const float grow = 8.f / sc;
  float m[QT], l[QT];
  f32x16 O[QT][2];
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    m[t] = -1e30f;   // below every score (fp16 operands: |q'.k'| < 2^39)
    l[t] = 0.f;
    O[t][0] = O[t][1] = zero16();
  }
  const TrOff tr;
  const int kfirst = max(0, q0 - a.window) / SWA_BK * SWA_BK;
  const int kend = min(a.T, q0 + BQ);
  fetch(kfirst);
  stage(0);
  __syncthreads();
  int buf = 0;
  for (int kb0 = kfirst; kb0 < kend; kb0 += SWA_BK, buf ^= 1) {
    const bool more = kb0 + SWA_BK < kend;
    if (more) fetch(kb0 + SWA_BK);
    // (a block entirely in the future or out of the window of this wave's queries is skipped)
    if (qw < a.T && kb0 <= qw + 32 * QT - 1 && kb0 + SWA_BK - 1 >= qw - a.window) {
      f32x16 S[QT][2];
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int kb = 0; kb < 4; ++kb) {
          const frag kf = ld_row(Ks[buf], kt, kb, c, h);
#pragma unroll
          for (int t = 0; t < QT; ++t) S[t][kt] = M::mma(kf, qf[t][kb], kb == 0 ? zero16() : S[t][kt]);
        }
      // S[t][kt][r]: key kb0 + 32 kt + crow(r, h), query qw + 32 t + c
      if (!(kb0 + SWA_BK - 1 <= qw && qw + 32 * QT - 1 - kb0 <= a.window)) {
#pragma unroll
        for (int t = 0; t < QT; ++t)
#pragma unroll
          for (int kt = 0; kt < 2; ++kt)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              // visible: 0 <= tq - j <= window (a key past T is past every stored query)
              const int far = qw + 32 * t + c - (kb0 + 32 * kt + crow(r, h));
              S[t][kt][r] = (unsigned)far <= (unsigned)a.window ? S[t][kt][r] : -INFINITY;
            }
      }
      float mx[QT];
      bool up = false;
#pragma unroll
      for (int t = 0; t < QT; ++t) {
        // (maximum, not fmaxf: no canonicalising moves; a NaN score makes the query NaN either way)
        float x = S[t][0][0];
#pragma unroll
        for (int i = 1; i < 32; ++i) x = __builtin_elementwise_maximum(x, S[t][i / 16][i % 16]);
        float x0, x1;
        swap32(x, x0, x1);
        mx[t] = __builtin_elementwise_maximum(x0, x1);
        up |= mx[t] > m[t] + grow;
      }
      if (__any(up)) {
#pragma unroll
        for (int t = 0; t < QT; ++t) {
          const float mnew = fmaxf(m[t], mx[t]);
          const float al = __builtin_amdgcn_exp2f((m[t] - mnew) * sc);
          l[t] *= al;
          O[t][0] *= al;
          O[t][1] *= al;
          m[t] = mnew;
        }
      }
      frag pf[QT][2][2];
#pragma unroll
      for (int t = 0; t < QT; ++t) {
        const float mb = m[t] * sc;
        float ps = 0.f;
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            S[t][kt][r] = __builtin_amdgcn_exp2f(fmaf(S[t][kt][r], sc, -mb));   // masked -> 0
            ps += S[t][kt][r];
          }
#pragma unroll
          for (int kb = 0; kb < 2; ++kb) pf[t][kt][kb] = M::from_c(S[t][kt], kb);
        }
        l[t] += ps;
      }
      // A 32 x 32 tile that no query of it sees into is left out (its
      // probabilities are zeros, but 0 times an infinite value is not).  The
      // branches cost 3 % of the 512-query form (two copies of the products, one
      // without branches, spill 15-108 registers and take 1.5 to 2 times as long).
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        frag vf[2][2];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int I = 0; I < 2; ++I) vf[kb][I] = ld_tr(Vs[buf], tr, I, kt, kb);
#pragma unroll
        for (int t = 0; t < QT; ++t) {
          const int k0 = kb0 + 32 * kt, q32 = qs + 32 * t;
          if (k0 > q32 + 31 || k0 + 31 < q32 - a.window) continue;
#pragma unroll
          for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int I = 0; I < 2; ++I) O[t][I] = M::mma(vf[kb][I], pf[t][kt][kb], O[t][I]);
        }
      }
    }
    if (more) stage(buf ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int t = 0; t < QT; ++t) {
    const int tq = qw + 32 * t + c;
    // the two lane halves of a query hold the sums over complementary key rows
    float l0, l1;
    swap32(l[t], l0, l1);
    const float lt = l0 + l1;
    if (tq >= a.T) continue;
    const float inv = 1.f / lt;
    if (a.lse && h == 0) a.lse[(long long)bh * a.T + tq] = m[t] * a.scale + __logf(lt);   // every query sees itself: lt > 0
    const long long oo = (((long long)b * a.T + tq) * a.H + hh) * SWA_D;
#pragma unroll
    for (int I = 0; I < 2; ++I)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d0 = 32 * I + 8 * g + 4 * h;   // rows crow(4g + u, h) = d0 + u
        f32x4 v;
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = O[t][I][4 * g + u] * inv;
        st4<BF ? 1 : 2>(a.out, oo + d0, v);
      }
  }
}

// ---- backward ---------------------------------------------------------------
// With P = softmax(S), S = q'k'^T / sqrt(D) over the window, O = P v and the
// cotangent dO of O (the standard attention backward, recomputing P from the
// forward's log-normalisers):
//   dv_s = sum_t P_ts dO_t,   dP_ts = dO_t . v_s,   Delta_t = dO_t . O_t,
//   dS_ts = P_ts (dP_ts - Delta_t),
//   dk'_s = scale sum_t dS_ts q'_t,   dq'_t = scale sum_s dS_ts k'_s,
// then dq, dk = the inverse rotation of dq', dk' (the rotation is
// orthogonal).  Two kernels, each owning its outputs (no atomics, so the
// backward is bitwise reproducible): swa_bwd_kv_kernel per block of 128 keys
// loops over the queries that see them, swa_bwd_q_kernel per block of 128
// queries over their window's keys.

struct SwaBwdArgs {
  SwaArgs f;                        // the forward's arguments (out = the forward's output O)
  const void* dout;                 // (B, T, H, D) contiguous, io dtype
  const float* lse;                 // (B, H, T)
  float* delta;                     // (B, H, T) workspace: Delta_t
  void *dq, *dk, *dv;               // (B, T, H, D) contiguous, fp32 or the io dtype
};

// Delta_t = dO_t . O_t: eight lanes per (b, t, h) row of 64, 16 bytes each
template <bool BF>
__global__ void __launch_bounds__(256) swa_bwd_delta_kernel(SwaBwdArgs a) {
  const long long i = ((long long)blockIdx.x * 256 + threadIdx.x) >> 3;   // row of the contiguous arrays
  const long long n = (long long)a.f.B * a.f.T * a.f.H;
  float acc = 0.f;
  if (i < n) {
    const long long o = i * SWA_D + 8 * (threadIdx.x & 7);
    float x[8], g[8];
    unpack8<BF>(*reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(a.f.out) + o), x);
    unpack8<BF>(*reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(a.dout) + o), g);
#pragma unroll
    for (int u = 0; u < 8; ++u) acc = fmaf(x[u], g[u], acc);
  }
  acc = group_sum<8>(acc);
  if (i >= n || (threadIdx.x & 7)) return;
  const int hh = (int)(i % a.f.H);
  const long long bt = i / a.f.H;
  const int t = (int)(bt % a.f.T), b = (int)(bt / a.f.T);
  a.delta[((long long)b * a.f.H + hh) * a.f.T + t] = acc;
}

// dq, dk from the rotated gradients held as two C-layout tiles (rows d and
// d + 32, lane = token j) times scale, inverse-rotated and stored (fp32, or
// rounded to the io dtype: GD as st4's)
template <int GD>
__device__ __forceinline__ void store_unrot(const SwaArgs& f, void* dst, long long row, int j, int h,
                                            const f32x16 (&G)[2], float scale, bool rot) {
  constexpr int HD = SWA_D / 2;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    f32x4 v1, v2;
    f32x4u cs, sn;
    if (rot) {
      cs = *reinterpret_cast<const f32x4u*>(f.cos_tab + (long long)j * HD + 8 * g + 4 * h);
      sn = *reinterpret_cast<const f32x4u*>(f.sin_tab + (long long)j * HD + 8 * g + 4 * h);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {   // d = 8g + 4h + u: crow(4g + u, h)
      const float a1 = G[0][4 * g + u] * scale, a2 = G[1][4 * g + u] * scale;
      v1[u] = rot ? a1 * cs[u] + a2 * sn[u] : a1;
      v2[u] = rot ? a2 * cs[u] - a1 * sn[u] : a2;
    }
    st4<GD>(dst, row + 8 * g + 4 * h, v1);
    st4<GD>(dst, row + HD + 8 * g + 4 * h, v2);
  }
}

// dk, dv for 128 keys per workgroup (wave w: keys kw .. kw + 31), over the
// query blocks of 64 that see them, double-buffered as in the forward.  Tiles:
// S and dP as [query][key] (rows = queries, lanes = keys) so that P and dS are
// directly the B operands of dV^T = dO^T P and dK^T = Q^T dS (contraction over
// queries); one copy of the q' and dO rows serves both kinds of products
// (contiguous and transposing reads).  Bound by the VALU and the staging like
// the forward.  B4 T4001 H12, window 2048: 285-305 us (642 us single-buffered, with
// a second, transposed copy of both operands written half by half);
// swa_bwd_q_kernel 219 us (353), swa_bwd_delta_kernel 11 us (54 with one
// thread per row).  Twice the keys (queries) to a workgroup: no gain.
template <bool BF, int GD>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) swa_bwd_kv_kernel(SwaBwdArgs a) {
  using M = ModeF16;
  using frag = M::frag;
  const SwaArgs& f = a.f;
  constexpr int BKEY = 128;
  __shared__ __attribute__((aligned(16))) _Float16 Qs[2][SWA_TILE], Gs[2][SWA_TILE];   // q' and dO rows [t][d]
  __shared__ __attribute__((aligned(16))) float Ls[2][SWA_BK], Dl[2][SWA_BK];          // lse (base 2), Delta
  const int nkb = (f.T + BKEY - 1) / BKEY;
  const int lb = xcd_block();
  const int bh = lb / nkb, kblk = lb % nkb;
  const int b = bh / f.H, hh = bh % f.H;
  const int tid = threadIdx.x, lane = lane_id(), c = lane & 31, h = lane >> 5, w = wave_id();
  const int K0 = kblk * BKEY, kw = K0 + 32 * w, key = kw + c;
  const long long base_bh = (long long)b * f.sb + (long long)hh * f.sh;
  const long long gbase = ((long long)b * f.T * f.H + hh) * SWA_D, gst = (long long)f.H * SWA_D;
  const long long lrow = (long long)bh * f.T;
  constexpr float LOG2E = 1.4426950408889634f;

  // this lane's key: k' and v as B-operand fragments (k = d)
  frag kf[4], vf[4];
  load_frags<BF, true>(f, f.k, base_bh + (long long)key * f.st, key, h, kf);
  load_frags<BF, false>(f, f.v, base_bh + (long long)key * f.st, key, h, vf);

  SwaPiece<BF, true> pq;
  SwaPiece<BF, false> pg;
  float pl = 0.f;
  const int sr = tid >> 2, sp = tid & 3;
  auto fetch = [&](int qb0) {
    const int t = qb0 + sr;
    pq.load(f.q, base_bh + (long long)t * f.st, 8 * sp, t, f);
    pg.load(a.dout, gbase + t * gst, 8 * sp, t, f);
    if (tid < 2 * SWA_BK) {
      const int tt = qb0 + (tid & (SWA_BK - 1));
      pl = tt < f.T ? (tid < SWA_BK ? a.lse[lrow + tt] * LOG2E : a.delta[lrow + tt]) : 0.f;
    }
  };
  auto stage = [&](int buf) {
    f16x8 x1, x2;
    pq.rows(x1, x2);
    st_rows(Qs[buf], sr, sp, x1, x2);
    pg.rows(x1, x2);
    st_rows(Gs[buf], sr, sp, x1, x2);
    if (tid < 2 * SWA_BK) (tid < SWA_BK ? Ls[buf] : Dl[buf])[tid & (SWA_BK - 1)] = pl;
  };

  const float sc = f.scale * LOG2E;
  const TrOff tr;
  f32x16 dK[2] = {zero16(), zero16()}, dV[2] = {zero16(), zero16()};   // [d][key] tiles
  const int qend = (int)min((long long)f.T, (long long)K0 + BKEY + f.window);
  fetch(K0);
  stage(0);
  __syncthreads();
  int buf = 0;
  for (int qb0 = K0; qb0 < qend; qb0 += SWA_BK, buf ^= 1) {
    const bool more = qb0 + SWA_BK < qend;
    if (more) fetch(qb0 + SWA_BK);
#pragma unroll
    for (int qt = 0; qt < 2; ++qt) {
      const int t0 = qb0 + 32 * qt;
      // sub-tile with no query that sees any of this wave's keys
      if (kw >= f.T || t0 >= f.T || t0 + 31 < kw || t0 - (kw + 31) > f.window) continue;
      f32x16 S, dP;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        S = M::mma(ld_row(Qs[buf], qt, kb, c, h), kf[kb], kb == 0 ? zero16() : S);
        dP = M::mma(ld_row(Gs[buf], qt, kb, c, h), vf[kb], kb == 0 ? zero16() : dP);
      }
      // S[r]: query t0 + crow(r, h), key `key` (a query past T has q' = dO = 0: no contribution)
      const bool edge = !(t0 >= kw + 31 && t0 + 31 - kw <= f.window);
      f32x16 P, dS;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x4 lg = *reinterpret_cast<const f32x4*>(Ls[buf] + 32 * qt + 8 * g + 4 * h);
        const f32x4 dg = *reinterpret_cast<const f32x4*>(Dl[buf] + 32 * qt + 8 * g + 4 * h);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          P[4 * g + u] = __builtin_amdgcn_exp2f(fmaf(S[4 * g + u], sc, -lg[u]));
          dS[4 * g + u] = dP[4 * g + u] - dg[u];
        }
      }
      if (edge) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const bool ok = (unsigned)(t0 + crow(r, h) - key) <= (unsigned)f.window;
          P[r] = ok ? P[r] : 0.f;
          dS[r] = ok ? dS[r] : 0.f;
        }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) dS[r] *= P[r];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const frag pf = M::from_c(P, kb), sf = M::from_c(dS, kb);
#pragma unroll
        for (int I = 0; I < 2; ++I) {
          dV[I] = M::mma(ld_tr(Gs[buf], tr, I, qt, kb), pf, dV[I]);
          dK[I] = M::mma(ld_tr(Qs[buf], tr, I, qt, kb), sf, dK[I]);
        }
      }
    }
    if (more) stage(buf ^ 1);
    __syncthreads();
  }
  if (key >= f.T) return;
  const long long row = (((long long)b * f.T + key) * f.H + hh) * SWA_D;
  store_unrot<GD>(f, a.dk, row, key, h, dK, f.scale, true);
  store_unrot<GD>(f, a.dv, row, key, h, dV, 1.f, false);
}

// dq for 128 queries per workgroup (wave w: queries qw .. qw + 31), over the
// key blocks of 64 of their window, double-buffered.  Tiles as in the forward:
// S^T and dP^T as [key][query] (rows = keys, lanes = queries), so that dS^T is
// directly the B operand of dQ^T = K^T dS^T (contraction over keys).
template <bool BF, int GD>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) swa_bwd_q_kernel(SwaBwdArgs a) {
  using M = ModeF16;
  using frag = M::frag;
  const SwaArgs& f = a.f;
  constexpr int BQ = 128;
  __shared__ __attribute__((aligned(16))) _Float16 Ks[2][SWA_TILE], Vs[2][SWA_TILE];   // k' and v rows [key][d]
  const int nqb = (f.T + BQ - 1) / BQ;
  const int lb = xcd_block();
  const int bh = lb / nqb, qblk = lb % nqb;
  const int b = bh / f.H, hh = bh % f.H;
  const int tid = threadIdx.x, lane = lane_id(), c = lane & 31, h = lane >> 5, w = wave_id();
  const int q0 = qblk * BQ, qw = q0 + 32 * w, tq = qw + c;
  const long long base_bh = (long long)b * f.sb + (long long)hh * f.sh;
  const long long orow = (((long long)b * f.T + tq) * f.H + hh) * SWA_D;
  constexpr float LOG2E = 1.4426950408889634f;

  // this lane's query: q' and dO as B-operand fragments (k = d)
  frag qf[4], gf[4];
  load_frags<BF, true>(f, f.q, base_bh + (long long)tq * f.st, tq, h, qf);
  load_frags<BF, false>(f, a.dout, orow, tq, h, gf);
  const float lq = tq < f.T ? a.lse[(long long)bh * f.T + tq] * LOG2E : 0.f;
  const float dl = tq < f.T ? a.delta[(long long)bh * f.T + tq] : 0.f;

  SwaPiece<BF, true> pk;
  SwaPiece<BF, false> pv;
  const int sr = tid >> 2, sp = tid & 3;
  auto fetch = [&](int kb0) {
    const int j = kb0 + sr;
    const long long row = base_bh + (long long)j * f.st;
    pk.load(f.k, row, 8 * sp, j, f);
    pv.load(f.v, row, 8 * sp, j, f);
  };
  auto stage = [&](int buf) {
    f16x8 x1, x2;
    pk.rows(x1, x2);
    st_rows(Ks[buf], sr, sp, x1, x2);
    pv.rows(x1, x2);
    st_rows(Vs[buf], sr, sp, x1, x2);
  };

  const float sc = f.scale * LOG2E;
  const TrOff tr;
  f32x16 dQ[2] = {zero16(), zero16()};   // [d][query] tiles
  const int kfirst = max(0, q0 - f.window) / SWA_BK * SWA_BK;
  const int kend = min(f.T, q0 + BQ);
  fetch(kfirst);
  stage(0);
  __syncthreads();
  int buf = 0;
  for (int kb0 = kfirst; kb0 < kend; kb0 += SWA_BK, buf ^= 1) {
    const bool more = kb0 + SWA_BK < kend;
    if (more) fetch(kb0 + SWA_BK);
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      const int k0 = kb0 + 32 * kt;
      if (qw >= f.T || k0 > qw + 31 || k0 + 31 < qw - f.window) continue;
      f32x16 S, dP;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        S = M::mma(ld_row(Ks[buf], kt, kb, c, h), qf[kb], kb == 0 ? zero16() : S);
        dP = M::mma(ld_row(Vs[buf], kt, kb, c, h), gf[kb], kb == 0 ? zero16() : dP);
      }
      // S[r]: key k0 + crow(r, h), query tq (a key past T is past every stored query)
      const bool edge = !(k0 + 31 <= qw && qw + 31 - k0 <= f.window);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        S[r] = __builtin_amdgcn_exp2f(fmaf(S[r], sc, -lq));
        dP[r] -= dl;
      }
      if (edge) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const bool ok = (unsigned)(tq - (k0 + crow(r, h))) <= (unsigned)f.window;
          S[r] = ok ? S[r] : 0.f;
          dP[r] = ok ? dP[r] : 0.f;
        }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) S[r] *= dP[r];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const frag sf = M::from_c(S, kb);
#pragma unroll
        for (int I = 0; I < 2; ++I) dQ[I] = M::mma(ld_tr(Ks[buf], tr, I, kt, kb), sf, dQ[I]);
      }
    }
    if (more) stage(buf ^ 1);
    __syncthreads();
  }
  if (tq >= f.T) return;
  store_unrot<GD>(f, a.dq, orow, tq, h, dQ, f.scale, true);
}

atlas_status swa_setup(SwaArgs& a, int32_t B, int32_t T, int32_t H, int32_t D, int32_t window, const void* q,
                       const void* k, const void* v, void* out, int64_t stride_b, int64_t stride_t,
                       int64_t stride_h, int32_t io_dtype, const float* cos_tab, const float* sin_tab) {
  if (B < 1 || T < 1 || H < 1 || window < 0)
    return fail(ATLAS_ERR_INVALID_ARGUMENT, "bad sizes B=%d T=%d H=%d window=%d", B, T, H, window);
  if (D != SWA_D) return fail(ATLAS_ERR_UNSUPPORTED_SHAPE, "head dim %d not compiled (D = 64 only)", D);
  if (io_dtype != 1 && io_dtype != 2)
    return fail(ATLAS_ERR_INVALID_ARGUMENT, "io_dtype %d: bf16 (1) or fp16 (2) inputs only", io_dtype);
  if (!q || !k || !v || !out || !cos_tab || !sin_tab) return fail(ATLAS_ERR_INVALID_ARGUMENT, "NULL pointer");
  if ((stride_b | stride_t | stride_h) & 7 || stride_t < 1 || stride_h < 1)
    return fail(ATLAS_ERR_UNSUPPORTED_SHAPE, "q/k/v strides must be positive multiples of 8 elements");
  if ((long long)B * H * ((T + 127) / 128) > (1LL << 31) - 1) return fail(ATLAS_ERR_UNSUPPORTED_SHAPE, "grid too large");
  a.B = B; a.T = T; a.H = H; a.window = window; a.io_dtype = io_dtype;
  a.sb = stride_b; a.st = stride_t; a.sh = stride_h;
  a.q = q; a.k = k; a.v = v; a.out = out;
  a.cos_tab = cos_tab; a.sin_tab = sin_tab;
  a.scale = 1.f / sqrtf((float)D);
  a.lse = nullptr;
  return ATLAS_OK;
}

template <int NW, int QT>
void swa_launch_fwd_as(const SwaArgs& a, hipStream_t st) {
  const long long nqb = (a.T + 32 * NW * QT - 1) / (32 * NW * QT);
  const dim3 grid((unsigned)(a.B * a.H * nqb)), block(64 * NW);
  if (a.io_dtype == 1)
    hipLaunchKernelGGL((swa_fwd_kernel<NW, QT, true>), grid, block, 0, st, a);
  else
    hipLaunchKernelGGL((swa_fwd_kernel<NW, QT, false>), grid, block, 0, st, a);
}

// 512 queries per workgroup rotate and convert each key a quarter as often as
// 128 do, but stage up to 7 blocks that a wave of a narrow band skips (and, over
// the first `window` queries, up to 7 of the few there are), and fill the CUs
// more coarsely.  They are the faster choice where the sequence is long, the
// band wide and every CU gets at least three workgroups.  us, 128 / 512
// queries, H12: window 1024 at B12 T8192 617 / 624, B8 T12288 662 / 644, B6
// T16384 670 / 657; window 1536 at B24 T4096 714 / 779, B16 T6144 786 / 783, B12
// T8192 820 / 791, B6 T16384 893 / 816; window 2048 at B24 T4096 840 / 906, B12
// T8192 1001 / 937, B6 T16384 1096 / 984; window 4096 at B16 T6144 1384 / 1387,
// B12 T8192 1546 / 1471, B6 T16384 1848 / 1613; window 8192 at B6 T16384 2936 /
// 2626.  With 384 workgroups, B1 T16384, window 2048: 183 / 209.
atlas_status swa_launch_fwd(const SwaArgs& a, void* stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  const long long n512 = (long long)a.B * a.H * ((a.T + 511) / 512);
  if (n512 >= 3 * 256 && a.T >= 8192 && a.window >= (a.T >= 12288 ? 1024 : 1536))
    swa_launch_fwd_as<8, 2>(a, st);
  else
    swa_launch_fwd_as<4, 1>(a, st);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? ATLAS_OK : fail_hip(e, "swa launch");
}

template <bool BF, int GD>
void swa_launch_bwd(const SwaBwdArgs& a, hipStream_t st) {
  const long long rows = (long long)a.f.B * a.f.T * a.f.H;
  const unsigned n = (unsigned)((long long)a.f.B * a.f.H * ((a.f.T + 127) / 128));
  hipLaunchKernelGGL((swa_bwd_delta_kernel<BF>), dim3((unsigned)((rows + 31) / 32)), dim3(256), 0, st, a);
  hipLaunchKernelGGL((swa_bwd_kv_kernel<BF, GD>), dim3(n), dim3(256), 0, st, a);
  hipLaunchKernelGGL((swa_bwd_q_kernel<BF, GD>), dim3(n), dim3(256), 0, st, a);
}

}  // namespace
}  // namespace atlas

using namespace atlas;

extern "C" atlas_status atlas_swa_fwd(int32_t B, int32_t T, int32_t H, int32_t D, int32_t window,
                                      const void* q, const void* k, const void* v, void* out,
                                      int64_t stride_b, int64_t stride_t, int64_t stride_h, int32_t io_dtype,
                                      const float* cos_tab, const float* sin_tab, void* stream) {
  clear_error();
  SwaArgs a;
  const atlas_status r = swa_setup(a, B, T, H, D, window, q, k, v, out, stride_b, stride_t, stride_h, io_dtype,
                                   cos_tab, sin_tab);
  return r ? r : swa_launch_fwd(a, stream);
}

extern "C" atlas_status atlas_swa_fwd_lse(int32_t B, int32_t T, int32_t H, int32_t D, int32_t window,
                                          const void* q, const void* k, const void* v, void* out,
                                          int64_t stride_b, int64_t stride_t, int64_t stride_h, int32_t io_dtype,
                                          const float* cos_tab, const float* sin_tab, float* lse, void* stream) {
  clear_error();
  SwaArgs a;
  const atlas_status r = swa_setup(a, B, T, H, D, window, q, k, v, out, stride_b, stride_t, stride_h, io_dtype,
                                   cos_tab, sin_tab);
  if (r) return r;
  if (!lse) return fail(ATLAS_ERR_INVALID_ARGUMENT, "NULL lse");
  a.lse = lse;
  return swa_launch_fwd(a, stream);
}

extern "C" size_t atlas_swa_bwd_workspace_size(int32_t B, int32_t T, int32_t H) {
  if (B < 1 || T < 1 || H < 1) return 0;
  return (size_t)B * T * H * sizeof(float);
}

extern "C" atlas_status atlas_swa_bwd_as(int32_t B, int32_t T, int32_t H, int32_t D, int32_t window,
                                         const void* q, const void* k, const void* v, const void* out,
                                         const void* dout, const float* lse, int64_t stride_b, int64_t stride_t,
                                         int64_t stride_h, int32_t io_dtype, const float* cos_tab,
                                         const float* sin_tab, void* dq, void* dk, void* dv, int32_t grad_dtype,
                                         void* workspace, size_t workspace_bytes, void* stream) {
  clear_error();
  SwaBwdArgs a;
  atlas_status r = swa_setup(a.f, B, T, H, D, window, q, k, v, const_cast<void*>(out), stride_b, stride_t,
                             stride_h, io_dtype, cos_tab, sin_tab);
  if (r) return r;
  if (!dout || !lse || !dq || !dk || !dv) return fail(ATLAS_ERR_INVALID_ARGUMENT, "NULL pointer");
  if (grad_dtype != 0 && grad_dtype != io_dtype)
    return fail(ATLAS_ERR_INVALID_ARGUMENT, "grad_dtype %d: fp32 (0) or the io dtype %d", grad_dtype, io_dtype);
  const size_t need = atlas_swa_bwd_workspace_size(B, T, H);
  if (!workspace || workspace_bytes < need)
    return fail(ATLAS_ERR_WORKSPACE, "workspace %zu bytes < required %zu", workspace_bytes, need);
  auto mis = [](const void* p, int al) { return reinterpret_cast<uintptr_t>(p) % al != 0; };
  if (mis(out, 16) || mis(dout, 16) || mis(dq, 16) || mis(dk, 16) || mis(dv, 16) || mis(workspace, 4) ||
      mis(lse, 4))
    return fail(ATLAS_ERR_INVALID_ARGUMENT, "out, dout, dq, dk, dv must be 16-byte aligned");
  a.dout = dout;
  a.lse = lse;
  a.delta = static_cast<float*>(workspace);
  a.dq = dq;
  a.dk = dk;
  a.dv = dv;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (grad_dtype == 0) io_dtype == 1 ? swa_launch_bwd<true, 0>(a, st) : swa_launch_bwd<false, 0>(a, st);
  else io_dtype == 1 ? swa_launch_bwd<true, 1>(a, st) : swa_launch_bwd<false, 2>(a, st);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? ATLAS_OK : fail_hip(e, "swa backward launch");
}

extern "C" atlas_status atlas_swa_bwd(int32_t B, int32_t T, int32_t H, int32_t D, int32_t window,
                                      const void* q, const void* k, const void* v, const void* out,
                                      const void* dout, const float* lse, int64_t stride_b, int64_t stride_t,
                                      int64_t stride_h, int32_t io_dtype, const float* cos_tab,
                                      const float* sin_tab, float* dq, float* dk, float* dv, void* workspace,
                                      size_t workspace_bytes, void* stream) {
  return atlas_swa_bwd_as(B, T, H, D, window, q, k, v, out, dout, lse, stride_b, stride_t, stride_h, io_dtype,
                          cos_tab, sin_tab, dq, dk, dv, 0, workspace, workspace_bytes, stream);
}
