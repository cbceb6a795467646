// atlas_pe_batched: Polar-Express on a batch of small independent matrices,
// one wavefront per matrix (atlas_jax/memory_layer.py:43-71,
// kernels/triton_pe.py:26-69; with ATLAS_PE_NORM_NO_EPS the normalisation of
// optim.py:69-83).
//
// A (d1 x d2) input is processed in its wide orientation: if d1 > d2 the
// kernel works on X^T (PE(X)^T = PE(X^T)), so the Gram is always the smaller
// (D x D) one.  The matrix is zero-padded to the compiled (D, E) tile shape;
// zero rows/columns stay zero through every Newton-Schulz step, so padding
// does not change the result.  Wide sides of 129..256 are split over a pair
// of waves (128 columns each, the Gram summed through LDS).  Short sides of
// 65..128 run on a workgroup of six or eight waves per matrix (pe_wg_kernel,
// fp32 accuracy).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "atlas_pe.hpp"
#include "atlas_pe_split.hpp"
#include "atlas_scan.h"
#include "atlas_status.hpp"

namespace atlas {
namespace {

// ---- one wave's matrix between global memory and C-layout tiles --------------
// A rows x cols matrix (wide orientation, rows <= D, cols <= E) is addressed
// through a wave-uniform pointer and 32-bit offsets, and every load is issued
// unconditionally (out-of-range elements read element 0 and are replaced), so
// that all loads of a matrix are in flight together; a load under a per-element
// branch waits for the one before it (65 536 fp32 matrices of 56 x 56, 3 steps:
// 1197 us with branches, 767 without; 3023 on fp32 operands, with branches).  Polar-Express commutes with a permutation
// of the columns, so a wide matrix whose rows allow it gives lane c of the TJ
// column tiles TJ consecutive columns (one load per row); a tall one (stored
// transposed) has four consecutive rows of a column per lane by the C layout.
enum PEPath { PE_ELEM = 0, PE_TALL4 = 1, PE_WIDEV = 2 };

template <int DT>
__device__ __forceinline__ float pe_ld1(const void* x, int o) {
  if constexpr (DT == 0) return static_cast<const float*>(x)[o];
  else if constexpr (DT == 1) return __uint_as_float((uint32_t)static_cast<const uint16_t*>(x)[o] << 16);
  else return (float)static_cast<const _Float16*>(x)[o];
}
template <int DT>
__device__ __forceinline__ void pe_st1(void* y, int o, float v) {
  if constexpr (DT == 0) static_cast<float*>(y)[o] = v;
  else if constexpr (DT == 1) static_cast<__bf16*>(y)[o] = (__bf16)v;
  else static_cast<_Float16*>(y)[o] = (_Float16)v;
}
template <int N>
struct PEVec { typedef float type __attribute__((ext_vector_type(N))); };

// fp32 only for the two vector paths
template <int D, int E, int DT, int PATH>
__device__ __forceinline__ void pe_load(f32x16 (&X)[D / 32][E / 32], const void* x, int rows, int cols, bool tall) {
  constexpr int TI = D / 32, TJ = E / 32;
  const int c = lane_id() & 31, h = lane_id() >> 5;
  const int si = tall ? 1 : cols, sj = tall ? rows : 1;   // element strides of (i, j)
  if constexpr (PATH == PE_TALL4) {
#pragma unroll
    for (int I = 0; I < TI; ++I)
#pragma unroll
      for (int J = 0; J < TJ; ++J)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int i = 32 * I + 8 * q + 4 * h, j = 32 * J + c;
          const bool ok = i < rows && j < cols;
          const f32x4 v = *reinterpret_cast<const f32x4*>(static_cast<const float*>(x) + (ok ? j * rows + i : 0));
#pragma unroll
          for (int u = 0; u < 4; ++u) X[I][J][4 * q + u] = ok ? v[u] : 0.f;
        }
  } else if constexpr (PATH == PE_WIDEV) {
    typedef typename PEVec<TJ>::type vec;
#pragma unroll
    for (int I = 0; I < TI; ++I)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = 32 * I + crow(r, h), j = TJ * c;
        const bool ok = i < rows && j < cols;
        const vec v = *reinterpret_cast<const vec*>(static_cast<const float*>(x) + (ok ? i * cols + j : 0));
#pragma unroll
        for (int J = 0; J < TJ; ++J) X[I][J][r] = ok ? v[J] : 0.f;
      }
  } else {
#pragma unroll
    for (int I = 0; I < TI; ++I)
#pragma unroll
      for (int J = 0; J < TJ; ++J)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int i = 32 * I + crow(r, h), j = 32 * J + c;
          const bool ok = i < rows && j < cols;
          const float v = pe_ld1<DT>(x, ok ? i * si + j * sj : 0);
          X[I][J][r] = ok ? v : 0.f;
        }
  }
}
// X to y, laid out as pe_load reads it
template <int D, int E, int DT, int PATH>
__device__ __forceinline__ void pe_store(const f32x16 (&X)[D / 32][E / 32], void* y, int rows, int cols, bool tall) {
  constexpr int TI = D / 32, TJ = E / 32;
  // (opaque: the offsets are formed again rather than kept, spilled, across
  // Polar-Express)
  int lane = lane_id();
  asm volatile("" : "+v"(lane));
  const int c = lane & 31, h = lane >> 5;
  const int si = tall ? 1 : cols, sj = tall ? rows : 1;
#pragma unroll
  for (int I = 0; I < TI; ++I) {
    if constexpr (PATH == PE_TALL4) {
#pragma unroll
      for (int J = 0; J < TJ; ++J)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int i = 32 * I + 8 * q + 4 * h, j = 32 * J + c;
          if (i < rows && j < cols)
            *reinterpret_cast<f32x4*>(static_cast<float*>(y) + j * rows + i) =
                f32x4{X[I][J][4 * q], X[I][J][4 * q + 1], X[I][J][4 * q + 2], X[I][J][4 * q + 3]};
        }
    } else if constexpr (PATH == PE_WIDEV) {
      typedef typename PEVec<TJ>::type vec;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = 32 * I + crow(r, h), j = TJ * c;
        vec v;
#pragma unroll
        for (int J = 0; J < TJ; ++J) v[J] = X[I][J][r];
        if (i < rows && j < cols) *reinterpret_cast<vec*>(static_cast<float*>(y) + i * cols + j) = v;
      }
    } else {
#pragma unroll
      for (int J = 0; J < TJ; ++J)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int i = 32 * I + crow(r, h), j = 32 * J + c;
          if (i < rows && j < cols) pe_st1<DT>(y, i * si + j * sj, X[I][J][r]);
        }
    }
  }
}
// The widest path that a batch allows: fp32, every vector of every matrix
// aligned (X and Y to 16 bytes; a wide matrix's rows and size, a tall one's
// stored rows, a multiple of the vector).
inline int pe_path(int d1, int d2, int TJ, int dtype, const void* X, const void* Y) {
  if (dtype != 0 || ((reinterpret_cast<uintptr_t>(X) | reinterpret_cast<uintptr_t>(Y)) & 15)) return PE_ELEM;
  if (d1 > d2) return d2 % 4 == 0 ? PE_TALL4 : PE_ELEM;
  return TJ > 1 && d2 % TJ == 0 ? PE_WIDEV : PE_ELEM;
}

// fp32 compute mode, wide side <= 128: one wave per matrix on
// polar_express_wave_split.
template <int D, int E, int DT, int PATH>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
pe_split_kernel(long long n, int d1, int d2, int ns, float eps, const void* X, void* Y) {
  constexpr int TI = D / 32, TJ = E / 32;
  __shared__ __attribute__((aligned(16))) _Float16 xs_all[4 * PESplit<D, E>::ELEMS];
  const int w = __builtin_amdgcn_readfirstlane(wave_id());
  const long long mat = (long long)blockIdx.x * 4 + w;
  if (mat >= n) return;   // no workgroup barrier below
  const bool tall = d1 > d2;
  const int rows = tall ? d2 : d1, cols = tall ? d1 : d2;   // wide orientation
  const long long base = mat * (long long)d1 * d2 * (DT == 0 ? 4 : 2);
  f32x16 Xr[TI][TJ];
  pe_load<D, E, DT, PATH>(Xr, static_cast<const char*>(X) + base, rows, cols, tall);
  polar_express_wave_split<D, E>(Xr, ns, eps, xs_all + w * PESplit<D, E>::ELEMS);
  pe_store<D, E, DT, PATH>(Xr, static_cast<char*>(Y) + base, rows, cols, tall);
}

// fp16 operands, wide side <= 128: the scan's own Polar-Express
// (polar_express_wave_t: Gram operands transposed through a per-wave LDS
// staging area, iterate carried scaled), one wave per matrix.  With `vec` set
// (tall input whose short side is D, buffers aligned) the transposed layout
// is read and written as runs of 4 along the short side, which is what the
// C layout gives each lane; otherwise element by element.  FAST >= 0: fp32
// input and output with vec = FAST fixed at compile time (the backward's
// recompute); a kernel that keeps every dtype and load path spills.
template <int D, int E, int FAST>
__device__ __forceinline__ void pe_wave_t_one(long long mat, long long n, int d1, int d2, int ns, float eps,
                                              const void* X, void* Y, int dtype_, int vec_, _Float16* xs) {
  const int dtype = FAST >= 0 ? 0 : dtype_, vec = FAST >= 0 ? FAST : vec_;
  using PT = PEWaveT<D, E>;
  constexpr int TI = D / 32, TJ = E / 32;
  if (mat >= n) return;   // no workgroup barrier below
  const int c = lane_id() & 31, h = lane_id() >> 5;
  const bool tall = d1 > d2;
  const int rows = tall ? d2 : d1, cols = tall ? d1 : d2;
  const long long base = mat * (long long)d1 * d2;
  f32x16 Xr[TI][TJ];
  // vec 2 (wide input of exactly D x 128 floats, aligned): tile J's lane c
  // holds column 4c + J (Polar-Express is invariant under a common
  // permutation of the columns), one 16-byte load per row for four tiles
  const bool wide4 = TJ == 4 && vec == 2;
  if (wide4) {
#pragma unroll
    for (int I = 0; I < TI; ++I)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(static_cast<const float*>(X) + base +
                                                         (long long)(32 * I + crow(r, h)) * E + 4 * c);
#pragma unroll
        for (int J = 0; J < TJ; ++J) Xr[I][J][r] = v[J & 3];
      }
  }
#pragma unroll
  for (int I = 0; I < TI && !wide4; ++I)
#pragma unroll
    for (int J = 0; J < TJ; ++J) {
      const int j = 32 * J + c;
      if (vec == 1) {   // rows crow(4q + u, h) = 8q + 4h + u of column j: X^T[j][..] contiguous
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x4 v = j < cols ? load4_any(X, base + (long long)j * d2 + 32 * I + 8 * q + 4 * h, dtype)
                                   : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int u = 0; u < 4; ++u) Xr[I][J][4 * q + u] = v[u];
        }
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int i = 32 * I + crow(r, h);
          float v = 0.f;
          if (i < rows && j < cols) v = load_any(X, base + (tall ? (long long)j * d2 + i : (long long)i * d2 + j), dtype);
          Xr[I][J][r] = v;
        }
      }
    }
  const float ps = polar_express_wave_t<D, E>(Xr, ns, eps, xs);
  if (wide4) {
    // the lane's offset through opaque(): formed here rather than 32 row
    // addresses kept (spilled) across Polar-Express
    float* yl = static_cast<float*>(Y) + base + PT::opaque(4 * h * E + 4 * c);
#pragma unroll
    for (int I = 0; I < TI; ++I)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        *reinterpret_cast<f32x4*>(yl + (32 * I + 8 * (r / 4) + r % 4) * E) =
            f32x4{Xr[I][0][r] * ps, Xr[I][1 & (TJ - 1)][r] * ps, Xr[I][2 & (TJ - 1)][r] * ps,
                  Xr[I][3 & (TJ - 1)][r] * ps};
    return;
  }
#pragma unroll
  for (int I = 0; I < TI; ++I)
#pragma unroll
    for (int J = 0; J < TJ; ++J) {
      const int j = 32 * J + c;
      if (vec == 1) {
        if (j < cols) {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            store4_any(Y, base + (long long)j * d2 + 32 * I + 8 * q + 4 * h, dtype,
                       f32x4{Xr[I][J][4 * q] * ps, Xr[I][J][4 * q + 1] * ps, Xr[I][J][4 * q + 2] * ps,
                             Xr[I][J][4 * q + 3] * ps});
        }
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int i = 32 * I + crow(r, h);
          if (i < rows && j < cols)
            store_any(Y, base + (tall ? (long long)j * d2 + i : (long long)i * d2 + j), dtype, Xr[I][J][r] * ps);
        }
      }
    }
}

template <int D, int E, int FAST = -1>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
pe_wave_t_kernel(long long n, int d1, int d2, int ns, float eps, const void* X, void* Y, int dtype_, int vec_) {
  __shared__ __attribute__((aligned(16))) _Float16 xs_all[4 * PEWaveT<D, E>::ELEMS];
  pe_wave_t_one<D, E, FAST>((long long)blockIdx.x * 4 + wave_id(), n, d1, d2, ns, eps, X, Y, dtype_, vec_,
                            xs_all + wave_id() * PEWaveT<D, E>::ELEMS);
}

// The backward's recompute of both memories in one launch (fp32 in and out):
// blocks [0, ceil(n / 4)) take the n wide D x E matrices (Xa -> Ya, load path
// FA), the rest the n tall E x D ones (Xb -> Yb, load path FB), so that the
// second batch starts on every CU the first one frees.
template <int D, int E, int FA, int FB>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))
pe_wave_t_both_kernel(long long n, int ns, float eps, const float* Xa, float* Ya, const float* Xb, float* Yb) {
  __shared__ __attribute__((aligned(16))) _Float16 xs_all[4 * PEWaveT<D, E>::ELEMS];
  _Float16* xs = xs_all + wave_id() * PEWaveT<D, E>::ELEMS;
  const long long ba = (n + 3) / 4;
  if (blockIdx.x < ba)
    pe_wave_t_one<D, E, FA>((long long)blockIdx.x * 4 + wave_id(), n, D, E, ns, eps, Xa, Ya, 0, FA, xs);
  else
    pe_wave_t_one<D, E, FB>((long long)(blockIdx.x - ba) * 4 + wave_id(), n, E, D, ns, eps, Xb, Yb, 0, FB, xs);
}

// Two waves per matrix: wave 2p+half holds columns [128 half, 128 half + 128)
// of matrix 2 blockIdx + p (wide orientation).  Workgroups past the last
// matrix still run every step on zeros so that all barriers are reached.
template <class M, int D>
__global__ void __launch_bounds__(256)
pe_pair_kernel(long long n, int d1, int d2, int ns, float eps, const void* X, void* Y, int dtype) {
  constexpr int EH = 128, TI = D / 32, TJ = EH / 32;
  __shared__ __attribute__((aligned(16))) typename M::elem scr_all[4 * Scr<M>::template elems<D>()];
  __shared__ float xch[4][D * D];
  const int wv = wave_id(), pair = wv >> 1, half = wv & 1;
  const long long mat = (long long)blockIdx.x * 2 + pair;
  const bool live = mat < n;
  typename M::elem* scr = scr_all + wv * Scr<M>::template elems<D>();
  const int c = lane_id() & 31, h = lane_id() >> 5;
  const bool tall = d1 > d2;
  const int rows = tall ? d2 : d1, cols = tall ? d1 : d2;
  const long long base = (live ? mat : 0) * (long long)d1 * d2;
  f32x16 Xr[TI][TJ];
#pragma unroll
  for (int I = 0; I < TI; ++I)
#pragma unroll
    for (int J = 0; J < TJ; ++J)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = 32 * I + crow(r, h), j = EH * half + 32 * J + c;
        float v = 0.f;
        if (live && i < rows && j < cols)
          v = load_any(X, base + (tall ? (long long)j * d2 + i : (long long)i * d2 + j), dtype);
        Xr[I][J][r] = v;
      }
  // fp16: Gram operands transposed on the matrix cores (no staging area),
  // result = X * ps
  const float ps = polar_express_pair<M, D, EH>(Xr, ns, eps, sizeof(typename M::elem) == 2 ? nullptr : scr,
                                                xch[wv], xch[wv ^ 1], half);
  if (!live) return;
#pragma unroll
  for (int I = 0; I < TI; ++I)
#pragma unroll
    for (int J = 0; J < TJ; ++J)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = 32 * I + crow(r, h), j = EH * half + 32 * J + c;
        if (i < rows && j < cols)
          store_any(Y, base + (tall ? (long long)j * d2 + i : (long long)i * d2 + j), dtype, Xr[I][J][r] * ps);
      }
}

// One workgroup of NW waves per matrix whose short side is 65..128 (TI = 3 or
// 4 row tiles of 32; long side <= 32 NW <= 256), in fp32 accuracy in either
// compute mode: operands as two fp16 numbers (atlas_pe_split.hpp).  The iterate
// X (wide orientation, zero-padded to 32 TI rows and whole 32-column blocks) is
// held in registers as fp32 C-layout tiles, column block J by wave J.  Per
// Newton-Schulz step, with barriers between:
//   X's blocks staged in LDS as split rows, all at once;
//   Gram: each wave forms its upper tiles of G = X X^T over all blocks;
//   G shared as operand fragments (every lane writes the 16 bytes that the
//         same lane of the other waves reads; a lower tile is its mirror
//         transposed through its own slot), laid over the staged blocks;
//   B     = b G + c G^2, the same tiles, shared the same way;
//   X     <- a X + B X for the wave's column block.
// Every sum has a fixed order (bitwise reproducible).  2 048 matrices of 96 x
// 192, 5 steps: 317 us a call (369 us with one scale for all columns, at three
// waves per SIMD instead of four; 1019 us on fp32 operands, staged a block at a
// time with all nine Gram tiles).
template <int TI, int NW>
struct PEWg {
  static constexpr int DP = 32 * TI;
  static constexpr int NT = TI * (TI + 1) / 2;        // upper tiles
  static constexpr int NQ = (NT + NW - 1) / NW;       // of a wave, at most
  static constexpr int BLK = PESplit<DP, 32>::ELEMS;  // halves of a staged block
  static constexpr int FR = TI * TI * 2 * 2 * 512;    // halves of G or B as fragments
  static size_t lds_bytes(int nj) { return (size_t)std::max(nj * BLK, 2 * FR) * 2 + NW * sizeof(float); }
  // (I, I2 >= I) of upper tile t, row by row
  __device__ __forceinline__ static void tile(int t, int& I, int& I2) {
    I = 0;
    int n = TI;
    while (t >= n) {
      t -= n;
      --n;
      ++I;
    }
    I2 = I + t;
  }
};

template <int TI, int NW>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW == 6 ? 3 : 2)))
pe_wg_kernel(long long n, int d1, int d2, int ns, float eps, const void* X, void* Y, int dtype, int vec) {
  using W = PEWg<TI, NW>;
  using P = PESplit<W::DP, 32>;
  using T32 = PESplit<32, 32>;
  constexpr int NQ = W::NQ;
  constexpr float XS = 4096.f, AS = 2048.f, BS = 4096.f;   // |X| <= 2, |G| <= 4, |B| <= 8 as fp16 operands
  extern __shared__ __attribute__((aligned(16))) _Float16 wlds[];
  const int w = __builtin_amdgcn_readfirstlane(wave_id()), lane = lane_id();
  const long long mat = blockIdx.x;
  const bool tall = d1 > d2;
  const int rows = tall ? d2 : d1, cols = tall ? d1 : d2;   // wide orientation
  const int NJ = (cols + 31) / 32;                          // <= NW
  const bool own = w < NJ;
  float* red = reinterpret_cast<float*>(wlds + max(NJ * W::BLK, 2 * W::FR));
  _Float16 *fG = wlds, *fB = wlds + W::FR;
  const long long base = mat * (long long)d1 * d2 * (dtype == 0 ? 4 : 2);
  const char* Xm = static_cast<const char*>(X) + base;
  char* Ym = static_cast<char*>(Y) + base;

  auto slot = [&](_Float16* m, int K, int I, int kb) { return m + ((K * TI + I) * 2 + kb) * 1024; };
  auto put_frag = [&](_Float16* p, const SFrag& f) {
    *reinterpret_cast<f16x8*>(p + lane * 8) = f.hi;
    *reinterpret_cast<f16x8*>(p + 512 + lane * 8) = f.lo;
  };
  auto get_frag = [&](const _Float16* p) {
    return SFrag{*reinterpret_cast<const f16x8*>(p + lane * 8), *reinterpret_cast<const f16x8*>(p + 512 + lane * 8)};
  };
  static_assert(T32::ELEMS == 2 * 1024, "a tile's transposing scratch is its slot");
  auto share = [&](_Float16* m, const f32x16& t, int I, int I2, float s) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) put_frag(slot(m, I, I2, kb), split_c(t, kb, s));
    if (I != I2) {
      const int l = opaque_lane();
      _Float16* sc = slot(m, I2, I, 0);
      T32::put_tile(t, s, sc, l);
      const SFrag f0 = T32::get_tile(sc, 0, l), f1 = T32::get_tile(sc, 1, l);
      put_frag(slot(m, I2, I, 0), f0);
      put_frag(slot(m, I2, I, 1), f1);
    }
  };

  f32x16 Xr[TI];
  auto each = [&](auto&& f) {   // f(I, r, offset or -1) over this lane's elements
    const int l = opaque_lane(), c = l & 31, h = l >> 5, j = 32 * w + c;
    const int si = tall ? 1 : cols, sj = tall ? rows : 1;
#pragma unroll
    for (int I = 0; I < TI; ++I)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = 32 * I + crow(r, h);
        f(I, r, i < rows && j < cols ? i * si + j * sj : -1);
      }
  };
  if (vec) {   // tall fp32, rows % 4 == 0, aligned: four consecutive rows of a column
    const int c = lane & 31, h = lane >> 5, j = 32 * w + c;
#pragma unroll
    for (int I = 0; I < TI; ++I)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int i = 32 * I + 8 * q + 4 * h;
        const bool ok = i < rows && j < cols;
        const f32x4 v = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(Xm) + (ok ? j * rows + i : 0));
#pragma unroll
        for (int u = 0; u < 4; ++u) Xr[I][4 * q + u] = ok ? v[u] : 0.f;
      }
  } else if (dtype == 0) {
    each([&](int I, int r, int o) { const float v = pe_ld1<0>(Xm, max(o, 0)); Xr[I][r] = o >= 0 ? v : 0.f; });
  } else if (dtype == 1) {
    each([&](int I, int r, int o) { const float v = pe_ld1<1>(Xm, max(o, 0)); Xr[I][r] = o >= 0 ? v : 0.f; });
  } else {
    each([&](int I, int r, int o) { const float v = pe_ld1<2>(Xm, max(o, 0)); Xr[I][r] = o >= 0 ? v : 0.f; });
  }
  {
    float ss = 0.f;
#pragma unroll
    for (int I = 0; I < TI; ++I)
#pragma unroll
      for (int r = 0; r < 16; ++r) ss += Xr[I][r] * Xr[I][r];
    ss = wave_sum(ss);
    if (lane == 0) red[w] = ss;
    __syncthreads();
    float tot = 0.f;
#pragma unroll
    for (int i = 0; i < NW; ++i) tot += red[i];
    const float inv = 1.f / (sqrtf(tot + eps) * 1.01f + 1e-6f);
#pragma unroll
    for (int I = 0; I < TI; ++I) Xr[I] *= inv;
  }
  for (int st = 0; st < ns; ++st) {
    const float pa = kPE[st][0], pb = kPE[st][1], pc = kPE[st][2];
    if (own) {
      f32x16 b[TI][1];
#pragma unroll
      for (int I = 0; I < TI; ++I) b[I][0] = Xr[I];
      P::put_block(b, 0, XS, wlds + w * W::BLK, opaque_lane());
    }
    __syncthreads();
    f32x16 G[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      G[q] = zero16();
      if (w + NW * q < W::NT) {
        int I, I2;
        W::tile(w + NW * q, I, I2);
        const int l = opaque_lane();
#pragma unroll 2
        for (int J = 0; J < NJ; ++J)
#pragma unroll
          for (int kb = 0; kb < 2; ++kb)
            G[q] = mma_split(P::get(wlds + J * W::BLK, I, kb, l), P::get(wlds + J * W::BLK, I2, kb, l), G[q]);
      }
    }
    __syncthreads();   // the staged blocks have been read
#pragma unroll
    for (int q = 0; q < NQ; ++q)
      if (w + NW * q < W::NT) {
        int I, I2;
        W::tile(w + NW * q, I, I2);
        G[q] *= 1.f / (XS * XS);
        share(fG, G[q], I, I2, AS);
      }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NQ; ++q)
      if (w + NW * q < W::NT) {
        int I, I2;
        W::tile(w + NW * q, I, I2);
        f32x16 a2 = zero16();
#pragma unroll
        for (int K = 0; K < TI; ++K)
#pragma unroll
          for (int kb = 0; kb < 2; ++kb)
            a2 = mma_split(get_frag(slot(fG, K, I, kb)), get_frag(slot(fG, K, I2, kb)), a2);
        share(fB, pb * G[q] + (pc / (AS * AS)) * a2, I, I2, BS);
      }
    __syncthreads();
    if (own) {
      f32x16 acc[TI];
#pragma unroll
      for (int I = 0; I < TI; ++I) acc[I] = zero16();
      // the column's largest entry to [2^12, 2^13) (columns far below the others keep their bits)
      const int ke = column_exponent<TI>(Xr, 13);
      const float sc = __builtin_amdgcn_ldexpf(1.f, ke);
#pragma unroll
      for (int K = 0; K < TI; ++K)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          const SFrag x = split_c(Xr[K], kb, sc);
#pragma unroll
          for (int I = 0; I < TI; ++I) acc[I] = mma_split(get_frag(slot(fB, K, I, kb)), x, acc[I]);
          __builtin_amdgcn_sched_barrier(0);   // keeps later fragments' loads from being hoisted (registers)
        }
#pragma unroll
      for (int I = 0; I < TI; ++I) Xr[I] = pa * Xr[I] + acc[I] * __builtin_amdgcn_ldexpf(1.f / BS, -ke);
    }
    __syncthreads();   // B has been read: the blocks may be staged over it
  }
  if (!own) return;
  if (vec) {
    const int l = opaque_lane(), c = l & 31, h = l >> 5, j = 32 * w + c;
#pragma unroll
    for (int I = 0; I < TI; ++I)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int i = 32 * I + 8 * q + 4 * h;
        if (i < rows && j < cols)
          *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(Ym) + j * rows + i) =
              f32x4{Xr[I][4 * q], Xr[I][4 * q + 1], Xr[I][4 * q + 2], Xr[I][4 * q + 3]};
      }
  } else if (dtype == 0) {
    each([&](int I, int r, int o) { if (o >= 0) pe_st1<0>(Ym, o, Xr[I][r]); });
  } else if (dtype == 1) {
    each([&](int I, int r, int o) { if (o >= 0) pe_st1<1>(Ym, o, Xr[I][r]); });
  } else {
    each([&](int I, int r, int o) { if (o >= 0) pe_st1<2>(Ym, o, Xr[I][r]); });
  }
}

template <int TI, int NW>
atlas_status launch_wg(long long n, int d1, int d2, int ns, float eps, const void* X, void* Y, int dtype,
                       hipStream_t st) {
  using W = PEWg<TI, NW>;
  if (n > 0x7fffffffLL) return fail(ATLAS_ERR_UNSUPPORTED_SHAPE, "n too large for the workgroup kernel");
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(pe_wg_kernel<TI, NW>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)W::lds_bytes(NW));
  if (attr != hipSuccess) return fail_hip(attr, "pe_wg attribute");
  const int vec = pe_path(d1, d2, 1, dtype, X, Y) == PE_TALL4, nj = (std::max(d1, d2) + 31) / 32;
  hipLaunchKernelGGL((pe_wg_kernel<TI, NW>), dim3((unsigned)n), dim3(64 * NW), W::lds_bytes(nj), st, n, d1, d2, ns, eps,
                     X, Y, dtype, vec);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? ATLAS_OK : fail_hip(e, "pe_batched launch");
}

template <class M, int D>
atlas_status launch_pair(long long n, int d1, int d2, int ns, float eps, const void* X, void* Y, int dtype,
                         hipStream_t st) {
  const long long blocks = (n + 1) / 2;
  hipLaunchKernelGGL((pe_pair_kernel<M, D>), dim3((unsigned)blocks), dim3(256), 0, st, n, d1, d2, ns, eps, X, Y,
                     dtype);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? ATLAS_OK : fail_hip(e, "pe_batched launch");
}

template <int D, int E>
atlas_status launch_split(long long n, int d1, int d2, int ns, float eps, const void* X, void* Y, int dtype,
                          hipStream_t st) {
  const long long blocks = (n + 3) / 4;
  const int path = pe_path(d1, d2, E / 32, dtype, X, Y);
  using K = void (*)(long long, int, int, int, float, const void*, void*);
  auto go = [&](K k) { hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(256), 0, st, n, d1, d2, ns, eps, X, Y); };
  if (dtype == 1) go(pe_split_kernel<D, E, 1, PE_ELEM>);
  else if (dtype == 2) go(pe_split_kernel<D, E, 2, PE_ELEM>);
  else if (path == PE_TALL4) go(pe_split_kernel<D, E, 0, PE_TALL4>);
  else if (path == PE_WIDEV) go(pe_split_kernel<D, E, 0, (E > 32) ? PE_WIDEV : PE_ELEM>);
  else go(pe_split_kernel<D, E, 0, PE_ELEM>);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? ATLAS_OK : fail_hip(e, "pe_batched launch");
}

template <int D, int E>
atlas_status launch_t(long long n, int d1, int d2, int ns, float eps, const void* X, void* Y, int dtype,
                      hipStream_t st) {
  const long long blocks = (n + 3) / 4;
  const size_t align = dtype == 0 ? 16 : 8;
  const bool al = reinterpret_cast<uintptr_t>(X) % align == 0 && reinterpret_cast<uintptr_t>(Y) % align == 0;
  const int vec = !al ? 0 : (d1 > d2 && d2 == D) ? 1 : (d1 == D && d2 == E && E == 128 && dtype == 0) ? 2 : 0;
  if (dtype == 0 && vec == 1)
    hipLaunchKernelGGL((pe_wave_t_kernel<D, E, 1>), dim3((unsigned)blocks), dim3(256), 0, st, n, d1, d2, ns, eps, X, Y,
                       dtype, vec);
  else if (dtype == 0 && vec == 2)
    hipLaunchKernelGGL((pe_wave_t_kernel<D, E, 2>), dim3((unsigned)blocks), dim3(256), 0, st, n, d1, d2, ns, eps, X, Y,
                       dtype, vec);
  else
    hipLaunchKernelGGL((pe_wave_t_kernel<D, E>), dim3((unsigned)blocks), dim3(256), 0, st, n, d1, d2, ns, eps, X, Y,
                       dtype, vec);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? ATLAS_OK : fail_hip(e, "pe_batched launch");
}

template <class M>
atlas_status dispatch(long long n, int d1, int d2, int ns, float eps, const void* X, void* Y, int dtype,
                      hipStream_t st) {
  const int rows = d1 < d2 ? d1 : d2, cols = d1 < d2 ? d2 : d1;
  // six waves (two workgroups on a CU) where the columns fit them
  if (rows > 96) return launch_wg<4, 8>(n, d1, d2, ns, eps, X, Y, dtype, st);
  if (rows > 64) return cols <= 192 ? launch_wg<3, 6>(n, d1, d2, ns, eps, X, Y, dtype, st)
                                    : launch_wg<3, 8>(n, d1, d2, ns, eps, X, Y, dtype, st);
  const int D = rows <= 32 ? 32 : 64;
  if (cols > 128) return D == 32 ? launch_pair<M, 32>(n, d1, d2, ns, eps, X, Y, dtype, st)
                                 : launch_pair<M, 64>(n, d1, d2, ns, eps, X, Y, dtype, st);
  const int E = cols <= 32 ? 32 : (cols <= 64 ? 64 : 128);
  if constexpr (sizeof(typename M::elem) == 2) {
    if (D == 32 && E == 32) return launch_t<32, 32>(n, d1, d2, ns, eps, X, Y, dtype, st);
    if (D == 32 && E == 64) return launch_t<32, 64>(n, d1, d2, ns, eps, X, Y, dtype, st);
    if (D == 32 && E == 128) return launch_t<32, 128>(n, d1, d2, ns, eps, X, Y, dtype, st);
    if (D == 64 && E == 64) return launch_t<64, 64>(n, d1, d2, ns, eps, X, Y, dtype, st);
    return launch_t<64, 128>(n, d1, d2, ns, eps, X, Y, dtype, st);
  }
  if (D == 32 && E == 32) return launch_split<32, 32>(n, d1, d2, ns, eps, X, Y, dtype, st);
  if (D == 32 && E == 64) return launch_split<32, 64>(n, d1, d2, ns, eps, X, Y, dtype, st);
  if (D == 32 && E == 128) return launch_split<32, 128>(n, d1, d2, ns, eps, X, Y, dtype, st);
  if (D == 64 && E == 64) return launch_split<64, 64>(n, d1, d2, ns, eps, X, Y, dtype, st);
  return launch_split<64, 128>(n, d1, d2, ns, eps, X, Y, dtype, st);
}

}  // namespace

// fp16 Polar-Express of the backward's recompute for both memories of a
// chunk: n D x E matrices (Xa -> Ya) and n E x D ones (Xb -> Yb), fp32, in one
// launch when the one-wave kernel covers the shape and the buffers are
// 16-byte aligned; otherwise through atlas_pe_batched, one call per batch.
atlas_status pe_recompute_both(long long n, int D, int E, int ns, const float* Xa, float* Ya, const float* Xb,
                               float* Yb, hipStream_t st) {
  const bool al = ((reinterpret_cast<uintptr_t>(Xa) | reinterpret_cast<uintptr_t>(Ya) |
                    reinterpret_cast<uintptr_t>(Xb) | reinterpret_cast<uintptr_t>(Yb)) & 15) == 0;
  if (n > 0 && al && D == 64 && E == 128) {
    hipLaunchKernelGGL((pe_wave_t_both_kernel<64, 128, 2, 1>), dim3((unsigned)(2 * ((n + 3) / 4))), dim3(256), 0, st,
                       n, ns, 1e-12f, Xa, Ya, Xb, Yb);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? ATLAS_OK : fail_hip(e, "pe_batched launch");
  }
  atlas_status r = atlas_pe_batched(n, D, E, ns, ATLAS_PE_NORM_EPS, Xa, Ya, ATLAS_DTYPE_F32, ATLAS_COMPUTE_F16, st);
  return r ? r : atlas_pe_batched(n, E, D, ns, ATLAS_PE_NORM_EPS, Xb, Yb, ATLAS_DTYPE_F32, ATLAS_COMPUTE_F16, st);
}

}  // namespace atlas

using namespace atlas;

extern "C" atlas_status atlas_pe_batched(int64_t n, int32_t d1, int32_t d2, int32_t ns_steps, int32_t norm_mode,
                                         const void* X, void* Y, int32_t dtype, int32_t compute, void* stream) {
  clear_error();
  if (n < 0 || d1 < 1 || d2 < 1) return fail(ATLAS_ERR_INVALID_ARGUMENT, "bad sizes n=%lld d1=%d d2=%d", (long long)n, d1, d2);
  if (n == 0) return ATLAS_OK;
  if (!X || !Y) return fail(ATLAS_ERR_INVALID_ARGUMENT, "NULL X or Y");
  if (ns_steps < 0 || ns_steps > 5) return fail(ATLAS_ERR_INVALID_ARGUMENT, "ns_steps %d outside [0, 5]", ns_steps);
  if (norm_mode != ATLAS_PE_NORM_EPS && norm_mode != ATLAS_PE_NORM_NO_EPS)
    return fail(ATLAS_ERR_INVALID_ARGUMENT, "bad norm_mode %d", norm_mode);
  if (dtype < 0 || dtype > 2) return fail(ATLAS_ERR_INVALID_ARGUMENT, "bad dtype %d", dtype);
  const int rows = d1 < d2 ? d1 : d2, cols = d1 < d2 ? d2 : d1;
  if (rows > 128 || cols > 256)
    return fail(ATLAS_ERR_UNSUPPORTED_SHAPE, "matrix %dx%d: the kernels need min dim <= 128 and max dim <= 256",
                d1, d2);
  if (n > (1LL << 33)) return fail(ATLAS_ERR_UNSUPPORTED_SHAPE, "n too large");
  const float eps = norm_mode == ATLAS_PE_NORM_EPS ? 1e-12f : 0.f;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (compute == ATLAS_COMPUTE_F16) return dispatch<ModeF16>(n, d1, d2, ns_steps, eps, X, Y, dtype, st);
  if (compute == ATLAS_COMPUTE_F32) return dispatch<ModeF32>(n, d1, d2, ns_steps, eps, X, Y, dtype, st);
  return fail(ATLAS_ERR_INVALID_ARGUMENT, "bad compute mode %d", compute);
}
