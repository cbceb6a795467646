// Memory-layer prologue after the input projections (atlas_jax/memory_layer.py
// :606-633): causal depthwise convolutions of q/k/v (ShortConv, :303-329),
// RMS norm (:211-216) and the polynomial feature map (:459-466) with the
// q/k asymmetry (q: norm then map; k: map then norm), and the sigmoid gates
// (eta times max_lr).  One wave per (b, t, h) token-head: lane l owns
// channels h*D + l and h*D + l + 64 of q, k and v (head dims up to 128); the
// RMS norm is a wave reduction.
//
// Input: the output of ONE projection GEMM x @ W_all^T with columns
//   [q (H*D) | k (H*D) | v (H*D) | gates (n_gates*H) | retrieve (H, optional)]
// (W_all stacks c_q, c_k, c_v, gate_alpha, gate_eta, gate_theta[, gate_gamma]
// [, retrieve_gate]); gate biases are added here.  All arithmetic is fp32.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "atlas_common.hpp"
#include "atlas_scan.h"
#include "atlas_status.hpp"

namespace atlas {
namespace {

constexpr int PRO_WAVES = 4;   // token-heads per workgroup
constexpr int PRO_CH = 2;      // channels per lane (head dims up to 2 x 64)
constexpr int RMS_WAVES = 4;   // rows per workgroup of the row norm

struct ProArgs {
  int B, T, H, D, K, P, NG, has_r;
  const void* proj;
  long long ld;
  int proj_dtype;
  const float* conv_w;   // (3, H*D, K)
  const float* conv_b;   // (3, H*D)
  const float* poly;     // (P)
  const float* gate_b;   // (NG, H)
  float max_lr;
  void *q, *k, *v;
  int out_dtype;
  float* gates;          // (NG, B, T, H)
  float* retrieve;       // (B, T, H)
};

__device__ __forceinline__ float poly_map(float x, const float* a, int P) {
  // sum_{i=1..P} a[i-1] x^i, powers accumulated left to right (as :459-466)
  float out = a[0] * x, xp = x;
  for (int i = 1; i < P; ++i) {
    xp *= x;
    out += a[i] * xp;
  }
  return out;
}

__global__ void __launch_bounds__(PRO_WAVES * WAVE) prologue_kernel(ProArgs a) {
  const int lane = lane_id();
  const long long item = (long long)blockIdx.x * PRO_WAVES + wave_id();   // (b, t, h)
  const long long n_items = (long long)a.B * a.T * a.H;
  if (item >= n_items) return;
  const int h = (int)(item % a.H);
  const long long bt = item / a.H;
  const int t = (int)(bt % a.T), b = (int)(bt / a.T);
  const int HD = a.H * a.D;
  // lane owns channels d = lane + 64 u (u < PRO_CH): head dims up to 128
  float vals[PRO_CH][3];
  bool act[PRO_CH];
#pragma unroll
  for (int u = 0; u < PRO_CH; ++u) {
    act[u] = lane + WAVE * u < a.D;
    const int d = act[u] ? lane + WAVE * u : 0;
#pragma unroll
    for (int which = 0; which < 3; ++which) {
      const int ch = which * HD + h * a.D + d;
      float acc = a.conv_b[which * HD + h * a.D + d];
      for (int j = 0; j < a.K; ++j) {
        const int ts = t - (a.K - 1) + j;
        if (ts >= 0)
          acc += a.conv_w[((long long)which * HD + h * a.D + d) * a.K + j] *
                 load_any(a.proj, ((long long)b * a.T + ts) * a.ld + ch, a.proj_dtype);
      }
      vals[u][which] = act[u] ? acc : 0.f;
    }
  }
  float qv[PRO_CH], kv[PRO_CH];
  const float inv_d = 1.f / (float)a.D;
  float sq = 0.f;
#pragma unroll
  for (int u = 0; u < PRO_CH; ++u) sq += vals[u][0] * vals[u][0];
  const float rq = rsqrtf(wave_sum(sq) * inv_d + 1e-6f);
#pragma unroll
  for (int u = 0; u < PRO_CH; ++u) {
    qv[u] = vals[u][0] * rq;
    if (a.P > 0) qv[u] = poly_map(qv[u], a.poly, a.P);
    kv[u] = (a.P > 0 && act[u]) ? poly_map(vals[u][1], a.poly, a.P) : vals[u][1];
  }
  float sk = 0.f;
#pragma unroll
  for (int u = 0; u < PRO_CH; ++u) sk += kv[u] * kv[u];
  const float rk = rsqrtf(wave_sum(sk) * inv_d + 1e-6f);
#pragma unroll
  for (int u = 0; u < PRO_CH; ++u) {
    if (act[u]) {
      const long long o = item * a.D + lane + WAVE * u;   // (B, T, H, D) dense
      store_any(a.q, o, a.out_dtype, qv[u]);
      store_any(a.k, o, a.out_dtype, kv[u] * rk);
      store_any(a.v, o, a.out_dtype, vals[u][2]);
    }
  }
  // gates: lanes 0..NG-1; retrieve gate: lane NG
  const long long row = ((long long)b * a.T + t) * a.ld + 3LL * HD;
  if (lane < a.NG) {
    const float z = load_any(a.proj, row + (long long)lane * a.H + h, a.proj_dtype) + a.gate_b[lane * a.H + h];
    float g = 1.f / (1.f + __expf(-z));
    if (lane == 1) g *= a.max_lr;
    a.gates[(long long)lane * n_items + item] = g;
  } else if (lane == a.NG && a.has_r) {
    const float z = load_any(a.proj, row + (long long)a.NG * a.H + h, a.proj_dtype);
    a.retrieve[item] = 1.f / (1.f + __expf(-z));
  }
}

// Four consecutive channels on their way from memory: DT 0 fp32, 1 bf16, 2
// fp16 as loaded (converted where they are used, so that the next token's
// loads can be in flight); DT -1: any dtype and alignment, converted at once;
// DT -2: any dtype, as loaded, aligned to the four elements.
template <int DT>
struct Quad {
  uint2 w;
  __device__ __forceinline__ void load(const void* p, int64_t i, int) {
    w = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(p) + i);
  }
  __device__ __forceinline__ f32x4 get() const {
    if constexpr (DT == 1)
      return f32x4{__uint_as_float(w.x << 16), __uint_as_float(w.x & 0xffff0000u), __uint_as_float(w.y << 16),
                   __uint_as_float(w.y & 0xffff0000u)};
    const f16x4 h = __builtin_bit_cast(f16x4, w);
    return f32x4{(float)h[0], (float)h[1], (float)h[2], (float)h[3]};
  }
};
template <>
struct Quad<0> {
  f32x4 v;
  __device__ __forceinline__ void load(const void* p, int64_t i, int) {
    v = *reinterpret_cast<const f32x4*>(static_cast<const float*>(p) + i);
  }
  __device__ __forceinline__ f32x4 get() const { return v; }
};
template <>
struct Quad<-1> {
  f32x4 v;
  __device__ __forceinline__ void load(const void* p, int64_t i, int dtype) {
    v = f32x4{load_any(p, i, dtype), load_any(p, i + 1, dtype), load_any(p, i + 2, dtype), load_any(p, i + 3, dtype)};
  }
  __device__ __forceinline__ f32x4 get() const { return v; }
};
template <>
struct Quad<-2> {
  f32x4 v;   // (16-bit channels: in the first half)
  int dt;
  __device__ __forceinline__ void load(const void* p, int64_t i, int dtype) {
    dt = dtype;
    if (dtype == 0) {
      v = *reinterpret_cast<const f32x4*>(static_cast<const float*>(p) + i);
    } else {
      const float2 w = *reinterpret_cast<const float2*>(static_cast<const uint16_t*>(p) + i);
      v = f32x4{w.x, w.y, 0.f, 0.f};
    }
  }
  __device__ __forceinline__ f32x4 get() const {
    if (dt == 0) return v;
    const uint2 w{__float_as_uint(v[0]), __float_as_uint(v[1])};
    return dt == 1 ? Quad<1>{w}.get() : Quad<2>{w}.get();
  }
};
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
template <int DT>
__device__ __forceinline__ void put4(void* p, int64_t i, int dtype, f32x4 x) {
  if constexpr (DT == 0)
    *reinterpret_cast<f32x4*>(static_cast<float*>(p) + i) = x;
  else if constexpr (DT == 1)
    *reinterpret_cast<bf16x4*>(static_cast<__bf16*>(p) + i) =
        bf16x4{(__bf16)x[0], (__bf16)x[1], (__bf16)x[2], (__bf16)x[3]};
  else if constexpr (DT == 2)
    *reinterpret_cast<f16x4*>(static_cast<_Float16*>(p) + i) =
        f16x4{(_Float16)x[0], (_Float16)x[1], (_Float16)x[2], (_Float16)x[3]};
  else if constexpr (DT == -2)
    store4_any(p, i, dtype, x);
  else
#pragma unroll
    for (int u = 0; u < 4; ++u) store_any(p, i + u, dtype, x[u]);
}
// Sum over the QD = 4, 8 or 16 consecutive lanes of a head, the far lanes first
// (i ^ 8, i ^ 4, i ^ 2, i ^ 1: the order fixes the last bit, and with it the
// rounding of the 16-bit outputs).  Rotations of the row of 16 reach those
// partners: after i ^ 8 the values repeat every 8 lanes, and so on.
__device__ __forceinline__ float head_sum(float x, int QD) {
  if (QD == 16) {
    x += dpp_f<0x128>(x);
    x += dpp_f<0x124>(x);
    x += dpp_f<0x122>(x);
    return x + dpp_f<0x121>(x);
  }
  if (QD == 8) x += dpp_f<0x1B>(dpp_f<0x141>(x));   // i ^ 7, then i ^ 3
  x += dpp_f<0x4E>(x);
  return x + dpp_f<0xB1>(x);
}
__device__ __forceinline__ float dot4(f32x4 p, f32x4 q) { return (p[0] * q[0] + p[1] * q[1]) + (p[2] * q[2] + p[3] * q[3]); }
// the polynomial's coefficients in registers
struct Poly {
  float c[8];
  int P;
  __device__ __forceinline__ Poly(const float* poly, int P_) : P(P_) {
#pragma unroll
    for (int i = 0; i < 8; ++i) c[i] = i < P ? poly[i] : 0.f;
  }
  __device__ __forceinline__ float operator()(float x) const {
    float out = c[0] * x, xp = x;
#pragma unroll
    for (int i = 1; i < 8; ++i) {
      if (i >= P) break;
      xp *= x;
      out += c[i] * xp;
    }
    return out;
  }
  // poly'(x) = sum_i i c_i x^{i-1}
  __device__ __forceinline__ float slope(float x) const {
    float dp = c[0], xp = 1.f;
#pragma unroll
    for (int i = 1; i < 8; ++i) {
      if (i >= P) break;
      xp *= x;
      dp += (float)(i + 1) * c[i] * xp;
    }
    return dp;
  }
};

// Vectorised variant for D in {16, 32, 64} and conv_kernel <= 4 (every
// configuration of the reference): one thread per four consecutive channels
// of a token row (the same four channels of q, k and v), a block per
// (b, run of PRO_TT tokens).  The thread keeps its 3 x 4 x K convolution
// weights in registers and slides a window of the last K projection rows
// over its tokens, so each projection element is loaded once (and the K - 1
// rows before a run again), 4 channels per load (8 or 16 bytes), the next
// token's row while this one is computed; q, k, v are stored 4 channels per
// store.  The RMS norms reduce over the D/4 threads of a head on the VALU.
// Bound by the serial chain of a run's tokens where there are few and by
// memory where there are many: B8 T4096 H8 D64, bf16, 91 -> 61 us (209 MB needed,
// 3.4 TB/s; 289 MB moved, the rows before each run again), one row of 60 tokens 49 -> 7.5 us.  Runs of 16 tokens load a
// fifth less and take 59 us and 22 us, H12 117 us against 101.
constexpr int PRO_TT = 4;    // tokens per block

template <int K, int DT>
__global__ void __launch_bounds__(256) prologue_vec_kernel(ProArgs a, int nthr) {
  const int tid = threadIdx.x;
  const int nruns = (a.T + PRO_TT - 1) / PRO_TT;
  const int b = blockIdx.x / nruns, t0 = (blockIdx.x % nruns) * PRO_TT;
  const int HD = a.H * a.D, QD = a.D / 4;   // threads per head
  const bool act = tid < nthr;
  const int j = act ? tid : 0, ch = 4 * j;
  const int t1 = min(t0 + PRO_TT, a.T);
  const int64_t row0 = (int64_t)b * a.T * a.ld + ch;
  // window: x[m][i] = projection row t - (K - 1) + i (zero before the sequence)
  Quad<DT> xw[3][K], nx[3];
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const int ts = max(t0 - (K - 1) + i, 0);
#pragma unroll
    for (int m = 0; m < 3; ++m) xw[m][i].load(a.proj, row0 + ts * a.ld + m * HD, a.proj_dtype);
  }
  // gates (n_gates x H) and the retrieve gate (H): one thread each
  const int ng = a.NG * a.H, ngr = ng + (a.has_r ? a.H : 0);
  const int g0 = tid < ngr ? tid : 0;
  const float gb = tid < ng ? a.gate_b[tid] : 0.f;
  float gz = load_any(a.proj, row0 - ch + t0 * a.ld + 3LL * HD + g0, a.proj_dtype);
  f32x4 w[3][K], bias[3];
#pragma unroll
  for (int m = 0; m < 3; ++m) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const long long base = ((long long)m * HD + ch + u) * a.K;
#pragma unroll
      for (int tap = 0; tap < K; ++tap) w[m][tap][u] = a.conv_w[base + tap];
      bias[m][u] = a.conv_b[m * HD + ch + u];
    }
  }
  const Poly poly(a.poly, a.P);
  f32x4 x[3][K];
#pragma unroll
  for (int m = 0; m < 3; ++m)
#pragma unroll
    for (int i = 0; i < K; ++i)
      x[m][i] = t0 - (K - 1) + i >= 0 ? xw[m][i].get() : f32x4{0.f, 0.f, 0.f, 0.f};
  const float inv_d = 1.f / (float)a.D;
  const long long n_items = (long long)a.B * a.T * a.H;
  for (int t = t0; t < t1; ++t) {
    const int tn = min(t + 1, t1 - 1);   // the next token's loads
#pragma unroll
    for (int m = 0; m < 3; ++m) nx[m].load(a.proj, row0 + tn * a.ld + m * HD, a.proj_dtype);
    const float gzn = load_any(a.proj, row0 - ch + tn * a.ld + 3LL * HD + g0, a.proj_dtype);
    f32x4 v3[3];
#pragma unroll
    for (int m = 0; m < 3; ++m) {
      f32x4 acc = bias[m];
#pragma unroll
      for (int tap = 0; tap < K; ++tap) acc += w[m][tap] * x[m][tap];
      v3[m] = acc;
    }
    // q: norm then map; k: map then norm (memory_layer.py:612-616)
    f32x4 qv = v3[0] * rsqrtf(head_sum(dot4(v3[0], v3[0]), QD) * inv_d + 1e-6f);
    f32x4 kv = v3[1];
    if (a.P > 0) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        qv[u] = poly(qv[u]);
        kv[u] = poly(kv[u]);
      }
    }
    kv = kv * rsqrtf(head_sum(dot4(kv, kv), QD) * inv_d + 1e-6f);
    if (act) {
      const long long o = ((long long)b * a.T + t) * HD + ch;   // (B, T, H, D) dense
      put4<DT>(a.q, o, a.out_dtype, qv);
      put4<DT>(a.k, o, a.out_dtype, kv);
      put4<DT>(a.v, o, a.out_dtype, v3[2]);
    }
    for (int g = tid; g < ngr; g += blockDim.x) {   // (one pass unless there are more gates than threads)
      const long long item = ((long long)b * a.T + t) * a.H + (g % a.H);
      const float z = g == tid ? gz : load_any(a.proj, row0 - ch + t * a.ld + 3LL * HD + g, a.proj_dtype);
      if (g < ng) {
        const int gi = g / a.H;
        float gv = 1.f / (1.f + __expf(-(z + (g == tid ? gb : a.gate_b[g]))));
        if (gi == 1) gv *= a.max_lr;
        a.gates[(long long)gi * n_items + item] = gv;
      } else {
        a.retrieve[item] = 1.f / (1.f + __expf(-z));
      }
    }
    gz = gzn;
#pragma unroll
    for (int m = 0; m < 3; ++m) {
#pragma unroll
      for (int i = 0; i + 1 < K; ++i) x[m][i] = x[m][i + 1];
      x[m][K - 1] = nx[m].get();
    }
  }
}

// (its loads and stores are all aligned to four elements; the dtype is compiled
// in where the taps are the default four and it is one for both)
template <int K>
void launch_prologue_vec(const ProArgs& a, unsigned blocks, int threads, int nthr, hipStream_t st) {
  auto go = [&](void (*k)(ProArgs, int)) { hipLaunchKernelGGL(k, dim3(blocks), dim3(threads), 0, st, a, nthr); };
  const int dt = K == 4 && a.proj_dtype == a.out_dtype ? a.proj_dtype : -2;
  if (dt == 0) go(prologue_vec_kernel<K, K == 4 ? 0 : -2>);
  else if (dt == 1) go(prologue_vec_kernel<K, K == 4 ? 1 : -2>);
  else if (dt == 2) go(prologue_vec_kernel<K, K == 4 ? 2 : -2>);
  else go(prologue_vec_kernel<K, -2>);
}

// ---- backward ---------------------------------------------------------------
// Gradients of the prologue (memory_layer.py:606-633) for the cotangents of
// q, k, v, the gates and the retrieve gate, with respect to the projection
// output, the conv weights and biases, the polynomial coefficients and the
// gate biases.  Per channel c of q/k/v with conv output y and cotangent dy of
// y (below): dx_s = sum_j w_j dy_{s+K-1-j}, dw_j = sum_t dy_t x_{t-K+1+j},
// db = sum_t dy_t.  dy from the normalisations (n = y r, r = (mean y^2 +
// 1e-6)^{-1/2}: d y = r (dn - n <dn, n> / D)):
//   q = poly(n):          dn = dq poly'(n);   dpoly_i += <dq, n^i>
//   k = rms(kp), kp = poly(y):  dkp = rms backward of dk;  dy = dkp poly'(y);
//                         dpoly_i += <dkp, y^i>
//   v:                    dy = dv
// (without the polynomial, q = rms(y) and k = rms(y)); gates g = s(z + b)
// (eta's times max_lr) and the retrieve gate r = s(z): dz = dg * scale * s(1 - s).
// One block per (b, run of PRO_BR tokens) with the forward vector kernel's
// thread layout (four channels of q, k and v per thread, head reductions by
// lane shuffles); each block also recomputes dy for the K - 1 tokens after
// its run (the halo its last tokens' dx needs).  The weight gradients are
// per-block partial sums, added in block order by prologue_bwd_reduce_kernel
// (bitwise reproducible).
constexpr int PRO_BR = 64;   // tokens per backward block and partial sum

struct ProBwdArgs {
  ProArgs f;                  // forward arguments (q, k, v, gates, retrieve unused)
  const void *gq, *gk, *gv;   // (B, T, H, D) cotangents, dtype gdt
  int gdt;
  const float* ggates;        // (NG, B, T, H)
  const float* gret;          // (B, T, H) or NULL
  void* dproj;                // (B, T, dld), dtype ddt
  long long dld;
  int ddt;
  float* part;                // per block: dw (3*HD*K), db (3*HD), dgb (NG*H), dpoly (P)
  int part_len;
};

// A block holds G groups of gthr threads (the vector layout's, whole waves);
// group g takes an equal share of the run's tokens, with the next token's loads
// in flight, and the groups' weight gradients are added through LDS in order,
// so the partial sums are one per run as with one group.  Bound by the chain of
// a group's tokens and the traffic: B8 T4096 H8 D64, bf16, 702 -> 165 us (one
// group of 64 tokens, scalar loads, lane shuffles).  DT: dtype of proj, the
// cotangents and dproj, rows aligned to four elements (-1: any).
template <int K, int DT>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2)))
prologue_bwd_kernel(ProBwdArgs a, int nthr, int gthr, int G) {
  const ProArgs& f = a.f;
  const int tid = threadIdx.x % gthr, grp = threadIdx.x / gthr;
  const int nruns = (f.T + PRO_BR - 1) / PRO_BR;
  const int b = blockIdx.x / nruns, t0 = (blockIdx.x % nruns) * PRO_BR;
  const int share = (PRO_BR + G - 1) / G;
  const int g0 = t0 + grp * share, g1 = min(g0 + share, min(t0 + PRO_BR, f.T));   // owned tokens [g0, g1)
  const int HD = f.H * f.D, QD = f.D / 4;
  const bool act = tid < nthr;
  const int j = act ? tid : 0, ch = 4 * j;
  const float inv_d = 1.f / (float)f.D;
  const int64_t row0 = (int64_t)b * f.T * f.ld, orow0 = (int64_t)b * f.T * HD + ch, drow0 = (int64_t)b * f.T * a.dld;
  extern __shared__ __attribute__((aligned(16))) float plds[];
  // the taps in LDS (one copy for the groups: 48 registers fewer per thread,
  // which otherwise spill)
  f32x4 bias[3];
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    f32x4 wt[K];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const long long base = ((long long)m * HD + ch + u) * f.K;
      if (grp == 0) {
#pragma unroll
        for (int tap = 0; tap < K; ++tap) wt[tap][u] = f.conv_w[base + tap];
      }
      bias[m][u] = f.conv_b[m * HD + ch + u];
    }
    if (grp == 0) {
#pragma unroll
      for (int tap = 0; tap < K; ++tap) *reinterpret_cast<f32x4*>(plds + ((m * K + tap) * gthr + tid) * 4) = wt[tap];
    }
  }
  __syncthreads();
  auto w = [&](int m, int tap) { return *reinterpret_cast<const f32x4*>(plds + ((m * K + tap) * gthr + tid) * 4); };
  const Poly poly(f.poly, f.P);
  Quad<DT> x[3][K];   // windows: x rows t-K+1 .. t (as loaded; zeros before the sequence), dy rows t-K+1 .. t
  f32x4 dyw[3][K];
  f32x4 dw[3][K], db[3];
  const f32x4 z4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    db[m] = z4;
#pragma unroll
    for (int i = 0; i < K; ++i) {
      dw[m][i] = z4;
      dyw[m][i] = z4;
    }
#pragma unroll
    for (int i = 0; i < K - 1; ++i) {
      const int ts = g0 - (K - 1) + i;
      x[m][i].load(f.proj, row0 + min(max(ts, 0), f.T - 1) * f.ld + m * HD + ch, f.proj_dtype);
      if (ts < 0) x[m][i] = Quad<DT>{};
    }
  }
  float dpoly[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  const long long n_items = (long long)f.B * f.T * f.H;
  const int ng = f.NG * f.H, ngr = ng + (f.has_r ? f.H : 0);
  float dgb = 0.f;   // this thread's gate bias (g = tid < ng), summed over the group's tokens
  Quad<DT> nx[3], ng_[3];
  auto fetch = [&](int t) {   // token t's rows (clamped into the sequence: loaded past it, not used)
    const int64_t tc = min(t, f.T - 1);
#pragma unroll
    for (int m = 0; m < 3; ++m) nx[m].load(f.proj, row0 + tc * f.ld + m * HD + ch, f.proj_dtype);
    ng_[0].load(a.gq, orow0 + tc * HD, a.gdt);
    ng_[1].load(a.gk, orow0 + tc * HD, a.gdt);
    ng_[2].load(a.gv, orow0 + tc * HD, a.gdt);
  };
  if (g0 < g1) fetch(g0);
  // t runs over the owned tokens and the K - 1 after them: the halo's dy
  // (recomputed; zero past the sequence end) completes the last owned dx
  for (int t = g0; g0 < g1 && t < g1 + K - 1; ++t) {
    const bool valid = t < f.T, own = t < g1;
    f32x4 gq = z4, gk = z4, gv = z4;
#pragma unroll
    for (int m = 0; m < 3; ++m) x[m][K - 1] = nx[m];
    if (act) {
      gq = ng_[0].get();
      gk = ng_[1].get();
      gv = ng_[2].get();
    }
    fetch(t + 1);
    f32x4 dy[3] = {z4, z4, z4};
    if (valid) {   // uniform over the group's waves: the head sums below see every lane
      f32x4 y[3];
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        f32x4 acc = bias[m];
#pragma unroll
        for (int tap = 0; tap < K; ++tap) acc += w(m, tap) * x[m][tap].get();
        y[m] = acc;
      }
      // q: n = rms(y), q = poly(n)
      {
        const float r = rsqrtf(head_sum(dot4(y[0], y[0]), QD) * inv_d + 1e-6f);
        const f32x4 n = y[0] * r;
        f32x4 dn = gq;
        if (f.P > 0) {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            if (own) {
              float pw = n[u];
#pragma unroll
              for (int i = 0; i < 8; ++i) {
                if (i >= f.P) break;
                dpoly[i] += gq[u] * pw;
                pw *= n[u];
              }
            }
            dn[u] = gq[u] * poly.slope(n[u]);
          }
        }
        const float sdot = head_sum(dot4(dn, n), QD) * inv_d;
        dy[0] = (dn - n * sdot) * r;
      }
      // k: kp = poly(y), k = rms(kp)
      {
        f32x4 kp = y[1], dpy = {1.f, 1.f, 1.f, 1.f};
        if (f.P > 0) {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            kp[u] = poly(y[1][u]);
            dpy[u] = poly.slope(y[1][u]);
          }
        }
        const float r = rsqrtf(head_sum(dot4(kp, kp), QD) * inv_d + 1e-6f);
        const f32x4 kn = kp * r;
        const float sdot = head_sum(dot4(gk, kn), QD) * inv_d;
        const f32x4 dkp = (gk - kn * sdot) * r;
        if (f.P > 0 && own) {
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            float pw = y[1][u];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              if (i >= f.P) break;
              dpoly[i] += dkp[u] * pw;
              pw *= y[1][u];
            }
          }
        }
        dy[1] = dkp * dpy;
      }
      dy[2] = gv;
      if (!act) dy[0] = dy[1] = z4;
      if (own) {
#pragma unroll
        for (int m = 0; m < 3; ++m) {
          db[m] += dy[m];
#pragma unroll
          for (int tap = 0; tap < K; ++tap) dw[m][tap] += dy[m] * x[m][tap].get();
        }
        // gates and the retrieve gate (one thread each)
        for (int g = tid; g < ngr; g += gthr) {
          const long long item = ((long long)b * f.T + t) * f.H + (g % f.H);
          const float zz = load_any(f.proj, row0 + t * f.ld + 3LL * HD + g, f.proj_dtype);
          float dz;
          if (g < ng) {
            const int gi = g / f.H;
            const float sg = 1.f / (1.f + __expf(-(zz + f.gate_b[g])));
            dz = a.ggates[(long long)gi * n_items + item] * (gi == 1 ? f.max_lr : 1.f) * sg * (1.f - sg);
            if (g == tid) dgb += dz;
          } else {
            const float sg = 1.f / (1.f + __expf(-zz));
            dz = a.gret ? a.gret[item] * sg * (1.f - sg) : 0.f;
          }
          store_any(a.dproj, drow0 + t * a.dld + 3LL * HD + g, a.ddt, dz);
        }
      }
    }
#pragma unroll
    for (int m = 0; m < 3; ++m) dyw[m][K - 1] = dy[m];
    // dx of token s = t - (K - 1): sum_j w_j dy_{s+K-1-j} = sum_j w_j dyw[K-1-j]
    const int s_ = t - (K - 1);
    if (s_ >= g0 && act) {   // s_ < g1 by the loop bound
#pragma unroll
      for (int m = 0; m < 3; ++m) {
        f32x4 acc = z4;
#pragma unroll
        for (int tap = 0; tap < K; ++tap) acc += w(m, tap) * dyw[m][K - 1 - tap];
        put4<DT>(a.dproj, drow0 + s_ * a.dld + m * HD + ch, a.ddt, acc);
      }
    }
    // slide the windows
#pragma unroll
    for (int m = 0; m < 3; ++m)
#pragma unroll
      for (int i = 0; i + 1 < K; ++i) {
        x[m][i] = x[m][i + 1];
        dyw[m][i] = dyw[m][i + 1];
      }
  }
  // the groups' sums added to group 0's, in order
  auto each = [&](auto&& op) {
    int n = 0;
#pragma unroll
    for (int m = 0; m < 3; ++m)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
#pragma unroll
        for (int tap = 0; tap < K; ++tap) dw[m][tap][u] = op(dw[m][tap][u], n++);
        db[m][u] = op(db[m][u], n++);
      }
#pragma unroll
    for (int i = 0; i < 8; ++i) dpoly[i] = op(dpoly[i], n++);
    dgb = op(dgb, n);
  };
  __syncthreads();   // the taps have been read
  for (int g = 1; g < G; ++g) {
    if (grp == g) each([&](float v, int n) { return plds[n * gthr + tid] = v; });
    __syncthreads();
    if (grp == 0) each([&](float v, int n) { return v + plds[n * gthr + tid]; });
    __syncthreads();
  }
  // block partials: dw, db (per channel), dgb (per gate bias), dpoly (block sum)
  float* pt = a.part + (long long)blockIdx.x * a.part_len;
  if (grp == 0 && act) {
#pragma unroll
    for (int m = 0; m < 3; ++m)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
#pragma unroll
        for (int tap = 0; tap < K; ++tap) pt[((long long)m * HD + ch + u) * f.K + tap] = dw[m][tap][u];
        pt[3LL * HD * f.K + m * HD + ch + u] = db[m][u];
      }
  }
  if (grp == 0 && tid < ng) pt[3LL * HD * (f.K + 1) + tid] = dgb;
  float* red = plds;   // [P][4 waves]
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    if (i >= f.P) break;
    const float v = wave_sum(act ? dpoly[i] : 0.f);
    if (grp == 0 && (tid & 63) == 0) red[4 * i + tid / 64] = v;
  }
  __syncthreads();
  if (grp == 0 && tid < f.P) {
    float v = 0.f;
    for (int wv = 0; wv < gthr / WAVE; ++wv) v += red[4 * tid + wv];
    pt[3LL * HD * (f.K + 1) + ng + tid] = v;
  }
}

// the block partials summed in a fixed order into d_conv_w (3*HD*K), d_conv_b
// (3*HD), d_gate_b (NG*H) and d_poly (P), laid out consecutively in a partial:
// a block per 32 columns, eight rows of threads each over every eighth
// partial, their sums added in order (512 partials of 7 714: 121 -> 7 us; one
// thread per column left 31 blocks in a serial chain of loads)
__global__ void __launch_bounds__(256) prologue_bwd_reduce_kernel(const float* part, int nblk, int len, int n_w,
                                                                  int n_b, int n_g, float* dw, float* db, float* dg,
                                                                  float* dp) {
  __shared__ float red[8][32];
  const int c = threadIdx.x & 31, r = threadIdx.x >> 5, i = blockIdx.x * 32 + c;
  float s = 0.f;
  if (i < len) {
#pragma unroll 8
    for (int blk = r; blk < nblk; blk += 8) s += part[(long long)blk * len + i];
  }
  red[r][c] = s;
  __syncthreads();
  if (r || i >= len) return;
#pragma unroll
  for (int k = 1; k < 8; ++k) s += red[k][c];
  if (i < n_w) dw[i] = s;
  else if (i < n_w + n_b) db[i - n_w] = s;
  else if (i < n_w + n_b + n_g) dg[i - n_w - n_b] = s;
  else dp[i - n_w - n_b - n_g] = s;
}

// (up to 69 KiB of LDS, at 256 threads to a group and four taps: the limit is
// raised as for every launch that passes 64 KiB)
template <int K>
hipError_t launch_prologue_bwd(const ProBwdArgs& a, unsigned nblk, int gthr, int nthr, bool aligned, hipStream_t st) {
  const int G = std::min(512 / gthr, PRO_BR / 4);
  const size_t lds = (size_t)gthr * (12 * K + 12 + 9) * sizeof(float);
  auto go = [&](void (*k)(ProBwdArgs, int, int, int)) {
    if (lds > 64 * 1024) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(k),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k, dim3(nblk), dim3(G * gthr), lds, st, a, nthr, gthr, G);
    return hipGetLastError();
  };
  const int dt = K == 4 && aligned && a.f.proj_dtype == a.gdt && a.f.proj_dtype == a.ddt ? a.gdt : -1;
  if (dt == 0) return go(prologue_bwd_kernel<K, K == 4 ? 0 : -1>);
  if (dt == 1) return go(prologue_bwd_kernel<K, K == 4 ? 1 : -1>);
  if (dt == 2) return go(prologue_bwd_kernel<K, K == 4 ? 2 : -1>);
  return go(prologue_bwd_kernel<K, -1>);
}

}  // namespace
}  // namespace atlas

using namespace atlas;

namespace atlas {
namespace {

// y = x / sqrt(mean(x^2) + 1e-6) over rows of C elements, in fp32, rounded to
// the dtype once (memory_layer.py:211-216).  Bound by its launch for a prompt
// and by memory for long rows: one wave per row, 16 bytes per lane and load,
// the row read again from the cache for the write.  The separate element-wise
// passes were seven launches: bf16 (60, 512) 34 -> 9 us, (8192, 1024)
// 53 -> 9, (32768, 512) 90 -> 13 (5.1 TB/s).
template <int DT, int VEC>
__global__ void __launch_bounds__(RMS_WAVES * WAVE) rms_norm_kernel(long long rows, int C, const void* x, void* y) {
  const long long row = (long long)blockIdx.x * RMS_WAVES + wave_id();
  if (row >= rows) return;
  using T = std::conditional_t<DT == ATLAS_DTYPE_F32, float, unsigned short>;
  typedef T vec __attribute__((ext_vector_type(VEC)));
  const T* xr = static_cast<const T*>(x) + row * C;
  T* yr = static_cast<T*>(y) + row * C;
  float sq = 0.f;
#pragma unroll 4
  for (int i = lane_id() * VEC; i < C; i += WAVE * VEC) {
    const vec v = *reinterpret_cast<const vec*>(xr + i);
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      const T e = v[j];
      const float f = load_any(&e, 0, DT);
      sq = fmaf(f, f, sq);
    }
  }
  const float r = rsqrtf(wave_sum(sq) / (float)C + 1e-6f);
#pragma unroll 4
  for (int i = lane_id() * VEC; i < C; i += WAVE * VEC) {
    const vec v = *reinterpret_cast<const vec*>(xr + i);
    vec o;
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      const T e = v[j];
      T z;
      store_any(&z, 0, DT, load_any(&e, 0, DT) * r);
      o[j] = z;
    }
    *reinterpret_cast<vec*>(yr + i) = o;
  }
}

template <int DT>
void launch_rms_norm(long long rows, int C, const void* x, void* y, hipStream_t st) {
  constexpr int VEC = DT == ATLAS_DTYPE_F32 ? 4 : 8;
  const dim3 grid((unsigned)((rows + RMS_WAVES - 1) / RMS_WAVES)), block(RMS_WAVES * WAVE);
  // 16-byte accesses where every row starts on one, else element by element
  const bool vec = C % VEC == 0 && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y)) & 15) == 0;
  if (vec) hipLaunchKernelGGL((rms_norm_kernel<DT, VEC>), grid, block, 0, st, rows, C, x, y);
  else hipLaunchKernelGGL((rms_norm_kernel<DT, 1>), grid, block, 0, st, rows, C, x, y);
}

}  // namespace
}  // namespace atlas

extern "C" atlas_status atlas_rms_norm(int64_t rows, int32_t C, const void* x, void* y, int32_t dtype, void* stream) {
  clear_error();
  if (rows < 0 || C < 1) return fail(ATLAS_ERR_INVALID_ARGUMENT, "rows %lld, C %d", (long long)rows, C);
  if (dtype < 0 || dtype > 2) return fail(ATLAS_ERR_INVALID_ARGUMENT, "bad dtype");
  if (rows == 0) return ATLAS_OK;
  if (!x || !y) return fail(ATLAS_ERR_INVALID_ARGUMENT, "null pointer");
  if ((rows + RMS_WAVES - 1) / RMS_WAVES > 0x7fffffffLL) return fail(ATLAS_ERR_UNSUPPORTED_SHAPE, "too many rows");
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == ATLAS_DTYPE_F32) launch_rms_norm<ATLAS_DTYPE_F32>(rows, C, x, y, st);
  else if (dtype == ATLAS_DTYPE_BF16) launch_rms_norm<ATLAS_DTYPE_BF16>(rows, C, x, y, st);
  else launch_rms_norm<ATLAS_DTYPE_F16>(rows, C, x, y, st);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? ATLAS_OK : fail_hip(e, "rms_norm launch");
}

extern "C" atlas_status atlas_layer_prologue(int32_t B, int32_t T, int32_t H, int32_t D, int32_t conv_kernel,
                                             int32_t poly_degree, int32_t n_gates, int32_t has_retrieve,
                                             const void* proj, int64_t proj_ld, int32_t proj_dtype,
                                             const float* conv_w, const float* conv_b, const float* poly,
                                             const float* gate_b, float max_lr, void* q, void* k, void* v,
                                             int32_t out_dtype, float* gates, float* retrieve, void* stream) {
  clear_error();
  if (B < 1 || T < 1 || H < 1) return fail(ATLAS_ERR_INVALID_ARGUMENT, "B, T, H must be >= 1");
  if (D < 1 || D > PRO_CH * WAVE)
    return fail(ATLAS_ERR_UNSUPPORTED_SHAPE, "head dim %d outside [1, %d]", D, PRO_CH * WAVE);
  if (conv_kernel < 1 || conv_kernel > 16) return fail(ATLAS_ERR_INVALID_ARGUMENT, "conv_kernel %d", conv_kernel);
  if (poly_degree < 0 || poly_degree > 8) return fail(ATLAS_ERR_INVALID_ARGUMENT, "poly_degree %d", poly_degree);
  if (n_gates < 3 || n_gates > 4) return fail(ATLAS_ERR_INVALID_ARGUMENT, "n_gates %d must be 3 or 4", n_gates);
  if (proj_dtype < 0 || proj_dtype > 2 || out_dtype < 0 || out_dtype > 2)
    return fail(ATLAS_ERR_INVALID_ARGUMENT, "bad dtype");
  const long long need = 3LL * H * D + (long long)(n_gates + (has_retrieve ? 1 : 0)) * H;
  if (proj_ld < need) return fail(ATLAS_ERR_INVALID_ARGUMENT, "proj_ld %lld < %lld columns", (long long)proj_ld, need);
  if (!proj || !conv_w || !conv_b || !gate_b || !q || !k || !v || !gates || (poly_degree > 0 && !poly) ||
      (has_retrieve && !retrieve))
    return fail(ATLAS_ERR_INVALID_ARGUMENT, "null pointer");
  ProArgs a{B, T, H, D, conv_kernel, poly_degree, n_gates, has_retrieve ? 1 : 0, proj, proj_ld, proj_dtype,
            conv_w, conv_b, poly, gate_b, max_lr, q, k, v, out_dtype, gates, retrieve};
  hipStream_t st = static_cast<hipStream_t>(stream);
  // vectorised path: 4-channel loads need the projection row, its stride and
  // the outputs aligned to 4 elements
  const int esz = proj_dtype == 0 ? 4 : 2, osz = out_dtype == 0 ? 4 : 2;
  const bool vec = (D == 16 || D == 32 || D == 64) && conv_kernel <= 4 && H * D / 4 <= 256 &&
                   proj_ld % 4 == 0 && reinterpret_cast<uintptr_t>(proj) % (4 * esz) == 0 &&
                   reinterpret_cast<uintptr_t>(q) % (4 * osz) == 0 && reinterpret_cast<uintptr_t>(k) % (4 * osz) == 0 &&
                   reinterpret_cast<uintptr_t>(v) % (4 * osz) == 0;
  if (vec) {
    const int nthr = H * D / 4, threads = (nthr + WAVE - 1) / WAVE * WAVE;
    const long long blocks = (long long)B * ((T + PRO_TT - 1) / PRO_TT);
    if (blocks > 0x7fffffffLL) return fail(ATLAS_ERR_UNSUPPORTED_SHAPE, "too many token rows");
    switch (conv_kernel) {
      case 1: launch_prologue_vec<1>(a, (unsigned)blocks, threads, nthr, st); break;
      case 2: launch_prologue_vec<2>(a, (unsigned)blocks, threads, nthr, st); break;
      case 3: launch_prologue_vec<3>(a, (unsigned)blocks, threads, nthr, st); break;
      default: launch_prologue_vec<4>(a, (unsigned)blocks, threads, nthr, st); break;
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail_hip(e, "prologue launch");
    return ATLAS_OK;
  }
  const long long items = (long long)B * T * H;
  const long long blocks = (items + PRO_WAVES - 1) / PRO_WAVES;
  if (blocks > 0x7fffffffLL) return fail(ATLAS_ERR_UNSUPPORTED_SHAPE, "too many token-heads");
  hipLaunchKernelGGL(prologue_kernel, dim3((unsigned)blocks), dim3(PRO_WAVES * WAVE), 0, st, a);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail_hip(e, "prologue launch");
  return ATLAS_OK;
}

namespace {

// the backward's vector layout (every reference configuration): D 16/32/64,
// conv kernel <= 4, one block row of H*D/4 <= 256 threads that also covers
// the gate biases
bool prologue_bwd_supported(int H, int D, int K, int NG) {
  const int nthr = H * D / 4, threads = (nthr + WAVE - 1) / WAVE * WAVE;
  return (D == 16 || D == 32 || D == 64) && K >= 1 && K <= 4 && nthr <= 256 && NG * H <= threads;
}

}  // namespace

extern "C" size_t atlas_layer_prologue_bwd_workspace_size(int32_t B, int32_t T, int32_t H, int32_t D,
                                                          int32_t conv_kernel, int32_t poly_degree,
                                                          int32_t n_gates) {
  if (B < 1 || T < 1 || poly_degree < 0 || poly_degree > 8 || n_gates < 3 || n_gates > 4 ||
      !prologue_bwd_supported(H, D, conv_kernel, n_gates))
    return 0;
  const long long HD = (long long)H * D;
  const long long len = 3 * HD * (conv_kernel + 1) + (long long)n_gates * H + poly_degree;
  const long long nblk = (long long)B * ((T + PRO_BR - 1) / PRO_BR);
  return (size_t)(nblk * len) * sizeof(float);
}

extern "C" atlas_status atlas_layer_prologue_bwd_as(
    int32_t B, int32_t T, int32_t H, int32_t D, int32_t conv_kernel, int32_t poly_degree, int32_t n_gates,
    int32_t has_retrieve, const void* proj, int64_t proj_ld, int32_t proj_dtype, const float* conv_w,
    const float* conv_b, const float* poly, const float* gate_b, float max_lr, const void* dq, const void* dk,
    const void* dv, int32_t grad_dtype, const float* dgates, const float* dretrieve, void* dproj, int64_t dproj_ld,
    int32_t dproj_dtype, float* d_conv_w, float* d_conv_b, float* d_poly, float* d_gate_b, void* workspace, size_t workspace_bytes,
    void* stream) {
  clear_error();
  if (B < 1 || T < 1 || H < 1) return fail(ATLAS_ERR_INVALID_ARGUMENT, "B, T, H must be >= 1");
  if (n_gates < 3 || n_gates > 4) return fail(ATLAS_ERR_INVALID_ARGUMENT, "n_gates %d must be 3 or 4", n_gates);
  if (poly_degree < 0 || poly_degree > 8) return fail(ATLAS_ERR_INVALID_ARGUMENT, "poly_degree %d", poly_degree);
  if (!prologue_bwd_supported(H, D, conv_kernel, n_gates))
    return fail(ATLAS_ERR_UNSUPPORTED_SHAPE, "prologue backward compiled for D 16/32/64, conv kernel <= 4 and "
                "H*D <= 1024 (got H %d D %d K %d)", H, D, conv_kernel);
  if (proj_dtype < 0 || proj_dtype > 2 || grad_dtype < 0 || grad_dtype > 2 || dproj_dtype < 0 || dproj_dtype > 2)
    return fail(ATLAS_ERR_INVALID_ARGUMENT, "bad dtype");
  const long long ncols = 3LL * H * D + (long long)(n_gates + (has_retrieve ? 1 : 0)) * H;
  if (proj_ld < ncols || dproj_ld < ncols)
    return fail(ATLAS_ERR_INVALID_ARGUMENT, "proj_ld / dproj_ld below the %lld projection columns", ncols);
  if (!proj || !conv_w || !conv_b || !gate_b || !dq || !dk || !dv || !dgates || !dproj || !d_conv_w || !d_conv_b ||
      !d_gate_b || (poly_degree > 0 && (!poly || !d_poly)))
    return fail(ATLAS_ERR_INVALID_ARGUMENT, "null pointer");
  const size_t need = atlas_layer_prologue_bwd_workspace_size(B, T, H, D, conv_kernel, poly_degree, n_gates);
  if (!workspace || workspace_bytes < need)
    return fail(ATLAS_ERR_WORKSPACE, "workspace %zu bytes < required %zu", workspace_bytes, need);
  const int esz = proj_dtype == 0 ? 4 : 2, gsz = grad_dtype == 0 ? 4 : 2, dsz = dproj_dtype == 0 ? 4 : 2;
  auto mis = [](const void* p, int al) { return reinterpret_cast<uintptr_t>(p) % al != 0; };
  if (mis(dq, 4 * gsz) || mis(dk, 4 * gsz) || mis(dv, 4 * gsz) || mis(workspace, 4))
    return fail(ATLAS_ERR_INVALID_ARGUMENT, "the q/k/v cotangents must be 4-element aligned");
  ProBwdArgs a;
  a.f = ProArgs{B, T, H, D, conv_kernel, poly_degree, n_gates, has_retrieve ? 1 : 0, proj, proj_ld, proj_dtype,
                conv_w, conv_b, poly, gate_b, max_lr, nullptr, nullptr, nullptr, 0, nullptr, nullptr};
  a.gq = dq; a.gk = dk; a.gv = dv; a.gdt = grad_dtype;
  a.ggates = dgates; a.gret = has_retrieve ? dretrieve : nullptr;
  a.dproj = dproj; a.dld = dproj_ld; a.ddt = dproj_dtype;
  a.part = static_cast<float*>(workspace);
  const long long HD = (long long)H * D;
  const int n_w = (int)(3 * HD * conv_kernel), n_b = (int)(3 * HD), n_g = n_gates * H;
  a.part_len = n_w + n_b + n_g + poly_degree;
  const int nthr = H * D / 4, threads = (nthr + WAVE - 1) / WAVE * WAVE;
  const long long nblk = (long long)B * ((T + PRO_BR - 1) / PRO_BR);
  if (nblk > 0x7fffffffLL) return fail(ATLAS_ERR_UNSUPPORTED_SHAPE, "too many token rows");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const bool aligned = proj_ld % 4 == 0 && dproj_ld % 4 == 0 && !mis(proj, 4 * esz) && !mis(dproj, 4 * dsz);
  hipError_t e;
  switch (conv_kernel) {
    case 1: e = launch_prologue_bwd<1>(a, (unsigned)nblk, threads, nthr, aligned, st); break;
    case 2: e = launch_prologue_bwd<2>(a, (unsigned)nblk, threads, nthr, aligned, st); break;
    case 3: e = launch_prologue_bwd<3>(a, (unsigned)nblk, threads, nthr, aligned, st); break;
    default: e = launch_prologue_bwd<4>(a, (unsigned)nblk, threads, nthr, aligned, st); break;
  }
  if (e != hipSuccess) return fail_hip(e, "prologue backward launch");
  hipLaunchKernelGGL(prologue_bwd_reduce_kernel, dim3((unsigned)((a.part_len + 31) / 32)), dim3(256), 0, st,
                     a.part, (int)nblk, a.part_len, n_w, n_b, n_g, d_conv_w, d_conv_b, d_gate_b, d_poly);
  e = hipGetLastError();
  return e == hipSuccess ? ATLAS_OK : fail_hip(e, "prologue backward launch");
}

extern "C" atlas_status atlas_layer_prologue_bwd(
    int32_t B, int32_t T, int32_t H, int32_t D, int32_t conv_kernel, int32_t poly_degree, int32_t n_gates,
    int32_t has_retrieve, const void* proj, int64_t proj_ld, int32_t proj_dtype, const float* conv_w,
    const float* conv_b, const float* poly, const float* gate_b, float max_lr, const void* dq, const void* dk,
    const void* dv, int32_t grad_dtype, const float* dgates, const float* dretrieve, float* dproj, int64_t dproj_ld,
    float* d_conv_w, float* d_conv_b, float* d_poly, float* d_gate_b, void* workspace, size_t workspace_bytes,
    void* stream) {
  return atlas_layer_prologue_bwd_as(B, T, H, D, conv_kernel, poly_degree, n_gates, has_retrieve, proj, proj_ld,
                                     proj_dtype, conv_w, conv_b, poly, gate_b, max_lr, dq, dk, dv, grad_dtype, dgates,
                                     dretrieve, dproj, dproj_ld, 0, d_conv_w, d_conv_b, d_poly, d_gate_b, workspace,
                                     workspace_bytes, stream);
}
