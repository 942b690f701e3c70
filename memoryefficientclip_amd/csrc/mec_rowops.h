// O(N*D) and O(N) kernels around the MFMA hot loops: the normalisation /
// diagonal pre-pass, the loss finalize, and the gradient post-pass.  These are
// HBM-bound; one 64-lane wave owns one feature row.
#pragma once
#include <type_traits>

#include "mec_common.h"

namespace mec {

template <typename T> struct Elem;
template <> struct Elem<float> {
  static __device__ __forceinline__ float load(const float* p, int64_t i) { return p[i]; }
  static __device__ __forceinline__ void store(float* p, int64_t i, float v) { p[i] = v; }
};
template <> struct Elem<uint16_t> {  // bf16 bits
  static __device__ __forceinline__ float load(const uint16_t* p, int64_t i) { return bf16_to_f32(p[i]); }
  static __device__ __forceinline__ void store(uint16_t* p, int64_t i, float v) { p[i] = f32_to_bf16(v); }
};
template <> struct Elem<_Float16> {
  static __device__ __forceinline__ float load(const _Float16* p, int64_t i) { return (float)p[i]; }
  static __device__ __forceinline__ void store(_Float16* p, int64_t i, float v) { p[i] = (_Float16)v; }
};

// V consecutive elements of a row as floats, and back: one 16-byte vector (fp32
// V = 4, 16-bit V = 8; 16-byte aligned)
template <typename T> constexpr int kVec16 = 16 / (int)sizeof(T);
template <typename T>
__device__ __forceinline__ void load_vec(const T* __restrict__ p, float (&v)[kVec16<T>]) {
  if constexpr (sizeof(T) == 4) {
    const f32x4 u = *(const f32x4*)p;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = u[e];
  } else {
    typedef T tvec __attribute__((ext_vector_type(8)));
    const tvec u = *(const tvec*)p;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const T t = u[e];
      v[e] = Elem<T>::load(&t, 0);
    }
  }
}
template <typename T>
__device__ __forceinline__ void store_vec(T* __restrict__ p, const float (&v)[kVec16<T>]) {
  if constexpr (sizeof(T) == 4) {
    *(f32x4*)p = f32x4{v[0], v[1], v[2], v[3]};
  } else {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    u32x4 u;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      u[e] = std::is_same<T, uint16_t>::value ? pack2_bf16(v[2 * e], v[2 * e + 1]) : pack2_f16(v[2 * e], v[2 * e + 1]);
    *(u32x4*)p = u;
  }
}

// How the gradient matrix of split pairs is stored: its scale, the scale's
// inverse, and whether as fp32 values (wide) instead of pairs.
//
// A pair holds v with an error of at most 2^-23 |v| or 2^-25, whichever is
// larger, so a matrix of pairs has one scale for all of it: the largest 2^k with
// 2^k G'_ij <= 2^15 that the row sums allow, at least 2^14 (G' <= 2): G'_ij =
// E_ij (1/R_i + 1/C_j) <= row_off_i / R_i + col_off_j / C_j <= 2 max |kappa|.
// Row i of the gradient is a sum of terms whose sizes add up to at least its
// share s_i = row_off_i / R_i (columns: col_off_j / C_j), to which N entries
// off by 2^-25-k each (of either sign) add an error of about sqrt(N) 2^-25-k.
// With 2^k s_i >= sqrt(N) that is no more than 2^-25 s_i, an fp32 rounding.
// Where one row has less (pairs that match well beside one that does not: the
// small shares' entries fall below fp16's range, the lo parts first), or the
// scale stops at 2^39, the matrix is held wide, at fp32's range and precision,
// and contracted as three bf16 terms (mec_gemm_wide.h).  Distance of a row's
// off-diagonal sum from 64 bits, the largest over the rows, fp32 kernels, pairs
// throughout, this rule: 4097 x 768, T = 0.03, two y rows swapped: 3.9e-6, 1.0
// (nothing left of it), 3.5e-6; 4200 x 512, T = 0.02, all pairs matching (loss
// 4e-16) 9.0e-6, 0.12, 8.9e-6.
struct PairGrad {
  float scale, inv;
  bool wide;
};
constexpr int PAIR_G_MIN_EXP = -26;
__device__ __forceinline__ PairGrad pair_grad_scale(int N, const float* __restrict__ scl) {
  const float m = scl[SCL_KMAX], smin = scl[SCL_SMIN];
  int e = 0;  // 2 max |kappa| < 2^(e + 1)
  if (m < 0.5f) (void)frexpf(fmaxf(m, ldexpf(1.f, PAIR_G_MIN_EXP)), &e);
  PairGrad g{ldexpf(1.f, 14 - e), ldexpf(1.f, e - 14), false};
  if (!(g.scale * smin >= sqrtf((float)N))) {
    // (2^40: entries down to fp32's smallest keep their lower terms)
    g = PairGrad{ldexpf(1.f, 40), ldexpf(1.f, -40), true};
  }
  return g;
}
// The rows of a workgroup's first NW waves into SCL_KMAX and SCL_SMIN (k: |kappa|,
// s: share; 0 and infinity without a row; every thread calls it): one atomic of
// each per workgroup (one per wave was 10 us of atomics at n = 32768).
template <int NW>
__device__ __forceinline__ void pair_grad_range(float k, float s, float* __restrict__ scl) {
  __shared__ float s_k[NW], s_s[NW];
  for (int o = 32; o >= 1; o >>= 1) {
    k = fmaxf(k, __shfl_xor(k, o, 64));
    s = fminf(s, __shfl_xor(s, o, 64));
  }
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0 && w < NW) {
    s_k[w] = k;
    s_s[w] = s;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int q = 1; q < NW; ++q) {
      k = fmaxf(k, s_k[q]);
      s = fminf(s, s_s[q]);
    }
    atomicMax((unsigned int*)(scl + SCL_KMAX), __float_as_uint(k));
    atomicMin((unsigned int*)(scl + SCL_SMIN), __float_as_uint(s));
  }
}

// Per row i: rx = 1/max(||x_i||, 1e-12) (or 1), ry likewise, diag = x_i . y_i.
// Also clears the off-diagonal sum accumulators used by the sum-exp kernel.
// Follows F.normalize(dim=1) as applied at clip_loss.py:266-268 and the
// einsum('bi,bi->b') diagonal at clip_loss.py:206.
// VEC: 16-byte aligned rows, D a multiple of the vector.
template <typename T, bool NORM, bool VEC>
__global__ __launch_bounds__(256) void k_prepass(const T* __restrict__ X, int64_t ldx,
                                                 const T* __restrict__ Y, int64_t ldy, int N, int D,
                                                 float* __restrict__ ws, uint32_t* __restrict__ counter) {
  if (counter && blockIdx.x == 0 && threadIdx.x == 0) *counter = 0u;  // (k_finalize_all)
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= N) return;
  const T* x = X + (int64_t)row * ldx;
  const T* y = Y + (int64_t)row * ldy;
  float sx = 0.f, sy = 0.f, sxy = 0.f;
  if constexpr (VEC) {
    // (16-byte vectors; up to four of each row in flight)
    constexpr int V = kVec16<T>;
    for (int d0 = V * lane; d0 < D; d0 += 256 * V) {
      float a[4][V], b[4][V];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int d = d0 + 64 * V * k;
        if (d < D) {
          load_vec<T>(x + d, a[k]);
          load_vec<T>(y + d, b[k]);
        } else {
#pragma unroll
          for (int e = 0; e < V; ++e) a[k][e] = b[k][e] = 0.f;
        }
      }
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int e = 0; e < V; ++e) {
          sx = fmaf(a[k][e], a[k][e], sx);
          sy = fmaf(b[k][e], b[k][e], sy);
          sxy = fmaf(a[k][e], b[k][e], sxy);
        }
    }
  } else {
    for (int d = lane; d < D; d += 64) {
      float a = Elem<T>::load(x, d), b = Elem<T>::load(y, d);
      sx = fmaf(a, a, sx);
      sy = fmaf(b, b, sy);
      sxy = fmaf(a, b, sxy);
    }
  }
  sx = wave_sum(sx);
  sy = wave_sum(sy);
  sxy = wave_sum(sxy);
  if (lane == 0) {
    const int64_t n = N;
    float rx = 1.f, ry = 1.f;
    if (NORM) {
      rx = 1.f / fmaxf(sqrtf(sx), 1e-12f);
      ry = 1.f / fmaxf(sqrtf(sy), 1e-12f);
    }
    ws[WS_RX * n + row] = rx;
    ws[WS_RY * n + row] = ry;
    ws[WS_DIAG * n + row] = sxy;
    ws[WS_ROW_OFF * n + row] = 0.f;
    ws[WS_COL_OFF * n + row] = 0.f;
  }
}

// Loss epilogue (clip_loss.py:206-211, lit_loss.py:199-203) plus the per-row
// quantities the backward needs.  In natural-log units with t_i = (s_ii-1)/T:
//   R_i = row_off_i + e^{t_i},  l^r_i = ln R_i - t_i = softplus(ln row_off_i - t_i)
// which is the same cross-entropy term as -ln(2^Sv_i / R_i) in the reference,
// evaluated without cancellation.  CLIP averages (l^r + l^c)/2, LiT uses l^r.
// kappa_i = -(row_off_i/R_i + col_off_i/C_i) is the exact diagonal entry of
// the gradient matrix in units of a = grad_scale/(2N) (LiT: grad_scale/N).
// Two passes (rows, then the sum of per-workgroup partials), fp64
// accumulation in a fixed order: deterministic.
__device__ __forceinline__ double softplus_log_ratio(double off, double t) {
  if (!(off > 0.0)) return 0.0;
  double u = log(off) - t;
  return u > 0.0 ? u + log1p(exp(-u)) : log1p(exp(u));
}

// The off-diagonal share of row i's sum, and of column i's where that is less
// (CLIP): the smallest of what pair_grad_scale is told of.
template <bool LIT>
__device__ __forceinline__ float least_share(double ro, double R, double co, double C) {
  const float r = (float)(ro / R);
  return LIT ? r : fminf(r, (float)(co / C));
}

// The loss term of row i (a CLIP row and column, or a LiT row), and 1/R_i,
// 1/C_i and kappa_i into the workspace; -kappa_i and least_share.
template <bool LIT>
__device__ __forceinline__ double finalize_row(int i, int64_t n, double inv_t, float* __restrict__ ws, float& kout,
                                               float& sout) {
  const double s = (double)ws[WS_DIAG * n + i] * (double)ws[WS_RX * n + i] * (double)ws[WS_RY * n + i];
  const double t = (s - 1.0) * inv_t;
  const double e = exp(t);
  const double ro = ws[WS_ROW_OFF * n + i];
  const double R = ro + e;
  double acc = softplus_log_ratio(ro, t);
  ws[WS_INV_ROW * n + i] = (float)(1.0 / R);
  double kap = -(ro / R);
  double co = 0.0, C = 1.0;
  if (!LIT) {
    co = ws[WS_COL_OFF * n + i];
    C = co + e;
    acc += softplus_log_ratio(co, t);
    ws[WS_INV_COL * n + i] = (float)(1.0 / C);
    kap -= co / C;
  }
  ws[WS_KAPPA * n + i] = (float)kap;
  kout = -(float)kap;
  sout = least_share<LIT>(ro, R, co, C);
  return acc;
}

// Pass 1: one thread per row (rows beyond N contribute nothing), FIN_ROWS
// rows per workgroup; each workgroup writes the fp64 sum of its rows' loss
// terms to partial[blockIdx.x].  SINGLE (N <= FIN_SINGLE_ROWS): one
// workgroup of FIN_SINGLE_ROWS threads, one row each, writes the loss itself
// (no second pass).  One row per thread spreads the rows' fp64 work over N /
// 256 CUs: with one 1024-thread workgroup taking up to four rows per thread
// up to N = 4096, the finalize took 11 us at N = 2048 and 21 us at N = 4096
// (each row's loads, fp64 exp / log and stores one after the other on one
// CU), against 8.8 and 9.4 us for both passes now; up to 1024 rows the one
// workgroup stays faster than two launches (6 against 9 us).
constexpr int FIN_SINGLE_ROWS = 1024;
template <bool LIT, bool SINGLE>
__global__ __launch_bounds__(SINGLE ? FIN_SINGLE_ROWS : FIN_ROWS) void k_finalize_rows(
    int N, double inv_t, float* __restrict__ ws, double* __restrict__ partial, float* __restrict__ loss) {
  constexpr int NT = SINGLE ? FIN_SINGLE_ROWS : FIN_ROWS;
  __shared__ double red[NT / 64];
  const int64_t n = N;
  const int i = blockIdx.x * NT + threadIdx.x;
  float kap, share;
  double acc = i < N ? finalize_row<LIT>(i, n, inv_t, ws, kap, share) : 0.0;
  acc = wave_sum_f64(acc);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) red[w] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double tot = 0.0;
    for (int k = 0; k < NT / 64; ++k) tot += red[k];
    if (SINGLE)
      *loss = (float)(tot / (LIT ? (double)N : 2.0 * (double)N));
    else
      partial[blockIdx.x] = tot;
  }
}

// Pass 2 (one workgroup): loss = sum of the partials in a fixed order / (N or 2N).
template <bool LIT>
__global__ __launch_bounds__(1024) void k_finalize_sum(int N, int nparts, const double* __restrict__ partial,
                                                       float* __restrict__ loss) {
  __shared__ double red[16];
  double acc = 0.0;
  for (int k = threadIdx.x; k < nparts; k += blockDim.x) acc += partial[k];
  acc = wave_sum_f64(acc);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) red[w] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double tot = 0.0;
    for (int k = 0; k < (int)(blockDim.x >> 6); ++k) tot += red[k];
    *loss = (float)(tot / (LIT ? (double)N : 2.0 * (double)N));
  }
}

// The finalize of mec_forward in one launch: DET: the partial sums of the
// deterministic forward first (row i's Q row partials and P column partials,
// four threads per row, partials k, k + 4, ... each, then the four in order);
// finalize_row on FIN_ROWS rows; the workgroup's fp64 loss sum to partial[];
// and the last workgroup to arrive at `counter` (zeroed by the pre-pass) adds
// the partials in order and writes the loss.  The counter is the loss word
// itself, which nobody reads before the launch ends.  The handshake is a
// release / acquire of one thread per workgroup.  pair_scl (split pairs, else
// null) gets the rows' range (pair_grad_range).  Latency-bound: as separate
// launches (k_det_reduce with one thread per row adding 48 partials one after
// the other, rows, sum) it took 11 + 5 + 5 us at n = 6001, 16 + 5 + 5 us at 8192.
template <bool LIT, bool DET>
__global__ __launch_bounds__(DET ? 4 * FIN_ROWS : FIN_ROWS) void k_finalize_all(
    int N, double inv_t, float* __restrict__ ws, const float* __restrict__ rowpart, int Q,
    const float* __restrict__ colpart, int P, double* partial, uint32_t* counter, float* loss,
    float* __restrict__ pair_scl) {
  constexpr int NT = DET ? 4 * FIN_ROWS : FIN_ROWS;
  constexpr int MQ = DET_Q / 4, MP = DET_P / 4;
  __shared__ float s_r[DET ? 4 : 1][FIN_ROWS], s_c[DET ? 4 : 1][FIN_ROWS];
  __shared__ double red[NT / 64];
  __shared__ bool s_last;
  const int64_t n = N;
  const int r = threadIdx.x % FIN_ROWS, q = threadIdx.x / FIN_ROWS;
  const int i = blockIdx.x * FIN_ROWS + r;
  if constexpr (DET) {
    // every load at a valid address, issued back to back
    const int ic = min(i, N - 1);
    float rv[MQ], cv[LIT ? 1 : MP];
#pragma unroll
    for (int k = 0; k < MQ; ++k) rv[k] = rowpart[min(4 * k + q, Q - 1) * n + ic];
    if constexpr (!LIT) {
#pragma unroll
      for (int k = 0; k < MP; ++k) cv[k] = colpart[min(4 * k + q, P - 1) * n + ic];
    }
    float a = 0.f, b = 0.f;
#pragma unroll
    for (int k = 0; k < MQ; ++k) a += 4 * k + q < Q ? rv[k] : 0.f;
    s_r[q][r] = a;
    if constexpr (!LIT) {
#pragma unroll
      for (int k = 0; k < MP; ++k) b += 4 * k + q < P ? cv[k] : 0.f;
      s_c[q][r] = b;
    }
    __syncthreads();
    if (q == 0 && i < N) {
      ws[WS_ROW_OFF * n + i] = (s_r[0][r] + s_r[1][r]) + (s_r[2][r] + s_r[3][r]);
      if (!LIT) ws[WS_COL_OFF * n + i] = (s_c[0][r] + s_c[1][r]) + (s_c[2][r] + s_c[3][r]);
    }
  }
  // (the same thread reads back what it wrote)
  float kap = 0.f, share = __builtin_inff();
  double acc = q == 0 && i < N ? finalize_row<LIT>(i, n, inv_t, ws, kap, share) : 0.0;
  if (pair_scl) pair_grad_range<FIN_ROWS / 64>(kap, share, pair_scl);
  acc = wave_sum_f64(acc);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) red[w] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    double tot = 0.0;
    for (int k = 0; k < FIN_ROWS / 64; ++k) tot += red[k];
    __hip_atomic_store(&partial[blockIdx.x], tot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
  }
  __syncthreads();
  if (!s_last) return;
  double sum = 0.0;
  for (int k = threadIdx.x; k < (int)gridDim.x; k += NT)
    sum += __hip_atomic_load(&partial[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  sum = wave_sum_f64(sum);
  if (lane == 0) red[w] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    double tot = 0.0;
    for (int k = 0; k < NT / 64; ++k) tot += red[k];
    *loss = (float)(tot / (LIT ? (double)N : 2.0 * (double)N));
  }
}

// Gradient post-pass for one side.  With acc the off-diagonal contraction
// sum_{j != i} G'_ij * oth^_j (oth^ = normalised other side) and a the
// scale grad_scale/(2N) (LiT: /N):
//   d_own^_i = a * (acc_i + kappa_i * oth^_i)                       (diag term)
//   d_own_i  = r_i (d_own^_i - own^_i <own^_i, d_own^_i>)            (F.normalize bwd)
//            = r_i d_own^_i                                           (if ||own_i|| <= eps)
//   out_i    = grad_output * d_own_i                                 (clip_loss.py:252-254)
// out may alias acc (fp32 outputs): every element is read before it is written
// by the same lane.  One wave per row; rows of D <= 64 * POST_REG are read
// once (held in registers across the reduction), longer rows twice.
constexpr int POST_REG = 32;
// One side of the post-pass (the x side: own = x, oth = y, acc_x -> dx); the
// two sides share one launch: blockIdx.y picks the side.
template <typename T>
struct PostSide {
  const T* own;
  int64_t ld_own;
  const T* oth;
  int64_t ld_oth;
  const float* r_own;
  const float* r_oth;
  const float* acc;
  T* out;
  const float* part;  // nparts - 1 further parts of the accumulators, n x D each (contractions split over k)
};
// ACCR (fp32 data on the fp32 kernels): the accumulator row carries the
// row's own inverse norm, acc = r_i (sum_j G'_ij y^_j), since the
// contractions multiply H = diag(rx) G' diag(ry) with the raw inputs.  Then
// h = a (kappa_i r_i y^_i + acc) = r_i dx^_i, and the normalisation backward
// r_i (dx^ - x^ <x^, dx^>) is h - x^ <x^, h>: no division by the norm.
// Rows that are not 16-byte vectors, or longer than k_postpass_vec takes.
template <typename T, bool NORM, bool ACCR = false>
__global__ __launch_bounds__(256) void k_postpass(PostSide<T> s0, PostSide<T> s1, int N, int D,
                                                  const float* __restrict__ kappa, float a,
                                                  const float* __restrict__ grad_output, int nparts) {
  const PostSide<T>& sd = blockIdx.y ? s1 : s0;
  const T* __restrict__ own = sd.own;
  const int64_t ld_own = sd.ld_own;
  const T* __restrict__ oth = sd.oth;
  const int64_t ld_oth = sd.ld_oth;
  const float* __restrict__ r_own = sd.r_own;
  const float* __restrict__ r_oth = sd.r_oth;
  const float* acc = sd.acc;
  T* out = sd.out;
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= N) return;
  const T* xo = own + (int64_t)row * ld_own;
  const T* yo = oth + (int64_t)row * ld_oth;
  const float* ac = acc + (int64_t)row * D;
  const float* pt = sd.part + (int64_t)row * D;
  const int64_t ps = (int64_t)N * D;
  // accumulated sums of feature d: the parts in order
  auto accv = [&](int d) {
    float v = ac[d];
    for (int p = 0; p + 1 < nparts; ++p) v += pt[p * ps + d];
    return v;
  };
  T* o = out + (int64_t)row * D;
  const float ro = r_own[row];
  const float kq = kappa[row] * r_oth[row] * (ACCR ? ro : 1.f);
  const float go = grad_output ? *grad_output : 1.f;
  if (NORM) {
    float dot = 0.f;
    const bool clamped = ro >= 1e12f;
    if (D <= 64 * POST_REG) {
      // the row stays in registers between the reduction and the stores
      float g[POST_REG], xr[POST_REG];
#pragma unroll
      for (int k = 0; k < POST_REG; ++k) {
        const int d = lane + 64 * k;
        g[k] = 0.f;
        xr[k] = 0.f;
        if (d < D) {
          g[k] = a * fmaf(kq, Elem<T>::load(yo, d), accv(d));
          xr[k] = Elem<T>::load(xo, d) * ro;
          dot = fmaf(xr[k], g[k], dot);
        }
      }
      dot = wave_sum(dot);
#pragma unroll
      for (int k = 0; k < POST_REG; ++k) {
        const int d = lane + 64 * k;
        if (d < D) {
          const float v = ACCR ? (clamped ? g[k] : g[k] - xr[k] * dot) : (clamped ? ro * g[k] : ro * (g[k] - xr[k] * dot));
          Elem<T>::store(o, d, go * v);
        }
      }
      return;
    }
    for (int d = lane; d < D; d += 64) {
      float g = a * fmaf(kq, Elem<T>::load(yo, d), accv(d));
      dot = fmaf(Elem<T>::load(xo, d) * ro, g, dot);
    }
    dot = wave_sum(dot);
    for (int d = lane; d < D; d += 64) {
      float g = a * fmaf(kq, Elem<T>::load(yo, d), accv(d));
      const float xh = Elem<T>::load(xo, d) * ro;
      float v = ACCR ? (clamped ? g : g - xh * dot) : (clamped ? ro * g : ro * (g - xh * dot));
      Elem<T>::store(o, d, go * v);
    }
  } else {
    for (int d = lane; d < D; d += 64) {
      float g = a * fmaf(kq, Elem<T>::load(yo, d), accv(d));
      Elem<T>::store(o, d, go * g);
    }
  }
}

// k_postpass on 16-byte vectors, BOTH: both sides at once (else side s0, s1 naming
// the other side's input): one wave per row takes x_i, y_i and the accumulator
// rows (with their parts), so that x and y are read once instead of once per
// side.  HBM-bound: bf16 4096 x 768 with two parts 23 -> 12.5 us, 16384 x 1024 78
// -> 42 us (268 MB, 6.4 TB/s with the Infinity Cache's help), fp32 32768 x 1152
// 215 -> 146 us; one side, bf16 2048 x 768 with eight parts 14.7 -> 6.1 us.  Rows of up to NV x 64 vectors, 16-byte
// aligned (own, other, accumulators, parts and outputs; D a multiple of the
// vector).  The same arithmetic as k_postpass; only the order of the feature sum
// <x^, h> differs.  NV sizes the registers: 16 features per lane up to D = 1024,
// 32 up to D = 2048.
template <typename T, bool NORM, bool ACCR, bool BOTH, int NV>
__global__ __launch_bounds__(256) void k_postpass_vec(PostSide<T> s0, PostSide<T> s1, int N, int D,
                                                      const float* __restrict__ kappa, float a,
                                                      const float* __restrict__ grad_output, int nparts) {
  constexpr int V = kVec16<T>;
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= N) return;
  const T* x = s0.own + (int64_t)row * s0.ld_own;
  const T* y = s1.own + (int64_t)row * s1.ld_own;
  const int64_t ps = (int64_t)N * D, ro = (int64_t)row * D;
  const float rx = s0.r_own[row], ry = s1.r_own[row], kap = kappa[row];
  const float kx = kap * ry * (ACCR ? rx : 1.f), ky = kap * rx * (ACCR ? ry : 1.f);
  const float go = grad_output ? *grad_output : 1.f;
  float xv[NV][V], yv[NV][V], hx[NV][V], hy[NV][V];
  auto load_acc = [&](const float* p, float (&v)[V]) {
#pragma unroll
    for (int q = 0; q < V / 4; ++q) {
      const f32x4 u = *(const f32x4*)(p + 4 * q);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[4 * q + e] = u[e];
    }
  };
  // (an accumulator may be its side's output: every element is read before the
  // same lane writes it)
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int d = V * (lane + 64 * k);
    if (64 * V * k < D && d < D) {
      load_vec<T>(x + d, xv[k]);
      load_vec<T>(y + d, yv[k]);
      load_acc(s0.acc + ro + d, hx[k]);
      if (BOTH) load_acc(s1.acc + ro + d, hy[k]);
    } else {
#pragma unroll
      for (int e = 0; e < V; ++e) xv[k][e] = yv[k][e] = hx[k][e] = hy[k][e] = 0.f;
    }
  }
  for (int p = 0; p + 1 < nparts; ++p) {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int d = V * (lane + 64 * k);
      if (64 * V * k < D && d < D) {
        float u[V], w[V];
        load_acc(s0.part + p * ps + ro + d, u);
        if (BOTH) load_acc(s1.part + p * ps + ro + d, w);
#pragma unroll
        for (int e = 0; e < V; ++e) {
          hx[k][e] += u[e];
          if (BOTH) hy[k][e] += w[e];
        }
      }
    }
  }
  float dx = 0.f, dy = 0.f;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
#pragma unroll
    for (int e = 0; e < V; ++e) {
      hx[k][e] = a * fmaf(kx, yv[k][e], hx[k][e]);
      if (BOTH) hy[k][e] = a * fmaf(ky, xv[k][e], hy[k][e]);
      if (NORM) {
        xv[k][e] *= rx;
        dx = fmaf(xv[k][e], hx[k][e], dx);
        if (BOTH) {
          yv[k][e] *= ry;
          dy = fmaf(yv[k][e], hy[k][e], dy);
        }
      }
    }
  }
  if (NORM) {
    dx = wave_sum(dx);
    if (BOTH) dy = wave_sum(dy);
  }
  const bool cx = rx >= 1e12f, cy = ry >= 1e12f;
#pragma unroll
  for (int k = 0; k < NV; ++k) {
    const int d = V * (lane + 64 * k);
    if (64 * V * k < D && d < D) {
      float u[V], w[V];
#pragma unroll
      for (int e = 0; e < V; ++e) {
        u[e] = NORM && !cx ? hx[k][e] - xv[k][e] * dx : hx[k][e];
        // (grad_output last, as k_postpass)
        u[e] = NORM && !ACCR ? go * (rx * u[e]) : go * u[e];
        if (BOTH) {
          w[e] = NORM && !cy ? hy[k][e] - yv[k][e] * dy : hy[k][e];
          w[e] = NORM && !ACCR ? go * (ry * w[e]) : go * w[e];
        }
      }
      store_vec<T>(s0.out + ro + d, u);
      if (BOTH) store_vec<T>(s1.out + ro + d, w);
    }
  }
}

// One feature matrix to transpose: X (row pitch ldx), its row scales and the
// destination plane(s) (pitch ldt).  The transposes of the two sides share
// one launch: blockIdx.z picks the side.
template <typename T, typename TO = T>
struct TransSide {
  const T* X;
  int64_t ldx;
  const float* scale;
  TO* XT;
  TO* XTl;  // k_transpose_split with LO: the lo plane
};

// Transposed, normalised copy of one feature matrix for the backward's
// contractions: XT[d, i] = scale_i * X[i, d] (scale = 1/max(||x_i||, 1e-12)
// when NORM) for i < N and 0 for N <= i < ldt, rounded to T once.  64 features x
// 128 rows through LDS.  VEC (16-byte aligned rows, D a multiple of 8): 16-byte
// loads, 8 features per lane; the stores are 16-byte either way (8 rows i per
// lane, 256 contiguous bytes per feature).  HBM-bound.
// LDS: [i][d] with an odd pitch in 4-byte words: the 16 row groups of a
// feature's gather fall on 8 banks, two lanes each.
template <typename T, bool NORM, bool VEC>
__global__ __launch_bounds__(256) void k_transpose(TransSide<T> s0, TransSide<T> s1, int N, int D, int64_t ldt) {
  const TransSide<T>& sd = blockIdx.z ? s1 : s0;
  const T* __restrict__ X = sd.X;
  const int64_t ldx = sd.ldx;
  const float* __restrict__ scale = sd.scale;
  T* __restrict__ XT = sd.XT;
  static_assert(sizeof(T) == 2, "16-bit types");
  constexpr int TI = 128, TD = 64, P = TD + 2;
  __shared__ __attribute__((aligned(16))) uint16_t tile[TI * P];
  const int i0 = blockIdx.x * TI, d0 = blockIdx.y * TD;
  if constexpr (VEC) {
#pragma unroll
    for (int u = 0; u < TI * TD / 8 / 256; ++u) {
      const int v = threadIdx.x + 256 * u, r = v >> 3, c = (v & 7) * 8;
      const int i = i0 + r, d = d0 + c;
      float f[8];
      if (i < N && d < D) {
        load_vec<T>(X + (int64_t)i * ldx + d, f);
        if (NORM) {
          const float s = scale[i];
#pragma unroll
          for (int e = 0; e < 8; ++e) f[e] *= s;
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = 0.f;
      }
      uint32_t* o = (uint32_t*)&tile[r * P + c];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        o[e] = std::is_same<T, uint16_t>::value ? pack2_bf16(f[2 * e], f[2 * e + 1]) : pack2_f16(f[2 * e], f[2 * e + 1]);
    }
  } else {
    for (int r = threadIdx.x >> 6; r < TI; r += 4) {
      const int c = threadIdx.x & 63, i = i0 + r, d = d0 + c;
      float v = 0.f;
      if (i < N && d < D) {
        v = Elem<T>::load(X, (int64_t)i * ldx + d);
        if (NORM) v *= scale[i];
      }
      T t;
      Elem<T>::store(&t, 0, v);
      tile[r * P + c] = __builtin_bit_cast(uint16_t, t);
    }
  }
  __syncthreads();
  typedef uint16_t u16x8 __attribute__((ext_vector_type(8)));
#pragma unroll
  for (int u = 0; u < TI * TD / 8 / 256; ++u) {
    const int v = threadIdx.x + 256 * u, g = v & 15, c = v >> 4;
    const int d = d0 + c;
    if (d >= D) break;
    u16x8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = tile[(8 * g + e) * P + c];
    *(u16x8*)(XT + (int64_t)d * ldt + i0 + 8 * g) = o;
  }
}

// ------------------------------------------------- three-term bf16 split
// fp32 as the sum of two bf16 terms: hi = bf16(v), lo = bf16(v - hi), both
// rounded to nearest even (v - hi is exact in fp32), so v = hi + lo + r with
// |r| <= 2^-16 |v| (bf16 keeps 8 significant bits).  The bf16x3 mode forms
// every product a*b of the hot loops as hi_a*hi_b + lo_a*hi_b + hi_a*lo_b on
// the bf16 MFMA (fp32 accumulate); the dropped lo_a*lo_b and the two
// remainders bound the error of one product by about 3 * 2^-16 |ab|.
__device__ __forceinline__ void split2_bf16(float a, float b, uint32_t& hi, uint32_t& lo) {
  const uint16_t ha = f32_to_bf16(a), hb = f32_to_bf16(b);
  hi = (uint32_t)ha | ((uint32_t)hb << 16);
  lo = pack2_bf16(a - bf16_to_f32(ha), b - bf16_to_f32(hb));
}

// Split copies of the inputs for the similarity GEMMs of the bf16x3 mode.
// Row i of out (pitch ld3 elements) holds three segments of dp = D rounded up
// to 8 elements: ORDER 0 (x side) hi, lo, hi; ORDER 1 (y side) hi, hi, lo.
// The dot product of an x row with a y row over the 3 dp elements is then
// hi.hi + lo.hi + hi.lo, one bf16 GEMM with K = 3 dp.  Columns D .. dp-1 of
// each segment are zero.  NORM: the rows are normalized first (x_i rx_i in
// fp32, rx from the pre-pass), so that the GEMM kernels need no norm scaling.
// One thread per 8 columns; out and ld3 16-byte aligned.
template <int ORDER, bool NORM>
__global__ __launch_bounds__(256) void k_split3(const float* __restrict__ X, int64_t ldx, int N, int D, int dp,
                                                uint16_t* __restrict__ out, int64_t ld3,
                                                const float* __restrict__ rxv) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  const int vpr = dp / 8;
  const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (v >= (int64_t)N * vpr) return;
  const int i = (int)(v / vpr), d0 = (int)(v - (int64_t)i * vpr) * 8;
  const float* x = X + (int64_t)i * ldx;
  const float r = NORM ? rxv[i] : 1.f;
  u32x4 hi, lo;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int d = d0 + 2 * e;
    const float a = d < D ? x[d] * r : 0.f, b = d + 1 < D ? x[d + 1] * r : 0.f;
    uint32_t h, l;
    split2_bf16(a, b, h, l);
    hi[e] = h;
    lo[e] = l;
  }
  uint16_t* o = out + (int64_t)i * ld3 + d0;
  *(u32x4*)o = hi;
  *(u32x4*)(o + dp) = ORDER == 0 ? lo : hi;
  *(u32x4*)(o + 2 * dp) = ORDER == 0 ? hi : lo;
}

// bf16 copies of the inputs for the fp32-data / bf16-product mode: row i of
// out (pitch ldo) is bf16(x_i) (NORM: bf16(x_i rx_i)), round to nearest
// even, zero-padded to dp columns.  One thread per 8 columns; out and ldo
// 16-byte aligned.
template <bool NORM>
__global__ __launch_bounds__(256) void k_split1(const float* __restrict__ X, int64_t ldx, int N, int D, int dp,
                                                uint16_t* __restrict__ out, int64_t ldo,
                                                const float* __restrict__ rxv) {
  typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
  const int vpr = dp / 8;
  const int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (v >= (int64_t)N * vpr) return;
  const int i = (int)(v / vpr), d0 = (int)(v - (int64_t)i * vpr) * 8;
  const float* x = X + (int64_t)i * ldx;
  const float r = NORM ? rxv[i] : 1.f;
  u32x4 hi;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int d = d0 + 2 * e;
    hi[e] = pack2_bf16(d < D ? x[d] * r : 0.f, d + 1 < D ? x[d + 1] * r : 0.f);
  }
  *(u32x4*)(out + (int64_t)i * ldo + d0) = hi;
}

// k_transpose<float, NORM> into bf16 planes: XT_hi[d][i] = hi(v) and, when
// LO, XT_lo[d][i] = lo(v), with v = scale_i x_i[d] (fp32), zero for
// N <= i < ldt.
template <bool NORM, bool LO>
__global__ __launch_bounds__(256) void k_transpose_split(TransSide<float, uint16_t> s0,
                                                         TransSide<float, uint16_t> s1, int N, int D, int64_t ldt) {
  const TransSide<float, uint16_t>& sd = blockIdx.z ? s1 : s0;
  const float* __restrict__ X = sd.X;
  const int64_t ldx = sd.ldx;
  const float* __restrict__ scale = sd.scale;
  uint16_t* __restrict__ XTh = sd.XT;
  uint16_t* __restrict__ XTl = sd.XTl;
  __shared__ float tile[64][65];
  const int i0 = blockIdx.x * 64, d0 = blockIdx.y * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int r = ty; r < 64; r += 4) {
    const int i = i0 + r, d = d0 + tx;
    float v = 0.f;
    if (i < N && d < D) {
      v = X[(int64_t)i * ldx + d];
      if (NORM) v *= scale[i];
    }
    tile[r][tx] = v;
  }
  __syncthreads();
  for (int r = ty; r < 64; r += 4) {
    const int d = d0 + r, i = i0 + tx;
    if (d < D && i < ldt) {
      const float v = tile[tx][r];
      const uint16_t h = f32_to_bf16(v);
      XTh[(int64_t)d * ldt + i] = h;
      if (LO) XTl[(int64_t)d * ldt + i] = f32_to_bf16(v - bf16_to_f32(h));
    }
  }
}

// ------------------------------------------------------- fp16 split pairs
// fp32 as the sum of two fp16 terms, v = hi + lo + r with hi = fp16(v), lo =
// fp16(v - hi), both rounded to nearest even: |r| <= 2^-23 |v| while lo is a
// normal number, and never more than 2^-25 (half of fp16's smallest step).  The
// values are first scaled by a power of two that puts the largest one into
// [2^14, 2^15), so the second bound is 2^-39 of the largest value: what is lost
// below it is far smaller than the rounding of an fp32 sum.  The products hi hi
// + lo hi + hi lo leave out lo lo, at most 2^-22 of a product and of either
// sign.
__device__ __forceinline__ void split_pair4(const f32x4& v, uint2& hi, uint2& lo) {
  float h[4], l[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    h[e] = (float)(_Float16)v[e];
    // (an infinite value stays hi = inf, lo = 0)
    l[e] = __builtin_isinf(h[e]) ? 0.f : v[e] - h[e];
  }
  hi = uint2{pack2_f16(h[0], h[1]), pack2_f16(h[2], h[3])};
  lo = uint2{pack2_f16(l[0], l[1]), pack2_f16(l[2], l[3])};
}
// the power of two that puts m (the largest finite magnitude) into [2^14,
// 2^15), at most 2^126 (2^-113 at the least: m < 2^128); 1 for 0.  It and its
// inverse are normal numbers; a product of two need not be one (exp_mul,
// contract_store_again).
__device__ __forceinline__ float pair_scale(float m) {
  if (!(m > 0.f)) return 1.f;
  int s = 14 - ((int)(__float_as_uint(m) >> 23) - 127);
  s = s > 126 ? 126 : s;
  return __uint_as_float((uint32_t)(s + 127) << 23);
}
constexpr float PAIR_UNIT_SCALE = 16384.f;  // of rows that are normalized here (|v| <= 1)

// features d .. d + 3 of a row, zero from D on (vec: 16-byte aligned rows)
__device__ __forceinline__ f32x4 row_load4(const float* __restrict__ p, int d, int D, bool vec) {
  if (vec && d + 3 < D) return *(const f32x4*)(p + d);
  f32x4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = d + e < D ? p[d + e] : 0.f;
  return v;
}
// v (features d .. d + 3) into a row of pairs: every 32 features as 32 hi and
// then 32 lo values
__device__ __forceinline__ void pair_store4(uint16_t* __restrict__ out, int d, const f32x4& v) {
  uint2 hi, lo;
  split_pair4(v, hi, lo);
  uint16_t* o = out + (d >> 5) * 64 + (d & 31);
  *(uint2*)o = hi;
  *(uint2*)(o + 32) = lo;
}

struct PairRows {
  uint16_t* a;     // x rows as pairs, pitch 2 dp (dp = D rounded up to 32, zeros past D)
  uint16_t* b;     // y rows
  float* scl;      // the scales (SCL_X ..)
  int dp;
};

// Pre-pass of the split pairs, one wave per row: k_prepass's norms and
// diagonal.  NORM: also the pairs of x_i rx_i and y_i ry_i (one launch instead
// of a pre-pass and a split per side: rows of up to PAIR_REG x 256 features
// stay in registers between the reduction and the stores).  Otherwise the rows
// are split as they are, once the largest finite magnitude of each side is
// known: this launch leaves each workgroup's in the slots 1/R and 1/C (which
// the finalize fills later) for k_pair_rows.
constexpr int PAIR_REG = 8;
template <bool NORM>
__global__ __launch_bounds__(256) void k_pair_prepass(const float* __restrict__ X, int64_t ldx,
                                                      const float* __restrict__ Y, int64_t ldy, int N, int D, bool vec,
                                                      float* __restrict__ ws, PairRows pr,
                                                      uint32_t* __restrict__ counter) {
  __shared__ float s_mx[2][4];
  if (counter && blockIdx.x == 0 && threadIdx.x == 0) *counter = 0u;  // (k_finalize_all)
  if (blockIdx.x == 0 && threadIdx.x == 0) {  // (pair_grad_range)
    pr.scl[SCL_KMAX] = 0.f;
    pr.scl[SCL_SMIN] = __builtin_inff();
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int row = blockIdx.x * 4 + w;
  const int64_t n = N;
  float mx = 0.f, my = 0.f;
  if (row < N) {
    const float* x = X + (int64_t)row * ldx;
    const float* y = Y + (int64_t)row * ldy;
    f32x4 xv[PAIR_REG], yv[PAIR_REG];
    float sx = 0.f, sy = 0.f, sxy = 0.f;
    auto add = [&](const f32x4& a, const f32x4& b) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        sx = fmaf(a[e], a[e], sx);
        sy = fmaf(b[e], b[e], sy);
        sxy = fmaf(a[e], b[e], sxy);
        if (!NORM) {
          const float p = fabsf(a[e]), q = fabsf(b[e]);
          mx = p < __builtin_inff() ? fmaxf(mx, p) : mx;
          my = q < __builtin_inff() ? fmaxf(my, q) : my;
        }
      }
    };
    const bool inreg = pr.dp <= PAIR_REG * 256;
    if (inreg) {
#pragma unroll
      for (int k = 0; k < PAIR_REG; ++k) {
        const int d = 4 * lane + 256 * k;
        if (256 * k < D) {
          xv[k] = row_load4(x, d, D, vec);
          yv[k] = row_load4(y, d, D, vec);
        }
      }
#pragma unroll
      for (int k = 0; k < PAIR_REG; ++k)
        if (256 * k < D) add(xv[k], yv[k]);
    } else {
      for (int d = 4 * lane; d < D; d += 256) add(row_load4(x, d, D, vec), row_load4(y, d, D, vec));
    }
    sx = wave_sum(sx);
    sy = wave_sum(sy);
    sxy = wave_sum(sxy);
    float rx = 1.f, ry = 1.f;
    if (NORM) {
      rx = 1.f / fmaxf(sqrtf(sx), 1e-12f);
      ry = 1.f / fmaxf(sqrtf(sy), 1e-12f);
    }
    if (lane == 0) {
      ws[WS_RX * n + row] = rx;
      ws[WS_RY * n + row] = ry;
      ws[WS_DIAG * n + row] = sxy;
      ws[WS_ROW_OFF * n + row] = 0.f;
      ws[WS_COL_OFF * n + row] = 0.f;
    }
    if constexpr (NORM) {
      uint16_t* oa = pr.a + (int64_t)row * (2 * pr.dp);
      uint16_t* ob = pr.b + (int64_t)row * (2 * pr.dp);
      // (the power of two is exact: as x_i rx_i scaled)
      if (inreg) {
#pragma unroll
        for (int k = 0; k < PAIR_REG; ++k) {
          const int d = 4 * lane + 256 * k;
          if (d < pr.dp) {
            pair_store4(oa, d, xv[k] * rx * PAIR_UNIT_SCALE);
            pair_store4(ob, d, yv[k] * ry * PAIR_UNIT_SCALE);
          }
        }
      } else {
        for (int d = 4 * lane; d < pr.dp; d += 256) {
          pair_store4(oa, d, row_load4(x, d, D, vec) * rx * PAIR_UNIT_SCALE);
          pair_store4(ob, d, row_load4(y, d, D, vec) * ry * PAIR_UNIT_SCALE);
        }
      }
    }
  }
  if constexpr (NORM) {
    if (blockIdx.x == 0 && threadIdx.x < 4) pr.scl[threadIdx.x] = threadIdx.x < 2 ? PAIR_UNIT_SCALE : 1.f / PAIR_UNIT_SCALE;
  } else {
    for (int m = 32; m >= 1; m >>= 1) {
      mx = fmaxf(mx, __shfl_xor(mx, m, 64));
      my = fmaxf(my, __shfl_xor(my, m, 64));
    }
    if (lane == 0) {
      s_mx[0][w] = mx;
      s_mx[1][w] = my;
    }
    __syncthreads();
    if (threadIdx.x < 2) {
      const float* s = s_mx[threadIdx.x];
      ws[(threadIdx.x ? WS_INV_COL : WS_INV_ROW) * n + blockIdx.x] = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
    }
  }
}

// Pairs of rows that come normalized (k_pair_prepass<false> ran before): every
// workgroup takes the largest magnitudes from the nmax = ceil(N / 4) it left
// per side, and its share of the rows, one wave per row.
__global__ __launch_bounds__(256) void k_pair_rows(const float* __restrict__ X, int64_t ldx,
                                                   const float* __restrict__ Y, int64_t ldy, int N, int D, bool vec,
                                                   const float* __restrict__ ws, PairRows pr, int nmax) {
  __shared__ float s_mx[2][4];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t n = N;
  float mx = 0.f, my = 0.f;
  for (int k = threadIdx.x; k < nmax; k += 256) {
    mx = fmaxf(mx, ws[WS_INV_ROW * n + k]);
    my = fmaxf(my, ws[WS_INV_COL * n + k]);
  }
  for (int m = 32; m >= 1; m >>= 1) {
    mx = fmaxf(mx, __shfl_xor(mx, m, 64));
    my = fmaxf(my, __shfl_xor(my, m, 64));
  }
  if (lane == 0) {
    s_mx[0][w] = mx;
    s_mx[1][w] = my;
  }
  __syncthreads();
  const float sx = pair_scale(fmaxf(fmaxf(s_mx[0][0], s_mx[0][1]), fmaxf(s_mx[0][2], s_mx[0][3])));
  const float sy = pair_scale(fmaxf(fmaxf(s_mx[1][0], s_mx[1][1]), fmaxf(s_mx[1][2], s_mx[1][3])));
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    pr.scl[0] = sx;
    pr.scl[1] = sy;
    pr.scl[2] = 1.f / sx;
    pr.scl[3] = 1.f / sy;
  }
  for (int row = blockIdx.x * 4 + w; row < N; row += gridDim.x * 4) {
    const float* x = X + (int64_t)row * ldx;
    const float* y = Y + (int64_t)row * ldy;
    for (int d = 4 * lane; d < pr.dp; d += 256) {
      pair_store4(pr.a + (int64_t)row * (2 * pr.dp), d, row_load4(x, d, D, vec) * sx);
      pair_store4(pr.b + (int64_t)row * (2 * pr.dp), d, row_load4(y, d, D, vec) * sy);
    }
  }
}

// pair_grad_range of the rows' sums for a forward run stage by stage
// (mec_sumexp; mec_forward's finalize does it on the way): one thread per row.
template <bool LIT>
__global__ __launch_bounds__(256) void k_pair_range(int N, double inv_t, const float* __restrict__ ws,
                                                    float* __restrict__ scl) {
  const int64_t n = N;
  const int i = blockIdx.x * 256 + threadIdx.x;
  float k = 0.f, s = __builtin_inff();
  if (i < N) {
    const double e = exp(((double)ws[WS_DIAG * n + i] * (double)ws[WS_RX * n + i] * (double)ws[WS_RY * n + i] - 1.0) *
                         inv_t);
    const double ro = ws[WS_ROW_OFF * n + i], co = LIT ? 0.0 : (double)ws[WS_COL_OFF * n + i];
    k = (float)(ro / (ro + e)) + (LIT ? 0.f : (float)(co / (co + e)));
    s = least_share<LIT>(ro, ro + e, co, co + e);
  }
  pair_grad_range<4>(k, s, scl);
}

// k_transpose_split into pairs: row d of XT (pitch 2 ldt) holds, for every 32
// rows i, 32 hi and then 32 lo values of scale_i x_i[d] (NORM) times the side's
// pair scale, zero for N <= i < ldt (ldt a multiple of 64).  Two values of i
// per thread: 4-byte stores, 64 contiguous bytes per part.  Where the gradient
// matrix is held wide: the values themselves, fp32, row d of pitch ldt.  The
// first workgroup leaves the gradient matrix's scale in gscl (GradBufs).
template <bool NORM>
__global__ __launch_bounds__(256) void k_transpose_pairs(TransSide<float, uint16_t> s0, TransSide<float, uint16_t> s1,
                                                         int N, int D, int64_t ldt, const float* scl0,
                                                         const float* scl1, const float* __restrict__ scl,
                                                         float* gscl) {
  const TransSide<float, uint16_t>& sd = blockIdx.z ? s1 : s0;
  const float ps = blockIdx.z ? *scl1 : *scl0;
  const float* __restrict__ X = sd.X;
  const int64_t ldx = sd.ldx;
  const float* __restrict__ scale = sd.scale;
  uint16_t* __restrict__ XT = sd.XT;
  __shared__ float tile[64][65];
  const int i0 = blockIdx.x * 64, d0 = blockIdx.y * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int r = ty; r < 64; r += 4) {
    const int i = i0 + r, d = d0 + tx;
    float v = 0.f;
    if (i < N && d < D) {
      v = X[(int64_t)i * ldx + d];
      if (NORM) v *= scale[i];
      v *= ps;
    }
    tile[r][tx] = v;
  }
  const PairGrad pg = pair_grad_scale(N, scl);
  if (blockIdx.x + blockIdx.y + blockIdx.z + threadIdx.x == 0) {
    gscl[0] = pg.scale;
    gscl[1] = pg.inv;
    gscl[2] = pg.wide ? 1.f : 0.f;
  }
  __syncthreads();
  if (pg.wide) {
    float* __restrict__ XW = (float*)XT;
    for (int r = ty; r < 64 && d0 + r < D; r += 4) XW[(int64_t)(d0 + r) * ldt + i0 + tx] = tile[tx][r];
    return;
  }
  const int il = 2 * (threadIdx.x & 31);
  for (int r = threadIdx.x >> 5; r < 64; r += 8) {
    const int d = d0 + r;
    if (d >= D) break;
    const float a = tile[il][r], b = tile[il + 1][r];
    const float ha = (float)(_Float16)a, hb = (float)(_Float16)b;
    uint16_t* o = XT + (int64_t)d * (2 * ldt) + (int64_t)(i0 + (il & 32)) * 2 + (il & 31);
    *(uint32_t*)o = pack2_f16(ha, hb);
    *(uint32_t*)(o + 32) = pack2_f16(__builtin_isinf(ha) ? 0.f : a - ha, __builtin_isinf(hb) ? 0.f : b - hb);
  }
}

}  // namespace mec
