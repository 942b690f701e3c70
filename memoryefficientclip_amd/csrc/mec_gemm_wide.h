// Contractions of fp32 operands as three bf16 terms each, for the gradient
// matrices whose range fp16 pairs do not hold (pair_grad_scale): v = hi + mid +
// lo, every term rounded to bf16's 8 bits, 24 bits or more at fp32's range of
// exponents.  A product is the six of the nine terms' products down to 2^-18,
// lo hi + hi lo + mid mid + mid hi + hi mid + hi hi, smallest first; the three
// left out are below 2^-25 of it.  The six products of 16 k are summed in
// registers of their own before they are added to the tile's sums, which are so
// rounded once per 16 k (the fp32 MFMA: once per 2 k).
//
// Both operands are fp32 in the scratch (no more bytes than the pairs) and go
// through registers: a chunk of 32 k is loaded while the one before it is
// multiplied, split, and written to LDS as six planes of K-major rows.  Bound by
// the MFMA (12 per 32 x 32 block and chunk, against the pairs' 6) and the split
// (about 10 VALU operations a value), one after the other between barriers.
// CLIP step with wide contractions (one swapped pair at T = 0.02), pairs -> wide,
// and on the fp32 kernels: 4999 x 640 371 -> 641 us, 1154; 8192 x 768 951 -> 1892
// us, 3021; 32768 x 1152 21.2 -> 42.7 ms, 70.5.  At d = 64 they take longer than
// the fp32 kernels (8192 x 64 504 us, 437): three quarters of a tile are columns
// past d.
#pragma once
#include "mec_common.h"

namespace mec {
namespace gwide {

// B x B output tile: 256 (8 waves of 64 x 128) or 128 (4 waves of 64 x 64)
template <int B>
struct Tile {
  static_assert(B == 256 || B == 128, "the tile sizes of the pair contractions");
  static constexpr int BM = B, BN = B, WM = B / 64, WN = 2, TM = 64, TN = B / 2, FM = 2, FN = TN / 32;
  static constexpr int NT = 64 * WM * WN;
  static constexpr int KC = 32;               // k per chunk
  // bytes per staged row: 32 bf16, and 16 apart (16-byte reads of consecutive
  // rows then start 5 bank groups apart)
  static constexpr int PITCH = 80;
  static constexpr int PLANE = B * PITCH;
  static constexpr int LDS_BYTES = 6 * PLANE;  // A's hi, mid, lo, then B's
};

// One operand: a buffer of `klen` (a multiple of 32) k and up to TL::BM rows, and
// this thread's 4 rows x 4 k of its chunks.  km: K-major (row r at p + r ld, k
// contiguous), else k-row-major (k at p + k ld, rows contiguous).  Rows from
// `rows` on read as 0 (K-major; they end in output that is not stored).  Offsets
// stay below 2^31 bytes: (255 ld + klen) x 4 with ld <= 2^20, or klen x ld x 4
// within a block.
template <class TL>
struct Source {
  __amdgpu_buffer_rsrc_t r;
  bool km;
  uint32_t estep, kstep;  // byte steps of a load's element (row, k) and of k (k-row-major: both the k-row)
  __device__ __forceinline__ Source(bool km_, const float* p, int64_t ld, int rows, int klen) : km(km_) {
    const int64_t n = km ? (rows - 1) * ld + klen : (klen - 1) * ld + TL::BM;
    r = __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)(n * 4), 0x00020000);
    estep = (uint32_t)ld * 4;
    kstep = km ? 4 : estep;
  }
  __device__ __forceinline__ void load(int k, f32x4 (&v)[4]) const {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    uint32_t t = threadIdx.x;
    asm volatile("" : "+v"(t));  // (the addresses are formed here: kept across the loop they spill)
    const uint32_t vo = km ? (t >> 3) * 4 * estep + (t & 7) * 16 : t / (TL::BM / 4) * 4 * estep + t % (TL::BM / 4) * 16;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const u32x4 u = __builtin_amdgcn_raw_buffer_load_b128(r, vo, k * kstep + e * estep, 0);
      v[e] = __builtin_bit_cast(f32x4, u);
    }
  }
};

// 4 consecutive k of one row as three bf16 terms, a plane apart
template <class TL>
__device__ __forceinline__ void split4(float f0, float f1, float f2, float f3, char* o) {
#pragma unroll
  for (int pl = 0; pl < 3; ++pl) {
    const uint2 u = uint2{pack2_bf16(f0, f1), pack2_bf16(f2, f3)};
    *(uint2*)(o + pl * TL::PLANE) = u;
    f0 -= __uint_as_float(u.x << 16);
    f1 -= __uint_as_float(u.x & 0xffff0000u);
    f2 -= __uint_as_float(u.y << 16);
    f3 -= __uint_as_float(u.y & 0xffff0000u);
  }
}
// A chunk as three planes of K-major rows at `lds`
template <class TL>
__device__ __forceinline__ void split_store(bool km, const f32x4 (&v)[4], char* lds) {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));  // (as in Source::load)
  if (km) {
    char* o = lds + (t >> 3) * 4 * TL::PITCH + 8 * (t & 7);
#pragma unroll
    for (int e = 0; e < 4; ++e) split4<TL>(v[e][0], v[e][1], v[e][2], v[e][3], o + e * TL::PITCH);
  } else {
    char* o = lds + t % (TL::BM / 4) * 4 * TL::PITCH + t / (TL::BM / 4) * 8;
#pragma unroll
    for (int e = 0; e < 4; ++e) split4<TL>(v[0][e], v[1][e], v[2][e], v[3][e], o + e * TL::PITCH);
  }
}

// acc = sum over k in [0, klen) (in whole chunks: the operands hold zeros up to
// a multiple of 32) of A[m][k] B[n][k]; the caller's LDS is free on return only
// after a barrier
template <class TL>
__device__ __forceinline__ void run(bool akm, const float* __restrict__ a, int64_t lda, const float* __restrict__ b,
                                    int64_t ldb, int b_rows, int klen, char* lds, f32x16 (&acc)[TL::FM][TL::FN]) {
  klen = (klen + 31) & ~31;
  const Source<TL> sa(akm, a, lda, TL::BM, klen), sb(true, b, ldb, b_rows, klen);
#pragma unroll
  for (int i = 0; i < TL::FM; ++i)
#pragma unroll
    for (int j = 0; j < TL::FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  f32x4 va[4], vb[4];
  sa.load(0, va);
  sb.load(0, vb);
  for (int k = 0; k < klen; k += TL::KC) {
    __syncthreads();  // every wave is done with the chunk before
    split_store<TL>(akm, va, lds);
    split_store<TL>(true, vb, lds + 3 * TL::PLANE);
    if (k + TL::KC < klen) {
      sa.load(k + TL::KC, va);
      sb.load(k + TL::KC, vb);
    }
    __syncthreads();
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));  // (as in Source::load)
    const int lane = t & 63, w = t >> 6, wm = w / TL::WN, wn = w % TL::WN;
    // (a wave whose columns hold no row of B leaves its sums at 0)
    if (__builtin_amdgcn_readfirstlane(b_rows - wn * TL::TN) <= 0) continue;
    const char* ra = lds + (wm * TL::TM + (lane & 31)) * TL::PITCH + 16 * (lane >> 5);
    const char* rb = lds + 3 * TL::PLANE + (wn * TL::TN + (lane & 31)) * TL::PITCH + 16 * (lane >> 5);
#pragma unroll
    for (int s = 0; s < TL::KC / 16; ++s) {
      i16x8 fa[TL::FM][3];
#pragma unroll
      for (int i = 0; i < TL::FM; ++i)
#pragma unroll
        for (int pl = 0; pl < 3; ++pl)
          fa[i][pl] = *(const i16x8*)(ra + pl * TL::PLANE + i * 32 * TL::PITCH + 32 * s);
#pragma unroll
      for (int j = 0; j < TL::FN; ++j) {
        i16x8 fb[3];
#pragma unroll
        for (int pl = 0; pl < 3; ++pl) fb[pl] = *(const i16x8*)(rb + pl * TL::PLANE + j * 32 * TL::PITCH + 32 * s);
        constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
        for (int i = 0; i < TL::FM; ++i) {
          f32x16 u;
#pragma unroll
          for (int r = 0; r < 16; ++r) u[r] = 0.f;
#pragma unroll
          for (int q = 0; q < 6; ++q) u = mfma16_32x32x16<false>(fa[i][PA[q]], fb[PB[q]], u);
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[i][j][r] += u[r];
        }
        // (the next block's reads stay behind: with all of them ahead the
        // registers do not last)
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
}

}  // namespace gwide
}  // namespace mec
