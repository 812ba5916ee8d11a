// BF16x3 product tiles: a work-group's 64 x 64 tile of op(A) op(B) from FP32 operands, each split
// into bf16 hi + lo (hi = RNE(x), lo = RNE(x - hi)) on its way into LDS; per 32 of K each
// accumulator takes lo hi, hi lo, hi hi on v_mfma_f32_16x16x32_bf16 (the dropped lo lo term leaves
// ~2^-16 relative error per product).
//
// K advances in stages of 64: the next stage's loads are in flight during the products of the current one.
// BUFS = 2 stages in LDS let its conversion meet one barrier per stage; with BUFS = 1 twice as many
// work-groups fit on a CU (four of 37 KB), the better use where there are as many. Every thread converts 8
// consecutive k of one row at a time, so both parts go to LDS as 16-byte writes whatever the
// operand's order in memory (k-contiguous rows by two float4, k-strided columns by 8 coalesced
// dwords); rows of 72 bf16 (36 banks) keep the 16-byte reads and writes of 16 lanes apart.
#pragma once
#include "pib_common.hpp"

namespace pib {

typedef float f32x4t __attribute__((ext_vector_type(4)));
typedef float f32x2t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2t __attribute__((ext_vector_type(2)));
typedef unsigned u32x4t __attribute__((ext_vector_type(4)));

constexpr int kTile3 = 64, kStage3 = 64, kRow3 = kStage3 + 8;

struct Stage3 {  // one stage of both operands
  unsigned short Ah[kTile3][kRow3], Al[kTile3][kRow3], Bh[kTile3][kRow3], Bl[kTile3][kRow3];
};

// A thread's 16 values of a stage: two runs of 8 consecutive k.
// KS (k strided): p = the thread's column (t % 64) at k = 0; else p = its row (t / 8) at k = 0, its
// second run 32 rows on. Past kend (a last stage of 32) the last run again: no product takes it.
template <bool KS>
__device__ __forceinline__ void load3(const float* __restrict__ p, int64_t ld, int64_t k0, int64_t kend, int t,
                                      float (&v)[2][8]) {
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    if constexpr (KS) {
      const int64_t k = min(k0 + 8 * (__builtin_amdgcn_readfirstlane(t >> 6) + 4 * c), kend - 8);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[c][e] = p[(k + e) * ld];
    } else {
      const int64_t k = min(k0 + 8 * (t & 7), kend - 8);
      const float* q = p + c * 32 * ld + k;
      const f32x4t a = *(const f32x4t*)q, b = *(const f32x4t*)(q + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[c][e] = a[e];
        v[c][4 + e] = b[e];
      }
    }
  }
}

// 8 floats to packed bf16 hi and lo
__device__ __forceinline__ void split8(const float (&v)[8], u32x4t& h, u32x4t& l) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float x = v[2 * e], y = v[2 * e + 1];
    const unsigned u = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2t{x, y}, bf16x2t));
    const float xl = x - __uint_as_float(u << 16), yl = y - __uint_as_float(u & 0xffff0000u);
    h[e] = u;
    l[e] = __builtin_bit_cast(unsigned, __builtin_convertvector(f32x2t{xl, yl}, bf16x2t));
  }
}

template <bool KS>
__device__ __forceinline__ void store3(unsigned short (*H)[kRow3], unsigned short (*L)[kRow3], int t,
                                       const float (&v)[2][8]) {
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    u32x4t h, l;
    split8(v[c], h, l);
    const int row = KS ? (t & 63) : (t >> 3) + 32 * c, k = 8 * (KS ? (t >> 6) + 4 * c : (t & 7));
    *(u32x4t*)&H[row][k] = h;
    *(u32x4t*)&L[row][k] = l;
  }
}

// The products of one stage: wave w holds the 32 x 32 sub-tile (w / 2, w % 2) as 2 x 2
// blocks; element r of acc[i][j] is row 32 (w / 2) + 16 i + 4 (lane / 16) + r, column
// 32 (w % 2) + 16 j + lane % 16.
__device__ __forceinline__ void products3(const Stage3& s, int t, int slabs, f32x4t (&acc)[2][2]) {
  const int lane = t & 63, wr = (t >> 7) & 1, wc = (t >> 6) & 1;
#pragma unroll
  for (int sl = 0; sl < 2; ++sl) {
    if (sl >= slabs) break;  // uniform
    const int k = 32 * sl + 8 * (lane >> 4);
    bf16x8t ah[2], al[2], bh[2], bl[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int r = wr * 32 + i * 16 + (lane & 15), c = wc * 32 + i * 16 + (lane & 15);
      ah[i] = __builtin_bit_cast(bf16x8t, *(const u32x4t*)&s.Ah[r][k]);
      al[i] = __builtin_bit_cast(bf16x8t, *(const u32x4t*)&s.Al[r][k]);
      bh[i] = __builtin_bit_cast(bf16x8t, *(const u32x4t*)&s.Bh[c][k]);
      bl[i] = __builtin_bit_cast(bf16x8t, *(const u32x4t*)&s.Bl[c][k]);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[i], bh[j], acc[i][j], 0, 0, 0);
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bl[j], acc[i][j], 0, 0, 0);
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bh[j], acc[i][j], 0, 0, 0);
      }
  }
}

// A tile's sum over [kbeg, kend), a multiple of 32. KSA / KSB: the operand is strided in k; pa / pb:
// the thread's column or row (see load3).
template <bool KSA, bool KSB, int BUFS>
__device__ __forceinline__ void tile3(const float* __restrict__ pa, int64_t lda, const float* __restrict__ pb,
                                      int64_t ldb, int64_t kbeg, int64_t kend, int t, Stage3* lds,
                                      f32x4t (&acc)[2][2]) {
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4t{0.f, 0.f, 0.f, 0.f};
  float va[2][8], vb[2][8];
  auto put = [&](Stage3& s) {
    store3<KSA>(s.Ah, s.Al, t, va);
    store3<KSB>(s.Bh, s.Bl, t, vb);
  };
  load3<KSA>(pa, lda, kbeg, kend, t, va);
  load3<KSB>(pb, ldb, kbeg, kend, t, vb);
  put(lds[0]);
  __syncthreads();
  int b = 0;
  for (int64_t k0 = kbeg; k0 < kend; k0 += kStage3) {
    const bool more = k0 + kStage3 < kend;
    if (more) {
      load3<KSA>(pa, lda, k0 + kStage3, kend, t, va);
      load3<KSB>(pb, ldb, k0 + kStage3, kend, t, vb);
    }
    products3(lds[b], t, kend - k0 >= kStage3 ? 2 : 1, acc);
    if (!more) break;  // uniform
    if constexpr (BUFS == 2)
      b ^= 1;
    else
      __syncthreads();  // the stage has been read
    put(lds[b]);
    __syncthreads();
  }
}

}  // namespace pib
