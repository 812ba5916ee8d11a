// Training pass of the learned proposal (BF16x3 products): the inverse flow with everything its
// backward needs, and the gradient of -sum_b c_b log q(R_b) from the gradient of log rho.
//
// Every layer acts on each sample by itself, so a work-group takes 16 samples through all layers in
// one launch, forward or backward: the operands of its products stay in LDS as bf16 hi + lo, the
// weights come from L2 in the matrix instruction's own order (k_train_weights lays them out once per
// pass), 2 KB per 16 outputs and 32 inputs, and no layer waits for a launch or for other samples.
// What bounds it is that stream, 1.8 MB per work-group and layer at D = 1,024, hidden 256: 37 bytes
// per cycle and CU, the same with 64 to 256 KB of it in flight and with 64 or 128 CUs at it (without
// the loads the forward takes 100 of its 174 us, without products and couplings 160). Wider row
// blocks would halve the stream and leave half the chip idle at the few thousand samples of a
// training batch.
// The gradients of weights and biases need all samples and nothing of each other: one launch for
// those of all layers, 128 x 128 tiles (k_weight_grads).
// MI355X, 2,048 samples of D = 1,024, hidden 256, 8 layers: 1.75 ms as 72 products with 40 second
// passes, 24 column sums, couplings and copies; 0.78 as 3 launches per layer and direction with the
// couplings as epilogues (64 x 64 tiles, 8 to 16 us each, 4 of them latency); 0.45 so (weights' order
// 17 us, forward 174, backward 173, gradients 81).
#include <algorithm>

#include "pib_flow.hpp"
#include "pib_gemm3.hpp"

namespace pib {

constexpr int kTrainWaves = 8, kTrainRows = 16;
constexpr size_t kTrainLds = 160 * 1024;

struct TrainDims {
  int H, h, D;
  __host__ __device__ int64_t per_layer() const { return (int64_t)H * h + h + (int64_t)h * h + h + (int64_t)h * D + D; }
  __host__ __device__ int64_t frags() const { return 2 * ((int64_t)H * h + (int64_t)h * h + (int64_t)h * D); }  // shorts
};
struct Net {
  const float *W1, *b1, *W2, *b2, *W3, *b3;
};
__host__ __device__ inline Net net(const TrainDims& d, const float* base, int l) {
  const float* p = base + l * d.per_layer();
  Net n;
  n.W1 = p;
  n.b1 = n.W1 + (int64_t)d.H * d.h;
  n.W2 = n.b1 + d.h;
  n.b2 = n.W2 + (int64_t)d.h * d.h;
  n.W3 = n.b2 + d.h;
  n.b3 = n.W3 + (int64_t)d.h * d.D;
  return n;
}

// The halves of z: a layer changes one half and the next conditions on it, so step t (layer L-1-t)
// writes half t, conditions on half t-1 and transforms half t-2; -1 and -2 are z0's, the last two z1's.
struct Half {
  float* p;
  int64_t ld;
};
__host__ __device__ inline Half half(const TrainArgs& a, int t) {
  const int H = a.D / 2, first_a = (a.L - 1) % 2 ? H : 0;  // conditioning offset of layer L - 1
  if (t == -1) return {a.z0 + first_a, a.D};
  if (t == -2) return {a.z0 + (H - first_a), a.D};
  if (t >= a.L - 2) return {a.z1 + (t == a.L - 1 ? H : 0), a.D};
  return {a.halves + (int64_t)t * a.B * H, H};
}

__device__ __forceinline__ unsigned short bf_hi(float x) { return __builtin_bit_cast(unsigned short, (__bf16)x); }
__device__ __forceinline__ float bf_f(unsigned short h) { return __uint_as_float((unsigned)h << 16); }

// ------------------------------------------------------------------ weights in product order
// Blocks of 16 outputs n and 32 inputs k of a product's B operand: lane l's 8 elements
// B[k0 + 8 (l / 16) + e][n0 + l % 16], hi of all lanes, then lo; blocks of one n consecutive in k.
// FORWARD B = W (inputs x outputs), else B = W^T. One wave per block.
__global__ void __launch_bounds__(256) k_train_weights(TrainDims d, const float* params, int64_t blocks,
                                                       unsigned short* fwd, unsigned short* bwd) {
  const int lane = threadIdx.x & 63;
  const int64_t per = d.frags() / 1024;
  for (int64_t b = (int64_t)blockIdx.x * 4 + threadIdx.x / 64; b < 2 * blocks; b += (int64_t)gridDim.x * 4) {
    const bool back = b >= blocks;
    const int64_t q = back ? b - blocks : b;
    const int l = (int)(q / per);
    int64_t i = q - l * per;
    const Net n = net(d, params, l);
    const int64_t n1 = (int64_t)d.H * d.h / 512, n2 = (int64_t)d.h * d.h / 512;
    const float* W = n.W1;
    int K = d.H, N = d.h;
    if (i >= n1 + n2) {
      W = n.W3; K = d.h; N = d.D; i -= n1 + n2;
    } else if (i >= n1) {
      W = n.W2; K = d.h; i -= n1;
    }
    const int slabs = (back ? N : K) / 32;
    const int nt = (int)(i / slabs), ks = (int)(i - (int64_t)nt * slabs);
    const int o = 16 * nt + (lane & 15), k = 32 * ks + 8 * (lane >> 4);
    const float* p = back ? W + (int64_t)o * N + k : W + (int64_t)k * N + o;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = back ? p[e] : p[(int64_t)e * N];
    u32x4t h, lo;
    split8(v, h, lo);
    unsigned short* out = (back ? bwd : fwd) + q * 1024 + lane * 8;
    *(u32x4t*)out = h;
    *(u32x4t*)(out + 512) = lo;
  }
}

// ------------------------------------------------------------------ products of 16 rows
// hi and lo rows of `ld` shorts (K + 8: 16 lanes' 16-byte reads on distinct banks)
struct Rows16 {
  unsigned short *h, *l;
  int ld;
  __device__ __forceinline__ void put(int row, int col, float v) const {
    const unsigned short x = bf_hi(v);
    h[row * ld + col] = x;
    l[row * ld + col] = bf_hi(v - bf_f(x));
  }
};
__device__ __forceinline__ Rows16 rows16(unsigned short*& p, int K) {
  Rows16 r{p, p + kTrainRows * (K + 8), K + 8};
  p += 2 * kTrainRows * (K + 8);
  return r;
}

// A pair of 16-column blocks of a weight matrix in product order
struct Pair {
  const unsigned short *a, *b;
};

// One slab (32 of K) of a pair: acc += lo hi, hi lo, hi hi
__device__ __forceinline__ void slab16(const Rows16& A, int ao, int s, const u32x4t (&f)[4], f32x4t (&acc)[2]) {
  const bf16x8t ah = __builtin_bit_cast(bf16x8t, *(const u32x4t*)(A.h + ao + 32 * s));
  const bf16x8t al = __builtin_bit_cast(bf16x8t, *(const u32x4t*)(A.l + ao + 32 * s));
  bf16x8t b[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) b[j] = __builtin_bit_cast(bf16x8t, f[j]);
#pragma unroll
  for (int j = 0; j < 2; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, b[j], acc[j], 0, 0, 0);
#pragma unroll
  for (int j = 0; j < 2; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, b[2 + j], acc[j], 0, 0, 0);
#pragma unroll
  for (int j = 0; j < 2; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, b[j], acc[j], 0, 0, 0);
}
__device__ __forceinline__ void load16(const Pair& p, int64_t slab, int lane, u32x4t (&f)[4]) {
  const int64_t o = slab * 1024 + lane * 8;
  f[0] = *(const u32x4t*)(p.a + o);
  f[1] = *(const u32x4t*)(p.b + o);
  f[2] = *(const u32x4t*)(p.a + o + 512);
  f[3] = *(const u32x4t*)(p.b + o + 512);
}

// The weights of a wave's products as one stream of slabs, kSlabs of 4 KB ahead of their use.
// RING (every K a multiple of kSlabs slabs = 128): a slab's registers take the load of the slab
// kSlabs further on, across products, layers and barriers, so that the stream never drains (each product
// for itself, D = 1,024, hidden 256: forward 238, backward 268 us; eight slabs ahead 190, 222).
// Otherwise each product loads half of them ahead for itself.
constexpr int kSlabs = 4;
struct Ring {
  u32x4t f[kSlabs][4];
};

// out = A B for the pair `cur` (element r of out[j]: row 4 (lane / 16) + r, column lane % 16); per
// block the sum over `splits` equal parts of K, each an accumulator chain: the plain product's
// arithmetic with its partial tiles (gemm_splits). next: the wave's next pair.
template <bool RING>
__device__ __forceinline__ void product16(Ring& ring, const Rows16& A, int K, int splits, const Pair& cur,
                                          const Pair& next, int lane, f32x4t (&out)[2]) {
  const int n = K / 32, chain = n / splits, ao = (lane & 15) * A.ld + 8 * (lane >> 4);
  f32x4t acc[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) out[j] = acc[j] = f32x4t{0.f, 0.f, 0.f, 0.f};
  bool first = true;
  int left = chain;
  auto part = [&]() {
    left = chain;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      out[j] = first ? acc[j] : out[j] + acc[j];
      acc[j] = f32x4t{0.f, 0.f, 0.f, 0.f};
    }
    first = false;
  };
  if constexpr (RING) {
    for (int s0 = 0; s0 < n; s0 += kSlabs) {
      const bool last = s0 + kSlabs == n;
      const Pair from{last ? next.a : cur.a + (s0 + kSlabs) * 1024, last ? next.b : cur.b + (s0 + kSlabs) * 1024};
#pragma unroll
      for (int u = 0; u < kSlabs; ++u) {
        slab16(A, ao, s0 + u, ring.f[u], acc);
        load16(from, u, lane, ring.f[u]);
      }
      if ((left -= kSlabs) == 0) part();  // uniform
    }
  } else {
    constexpr int U = kSlabs / 2;
#pragma unroll
    for (int u = 0; u < U; ++u) load16(cur, min(u, n - 1), lane, ring.f[u]);
    for (int s0 = 0; s0 < n; s0 += U) {
#pragma unroll
      for (int u = 0; u < U; ++u) load16(cur, min(s0 + U + u, n - 1), lane, ring.f[U + u]);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (s0 + u < n) {  // uniform
          slab16(A, ao, s0 + u, ring.f[u], acc);
          if (--left == 0) part();
        }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int j = 0; j < 4; ++j) ring.f[u][j] = ring.f[U + u][j];
    }
  }
}

template <bool RING>
__device__ __forceinline__ void ring_start(Ring& ring, const Pair& p, int lane) {
  if constexpr (RING)
#pragma unroll
    for (int u = 0; u < kSlabs; ++u) load16(p, u, lane, ring.f[u]);
}

// pair p of a product with K inputs: neighbouring blocks, or (couplings) block p of either half
__device__ __forceinline__ Pair pair_at(const unsigned short* frag, int K, int p, int second) {
  const int64_t bs = (int64_t)(K / 32) * 1024;
  return second ? Pair{frag + p * bs, frag + (second + p) * bs} : Pair{frag + 2 * p * bs, frag + (2 * p + 1) * bs};
}

struct TrainSplits {
  int f1, f2, f3, b2, b1, bz;  // forward products, dh2, dh1, dz
};

// a hidden layer: out = relu(A W + bias), to memory and to LDS
template <bool RING>
__device__ __forceinline__ void hidden16(Ring& ring, const Rows16& A, int K, int h, int splits,
                                         const unsigned short* frag, const Pair& next, const float* bias,
                                         const Rows16& O, float* out, int wave, int lane) {
  const int col = lane & 15, row = 4 * (lane >> 4);
  for (int p = wave; p < h / 32; p += kTrainWaves) {
    const float bv[2] = {bias[32 * p + col], bias[32 * p + 16 + col]};
    f32x4t v[2];
    product16<RING>(ring, A, K, splits, pair_at(frag, K, p, 0),
                    p + kTrainWaves < h / 32 ? pair_at(frag, K, p + kTrainWaves, 0) : next, lane, v);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float x = v[j][r] + bv[j];
        x = x > 0.f ? x : 0.f;
        const int c = 32 * p + 16 * j + col;
        out[(row + r) * h + c] = x;
        O.put(row + r, c, x);
      }
  }
}

template <bool RING>
__global__ void __launch_bounds__(64 * kTrainWaves) k_train_forward(TrainArgs a, TrainSplits sp) {
  extern __shared__ __align__(16) unsigned short lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int H = a.D / 2, h = a.hidden, D = a.D;
  const TrainDims d{H, h, D};
  const int64_t m0 = (int64_t)blockIdx.x * kTrainRows;
  unsigned short* lp = lds;
  const Rows16 C = rows16(lp, H), R1 = rows16(lp, h), R2 = rows16(lp, h);
  Ring ring;
  ring_start<RING>(ring, pair_at(a.fwd + (a.L - 1) * d.frags(), H, wave, 0), lane);
  const Half c0 = half(a, -1);
  for (int e = threadIdx.x; e < kTrainRows * H; e += 64 * kTrainWaves)
    C.put(e / H, e % H, c0.p[(m0 + e / H) * c0.ld + e % H]);
  const int col = lane & 15, row = 4 * (lane >> 4);
  double ld[4] = {0.0, 0.0, 0.0, 0.0};
  for (int t = 0; t < a.L; ++t) {
    const int l = a.L - 1 - t;
    const Net n = net(d, a.params, l);
    const unsigned short *f1 = a.fwd + l * d.frags(), *f2 = f1 + 2 * (int64_t)H * h, *f3 = f2 + 2 * (int64_t)h * h;
    const Half in = half(a, t - 2), out = half(a, t);
    __syncthreads();
    hidden16<RING>(ring, C, H, h, sp.f1, f1, pair_at(f2, h, wave, 0), n.b1, R1, a.h1 + (l * a.B + m0) * h, wave, lane);
    __syncthreads();
    hidden16<RING>(ring, R1, h, h, sp.f2, f2, pair_at(f3, h, wave, H / 16), n.b2, R2, a.h2 + (l * a.B + m0) * h, wave, lane);
    __syncthreads();
    float* o = a.o + (l * a.B + m0) * D;
    const Pair after = l ? pair_at(f1 - d.frags(), H, wave, 0) : pair_at(f3, h, wave, H / 16);
    for (int p = wave; p < H / 16; p += kTrainWaves) {
      const int c = 16 * p + col;
      const float b0 = n.b3[c], b1 = n.b3[H + c];
      float z[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) z[r] = in.p[(m0 + row + r) * in.ld + c];
      f32x4t v[2];
      product16<RING>(ring, R2, h, sp.f3, pair_at(f3, h, p, H / 16),
                      p + kTrainWaves < H / 16 ? pair_at(f3, h, p + kTrainWaves, H / 16) : after, lane, v);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float raw = v[0][r] + b0, sh = v[1][r] + b1;
        o[(row + r) * D + c] = raw;
        o[(row + r) * D + H + c] = sh;
        const float s = a.smax * tanhf(raw / a.smax);
        const float x = (z[r] - sh) * expf(-s);
        out.p[(m0 + row + r) * out.ld + c] = x;
        C.put(row + r, c, x);
        ld[r] += (double)s;
      }
    }
  }
#pragma unroll
  for (int m = 1; m < 16; m *= 2)
#pragma unroll
    for (int r = 0; r < 4; ++r) ld[r] += __shfl_xor(ld[r], m, 64);
  __syncthreads();
  double* sums = (double*)lds;
  if (col == 0)
#pragma unroll
    for (int r = 0; r < 4; ++r) sums[wave * kTrainRows + row + r] = ld[r];
  __syncthreads();
  if (threadIdx.x < kTrainRows) {
    double v = 0.0;
    for (int w = 0; w < kTrainWaves; ++w) v += sums[w * kTrainRows + threadIdx.x];
    a.logdet[m0 + threadIdx.x] = -v;
  }
}

// One element of a coupling's backward (as k_coupling_inv_bwd): o = (raw, t), y the saved input, g = dL/dz
__device__ __forceinline__ void couple_back(const float smax, const float raw, const float t, const float y,
                                            const float g, const float cb, float& draw, float& dt, float& dz) {
  const float th = tanhf(raw / smax);
  const float e = expf(-(smax * th));
  const float xb = (y - t) * e;
  draw = fmaf(-g, xb, cb) * (1.0f - th * th);
  dt = -g * e;
  dz = g * e;
}

// dX = (A W^T) * [kept > 0], to memory and to LDS
template <bool RING>
__device__ __forceinline__ void hidden16_back(Ring& ring, const Rows16& A, int K, int h, int splits,
                                              const unsigned short* frag, const Pair& next, const float* kept,
                                              const Rows16& O, float* out, int wave, int lane) {
  const int col = lane & 15, row = 4 * (lane >> 4);
  for (int p = wave; p < h / 32; p += kTrainWaves) {
    float m[2][4];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) m[j][r] = kept[(row + r) * h + 32 * p + 16 * j + col];
    f32x4t v[2];
    product16<RING>(ring, A, K, splits, pair_at(frag, K, p, 0),
                    p + kTrainWaves < h / 32 ? pair_at(frag, K, p + kTrainWaves, 0) : next, lane, v);
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float x = m[j][r] > 0.f ? v[j][r] : 0.f;
        const int c = 32 * p + 16 * j + col;
        out[(row + r) * h + c] = x;
        O.put(row + r, c, x);
      }
  }
}

template <bool RING>
__global__ void __launch_bounds__(64 * kTrainWaves) k_train_backward(TrainArgs a, TrainSplits sp) {
  extern __shared__ __align__(16) unsigned short lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int H = a.D / 2, h = a.hidden, D = a.D;
  const TrainDims d{H, h, D};
  const int64_t m0 = (int64_t)blockIdx.x * kTrainRows;
  unsigned short* lp = lds;
  const Rows16 O = rows16(lp, D), R2 = rows16(lp, h), R1 = rows16(lp, h);
  const int col = lane & 15, row = 4 * (lane >> 4);
  Ring ring;
  ring_start<RING>(ring, pair_at(a.bwd + 2 * ((int64_t)H * h + (int64_t)h * h), D, wave, 0), lane);
  {  // layer 0's coupling: dz comes from log rho alone
    const Half y = half(a, a.L - 3);
    float* o = a.o + m0 * D;
    for (int e = threadIdx.x; e < kTrainRows * H; e += 64 * kTrainWaves) {
      const int r = e / H, c = e - r * H;
      float* z = a.dz + (m0 + r) * D + H + c;
      float draw, dt, dz;
      couple_back(a.smax, o[r * D + c], o[r * D + H + c], y.p[(m0 + r) * y.ld + c], *z, (float)a.c[m0 + r], draw, dt, dz);
      o[r * D + c] = draw;
      o[r * D + H + c] = dt;
      *z = dz;
      O.put(r, c, draw);
      O.put(r, H + c, dt);
    }
  }
  float cb[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) cb[r] = (float)a.c[m0 + row + r];
  for (int l = 0; l < a.L; ++l) {
    const unsigned short *f1 = a.bwd + l * d.frags(), *f2 = f1 + 2 * (int64_t)H * h, *f3 = f2 + 2 * (int64_t)h * h;
    __syncthreads();
    hidden16_back<RING>(ring, O, D, h, sp.b2, f3, pair_at(f2, h, wave, 0), a.h2 + (l * a.B + m0) * h, R2, a.dh2 + (l * a.B + m0) * h, wave, lane);
    __syncthreads();
    hidden16_back<RING>(ring, R2, h, h, sp.b1, f2, pair_at(f1, h, wave, 0), a.h1 + (l * a.B + m0) * h, R1, a.dh1 + (l * a.B + m0) * h, wave, lane);
    if (l == a.L - 1) break;  // the gradient at the samples themselves is not asked for
    __syncthreads();
    // the conditioning half's gradient is complete with this product: it is the half that layer
    // l + 1 transformed, whose coupling's backward follows element by element
    const Half y = half(a, a.L - 4 - l);
    float *o = a.o + ((l + 1) * a.B + m0) * D, *dz = a.dz + m0 * D + (l % 2 ? H : 0);
    const Pair after = pair_at(f3 + d.frags(), D, wave, 0);
    for (int p = wave; p < H / 32; p += kTrainWaves) {
      float raw[2][4], sh[2][4], yv[2][4], g[2][4];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int c = 32 * p + 16 * j + col, rr = row + r;
          raw[j][r] = o[rr * D + c];
          sh[j][r] = o[rr * D + H + c];
          yv[j][r] = y.p[(m0 + rr) * y.ld + c];
          g[j][r] = dz[(int64_t)rr * D + c];
        }
      f32x4t v[2];
      product16<RING>(ring, R1, h, sp.bz, pair_at(f1, h, p, 0),
                      p + kTrainWaves < H / 32 ? pair_at(f1, h, p + kTrainWaves, 0) : after, lane, v);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int c = 32 * p + 16 * j + col, rr = row + r;
          float draw, dt, dzv;
          couple_back(a.smax, raw[j][r], sh[j][r], yv[j][r], v[j][r] + g[j][r], cb[r], draw, dt, dzv);
          o[rr * D + c] = draw;
          o[rr * D + H + c] = dt;
          dz[(int64_t)rr * D + c] = dzv;
          O.put(rr, c, draw);
          O.put(rr, H + c, dt);
        }
    }
  }
}

// ------------------------------------------------------------------ weight gradients
// dW = X^T dY and db = column sums of dY (in double), for up to kWeightProbs (X, dY) pairs; tiles of
// 128 x 128 of all pairs in one grid, each wave 64 x 32 of it (12 LDS reads per 24 matrix
// instructions). K = samples in stages of 32, two in LDS; a thread converts 8 consecutive samples of
// one column, so reads are coalesced rows and LDS takes 16-byte writes. M and N are multiples of 64:
// the half tile past the edge repeats the last column and is not stored. Every kWeightPart samples the
// accumulators go into a second sum: the matrix unit's rounding errors of one chain grow with the
// square of its length (32,768 equal samples: 2.1e-4 of the sum in one chain, 2.4e-6 so; the launch costs the same).
constexpr int kWeightProbs = 24;
struct WeightProb {
  const float* X;   // rows x M
  const float* dY;  // rows x N
  float* dW;        // M x N
  float* db;        // N
  int64_t ldx;
  int M, N;         // ld of dY and dW: N
};
struct WeightArgs {
  int n;
  int64_t rows;
  WeightProb p[kWeightProbs];
};
constexpr int kWTile = 128, kWRow = 32 + 8, kWeightPart = 256;
struct WeightStage {
  unsigned short Xh[kWTile][kWRow], Xl[kWTile][kWRow], Yh[kWTile][kWRow], Yl[kWTile][kWRow];
};

__global__ void __launch_bounds__(512) k_weight_grads(WeightArgs a) {
  extern __shared__ __align__(16) unsigned char wlds[];
  WeightStage* st = (WeightStage*)wlds;
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int wr = wave >> 2, wc = wave & 3;
  int tile = blockIdx.x, i = 0;
  for (; i < a.n - 1; ++i) {
    const int tiles = ((a.p[i].M + 127) / 128) * ((a.p[i].N + 127) / 128);
    if (tile < tiles) break;
    tile -= tiles;
  }
  const WeightProb& p = a.p[i];
  const int nt = (p.N + 127) / 128, m0 = tile / nt * 128, n0 = tile % nt * 128;
  const int tc = t & 127, tk = __builtin_amdgcn_readfirstlane(t >> 7);  // column, run of 8 samples
  const float* __restrict__ px = p.X + min(m0 + tc, p.M - 1) + 8 * tk * p.ldx;
  const float* __restrict__ py = p.dY + min(n0 + tc, p.N - 1) + (int64_t)8 * tk * p.N;
  const int64_t ldx = p.ldx, ldy = p.N;
  float vx[8], vy[8];
  double bs = 0.0;
  const bool sum = m0 == 0;
  auto load = [&](int64_t k0) {
#pragma unroll
    for (int e = 0; e < 8; ++e) vx[e] = px[(k0 + e) * ldx];
#pragma unroll
    for (int e = 0; e < 8; ++e) vy[e] = py[(k0 + e) * ldy];
  };
  auto put = [&](WeightStage& s) {
    u32x4t h, l;
    split8(vx, h, l);
    *(u32x4t*)&s.Xh[tc][8 * tk] = h;
    *(u32x4t*)&s.Xl[tc][8 * tk] = l;
    split8(vy, h, l);
    *(u32x4t*)&s.Yh[tc][8 * tk] = h;
    *(u32x4t*)&s.Yl[tc][8 * tk] = l;
    if (sum) {
      double u = 0.0;
#pragma unroll
      for (int e = 0; e < 8; ++e) u += (double)vy[e];
      bs += u;
    }
  };
  f32x4t acc[4][2], total[4][2];
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) acc[x][y] = total[x][y] = f32x4t{0.f, 0.f, 0.f, 0.f};
  auto part = [&]() {
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int y = 0; y < 2; ++y) {
        total[x][y] += acc[x][y];
        acc[x][y] = f32x4t{0.f, 0.f, 0.f, 0.f};
      }
  };
  load(0);
  put(st[0]);
  __syncthreads();
  int b = 0;
  for (int64_t k0 = 0; k0 < a.rows; k0 += 32, b ^= 1) {
    const bool more = k0 + 32 < a.rows;
    if (more) load(k0 + 32);
    const WeightStage& s = st[b];
    const int k = 8 * (lane >> 4);
    bf16x8t yh[2], yl[2];
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      const int c = wc * 32 + y * 16 + (lane & 15);
      yh[y] = __builtin_bit_cast(bf16x8t, *(const u32x4t*)&s.Yh[c][k]);
      yl[y] = __builtin_bit_cast(bf16x8t, *(const u32x4t*)&s.Yl[c][k]);
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int r = wr * 64 + x * 16 + (lane & 15);
      const bf16x8t xh = __builtin_bit_cast(bf16x8t, *(const u32x4t*)&s.Xh[r][k]);
      const bf16x8t xl = __builtin_bit_cast(bf16x8t, *(const u32x4t*)&s.Xl[r][k]);
#pragma unroll
      for (int y = 0; y < 2; ++y) acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xl, yh[y], acc[x][y], 0, 0, 0);
#pragma unroll
      for (int y = 0; y < 2; ++y) acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xh, yl[y], acc[x][y], 0, 0, 0);
#pragma unroll
      for (int y = 0; y < 2; ++y) acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xh, yh[y], acc[x][y], 0, 0, 0);
    }
    if (more) put(st[b ^ 1]);
    if ((k0 + 32) % kWeightPart == 0) part();  // uniform
    __syncthreads();
  }
  part();
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      const int col = n0 + wc * 32 + y * 16 + (lane & 15), row = m0 + wr * 64 + x * 16 + 4 * (lane >> 4);
      if (col < p.N && row < p.M)
#pragma unroll
        for (int r = 0; r < 4; ++r) p.dW[(int64_t)(row + r) * p.N + col] = total[x][y][r];
    }
  if (!sum) return;  // uniform
  double* sh = (double*)wlds;
  sh[t] = bs;
  __syncthreads();
  if (t < 128 && n0 + t < p.N) p.db[n0 + t] = (float)(((bs + sh[128 + t]) + sh[256 + t]) + sh[384 + t]);
}

// ------------------------------------------------------------------ launches
static int64_t weight_tiles(int M, int N) { return (int64_t)((M + 127) / 128) * ((N + 127) / 128); }

static TrainSplits train_splits(const TrainArgs& a, int num_cu) {
  const int H = a.D / 2, h = a.hidden;
  auto sp = [&](int N, int K) {
    GemmArgs g{};
    g.M = a.B; g.N = N; g.K = K; g.bf16x3 = 1;
    return gemm_splits(g, num_cu);
  };
  return {sp(h, H), sp(h, h), sp(a.D, h), sp(h, a.D), sp(h, h), sp(H, h)};
}

static size_t rows_lds(int K, int h) { return sizeof(unsigned short) * 2 * kTrainRows * ((K + 8) + 2 * (size_t)(h + 8)); }

size_t train_frags(const TrainArgs& a) {
  return 2 * (size_t)a.L * TrainDims{a.D / 2, a.hidden, a.D}.frags() * sizeof(unsigned short);
}

bool train_supported(const TrainArgs& a, int num_cu) {
  if (a.L < 2 || a.B <= 0 || a.B % 64 || a.hidden <= 0 || a.hidden % 64 || a.D <= 0 || a.D % 128) return false;
  if (rows_lds(a.D, a.hidden) > kTrainLds || a.B / kTrainRows > 0x7fffff) return false;
  // few weight tiles meet many samples: the plain products split the samples over the chip
  const int64_t tiles = a.L * (weight_tiles(a.hidden, a.D) + weight_tiles(a.hidden, a.hidden) + weight_tiles(a.D / 2, a.hidden));
  if (a.B > 4096 && tiles * 4 < num_cu) return false;
  return (((uintptr_t)a.params | (uintptr_t)a.grad | (uintptr_t)a.z0 | (uintptr_t)a.z1 | (uintptr_t)a.halves |
           (uintptr_t)a.h1 | (uintptr_t)a.h2 | (uintptr_t)a.o | (uintptr_t)a.dz | (uintptr_t)a.dh1 | (uintptr_t)a.dh2 |
           (uintptr_t)a.fwd | (uintptr_t)a.bwd) & 15) == 0;
}

template <bool RING>
static hipError_t launch_rows(bool back, const TrainArgs& a, int num_cu, hipStream_t s) {
  static unsigned long long set_f = 0, set_b = 0;
  const dim3 grid((unsigned)(a.B / kTrainRows)), block(64 * kTrainWaves);
  if (back) {
    if (hipError_t e = ensure_dynamic_lds((const void*)k_train_backward<RING>, kTrainLds, set_b)) return e;
    hipLaunchKernelGGL(k_train_backward<RING>, grid, block, rows_lds(a.D, a.hidden), s, a, train_splits(a, num_cu));
  } else {
    if (hipError_t e = ensure_dynamic_lds((const void*)k_train_forward<RING>, kTrainLds, set_f)) return e;
    hipLaunchKernelGGL(k_train_forward<RING>, grid, block, rows_lds(a.D / 2, a.hidden), s, a, train_splits(a, num_cu));
  }
  return hipGetLastError();
}
// the stream's conditions: every part of every K whole rings, every wave with a pair in each product
static bool train_ring(const TrainArgs& a, int num_cu) {
  const int H = a.D / 2, h = a.hidden;
  const TrainSplits s = train_splits(a, num_cu);
  auto whole = [](int K, int splits) { return K % (32 * kSlabs * splits) == 0; };
  return whole(H, s.f1) && whole(h, s.f2) && whole(h, s.f3) && whole(a.D, s.b2) && whole(h, s.b1) && whole(h, s.bz) &&
         h / 32 >= kTrainWaves && H / 32 >= kTrainWaves;
}

hipError_t launch_train_forward(const TrainArgs& a, int num_cu, hipStream_t s) {
  const TrainDims d{a.D / 2, a.hidden, a.D};
  const int64_t blocks = a.L * (d.frags() / 1024);
  const int64_t grid = std::min<int64_t>((2 * blocks + 3) / 4, 65536);
  hipLaunchKernelGGL(k_train_weights, dim3((unsigned)grid), dim3(256), 0, s, d, a.params, blocks, a.fwd, a.bwd);
  if (hipError_t e = hipGetLastError()) return e;
  return train_ring(a, num_cu) ? launch_rows<true>(false, a, num_cu, s) : launch_rows<false>(false, a, num_cu, s);
}

hipError_t launch_train_backward(const TrainArgs& a, int num_cu, hipStream_t s) {
  if (hipError_t e = train_ring(a, num_cu) ? launch_rows<true>(true, a, num_cu, s) : launch_rows<false>(true, a, num_cu, s))
    return e;
  static unsigned long long lds_set_w = 0;
  const int H = a.D / 2, h = a.hidden;
  const int64_t B = a.B;
  const TrainDims d{H, h, a.D};
  if (hipError_t e = ensure_dynamic_lds((const void*)k_weight_grads, 2 * sizeof(WeightStage), lds_set_w)) return e;
  for (int l0 = 0; l0 < a.L; l0 += kWeightProbs / 3) {
    WeightArgs w{};
    w.rows = B;
    int64_t tiles = 0;
    auto add = [&](const float* X, int64_t ldx, const float* dY, const float* dW, const float* db, int M, int N) {
      w.p[w.n++] = {X, dY, const_cast<float*>(dW), const_cast<float*>(db), ldx, M, N};
      tiles += weight_tiles(M, N);
    };
    for (int l = l0; l < std::min(a.L, l0 + kWeightProbs / 3); ++l) {
      const Net g = net(d, a.grad, l);
      const Half cond = half(a, a.L - 2 - l);
      add(a.h2 + l * B * h, h, a.o + l * B * a.D, g.W3, g.b3, h, a.D);
      add(a.h1 + l * B * h, h, a.dh2 + l * B * h, g.W2, g.b2, h, h);
      add(cond.p, cond.ld, a.dh1 + l * B * h, g.W1, g.b1, H, h);
    }
    if (tiles > 0x7fffff) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_weight_grads, dim3((unsigned)tiles), dim3(512), 2 * sizeof(WeightStage), s, w);
    if (hipError_t e = hipGetLastError()) return e;
  }
  return hipSuccess;
}

}  // namespace pib
