// Harmonic-rho bead sampler (draw_sample + transform_sampled_coordinates).
//
// Replaces pibronic/pimc/pimc.py:326-334 (normal draws with the source surface's standard
// deviations), :386-389 (categorical surface source) and :613-631 (R = U_circ . cc + d_src).
//
// Distribution: for mode j the bead coordinates of the reference are Gaussian with mean
// d_src,j and covariance Lambda_j^-1, Lambda_j = 2 coth_j I - csch_j C (C the ring adjacency
// matrix; pimc.py:401-404 lists its eigenvalues), independent of the surface. The reference
// draws in C's eigenbasis (a dense P x P transform). Here Lambda_j = L_j L_j^T is factored
// once on the host: a cyclic tridiagonal matrix has a Cholesky factor with only the diagonal,
// the subdiagonal and the last row non-zero, so x = L_j^-T z, z ~ N(0, I), is an exact draw
// from N(0, Lambda_j^-1) by an O(P) back substitution (the standard sampler for Gaussian
// Markov random fields, Rue 2001). Same distribution, O(P) instead of O(P^2) per row.
//
// Random numbers: Philox4x32-10 keyed by the run seed. The beads 4m..4m+3 of row (global
// sample s, mode j) take the four normals of the counter (s*N + j, m, 0): two Box-Muller
// pairs, each from a 32-bit radius uniform and a 32-bit angle uniform (FP32 transform, FP64
// recurrence); a radius uniform below 2^-20 is refined to 64 bits by the counter
// (s*N + j, m, 2), so that the tails reach ~9.4 sigma. The surface source of sample s uses
// the counter (s, 0, 1).
// Sources are drawn per sample rather than once per run (quirk Q5 of the reference draws them
// all up front; same distribution).
//
// Layout: a wave takes one mode of 64 consecutive samples, one lane per row (sample, mode), so
// the mode's factor entries are wave-uniform scalar loads. Each lane walks its beads
// downwards in chunks of 8 to 32; a chunk is staged in LDS and the wave then writes the 64 rows'
// chunk with consecutive lanes on consecutive addresses (64- to 256-byte row segments).
#include <algorithm>

#include "pib_common.hpp"
#include "pib_kernels.hpp"

namespace pib {

constexpr int kSampleWaves = 4;   // waves per work-group, each independent
// Beads staged per lane before a write-out: 8 up to 24 beads per row (see also below), else 16 (a whole 128-byte line
// where rows start on one), or 32 where rows start off a line and the launch writes more than the
// 256 MB of the memory-side cache. Half lines written apart reach memory one by one once the rows in
// flight exceed the L2, and so do the two ends of a run off the line, fewer in longer runs; short rows
// and cached writes lose more by the waves that the larger LDS tile displaces. MI355X, us with 8 / 16 / 32,
// A N P samples: 4 8 64 1e5 122 / 90 / 105, 8 16 64 1e5 271 / 160 / 184, 6 12 256 16,384 134 / 92 / 103,
// 4 8 101 60,000 206 / 181 / 142, 4 8 60 1e5 (384 MB) 16 / 32: 140 / 126, 6 12 250 16,384 178 / 140,
// 6 12 70 16,384 (110 MB) 33 / 36, 11 17 50 32,768 74 / 61 / 73; 2 6 24 1e5 29 / 33, 3 6 16 1e5 22.0 / 22.8,
// 2 3 12 1e4 5.6 / 6.3.
static int chunk_for(const SampleArgs* a, int n) {
  double all = 0.0, off = 0.0;
  int longest = 0;
  for (int i = 0; i < n; ++i) {
    const double bytes = 8.0 * a[i].B * a[i].N * a[i].P;
    const bool line = a[i].P % 16 == 0 && (uintptr_t)a[i].q % 128 == 0;
    all += bytes;
    if (!line && a[i].P >= 48) off += bytes;
    if (a[i].P > longest) longest = a[i].P;
  }
  if (longest <= 24) return 8;
  // in a small launch a last piece of 8 to 15 beads (written out with divisions) costs more than half lines do:
  // 3 28 2,000 7.9 / 8.5, 12 25 2,000 8.0 / 8.5, 3 28 20,000 9.6 / 10.2 with 8 / 16; 12 28 20,000 19.9 / 18.7
  if (longest < 48 && longest % 16 >= 8 && all < 16 * 1048576.0) return 8;
  return all > 256 * 1048576.0 && 2.0 * off > all ? 32 : 16;
}

__device__ __forceinline__ int draw_source(const SampleArgs& a, int64_t gsample) {
  if (a.A_rho == 1) return 0;
  const u32x4 r = philox4x32_10(u32x4{(uint32_t)gsample, (uint32_t)(gsample >> 32), 0u, 1u},
                                a.key0, a.key1);
  const double u = u53(r.x, r.y);
  int s = 0;
  while (s < a.A_rho - 1 && u >= a.cdf[s]) ++s;
  return s;
}

// the four normals of beads 4m..4m+3 of row grow: two Box-Muller pairs from one Philox call
// in FP32 with the hardware log2, square root and sin/cos (v_sin_f32 / v_cos_f32 take their
// argument in revolutions), widened to FP64. The radius uniform below 2^-20 is refined to 64
// bits (rounded to FP32 before its log2), so the tails reach ~9.4 sigma instead of the
// 6.7 sigma of a 32-bit uniform. The normals carry ~1e-7 relative error against an exact transform of the same
// uniforms: a shift of the sampled distribution far below the statistical error of any block
// (the estimator evaluates rho exactly at the coordinates drawn).
__device__ __forceinline__ void normal_quad(uint64_t grow, int m, uint32_t k0, uint32_t k1, double (&z)[4]) {
  const u32x4 r = philox4x32_10(u32x4{(uint32_t)grow, (uint32_t)(grow >> 32), (uint32_t)m, 0u}, k0, k1);
  float l2a = __log2f(((float)r.x + 0.5f) * 0x1.0p-32f);
  float l2b = __log2f(((float)r.z + 0.5f) * 0x1.0p-32f);
  if (r.x < (1u << 12) || r.z < (1u << 12)) {  // rare: P = 2^-19 per call
    const u32x4 t = philox4x32_10(u32x4{(uint32_t)grow, (uint32_t)(grow >> 32), (uint32_t)m, 2u}, k0, k1);
    if (r.x < (1u << 12)) l2a = __log2f((float)(((double)r.x * 0x1.0p32 + (double)t.x + 0.5) * 0x1.0p-64));
    if (r.z < (1u << 12)) l2b = __log2f((float)(((double)r.z * 0x1.0p32 + (double)t.z + 0.5) * 0x1.0p-64));
  }
  const float ra = __fsqrt_rn(-1.3862943611198906f * l2a), rb = __fsqrt_rn(-1.3862943611198906f * l2b);
  const float ua = ((float)r.y + 0.5f) * 0x1.0p-32f, ub = ((float)r.w + 0.5f) * 0x1.0p-32f;
  z[0] = (double)(ra * __builtin_amdgcn_cosf(ua));
  z[1] = (double)(ra * __builtin_amdgcn_sinf(ua));
  z[2] = (double)(rb * __builtin_amdgcn_cosf(ub));
  z[3] = (double)(rb * __builtin_amdgcn_sinf(ub));
}

// one unit of work of a wave: mode u % N of the sample group u / N
template <int CHUNK>
__device__ __forceinline__ void sample_unit(const SampleArgs& a, int64_t u, int64_t offset, int lane, double* stage) {
  const int P = a.P, N = a.N;
  constexpr int ld = CHUNK + 1;  // padded LDS row
  // wave-uniform: the sample group and the mode; every lane of the wave runs the same chunks
  const int64_t sg = u / N;
  const int j = (int)(u - sg * N);
  const int64_t s0 = sg * kWave;
  const int64_t s = s0 + lane;
  const bool live = s < a.B;
  const int64_t gs = offset + (live ? s : s0);
  const int src = live ? draw_source(a, gs) : 0;
  const uint64_t grow = (uint64_t)gs * (uint64_t)N + (uint64_t)j;
  // the mode's factor entries are the same for the whole wave: read through the constant
  // address space (the kernel never writes them), so they come by scalar loads
  typedef const double __attribute__((address_space(4))) cdouble;
  cdouble* dinv = (cdouble*)(a.chol + (int64_t)j * 3 * P);
  cdouble* sub = dinv + P;
  cdouble* last = sub + P;
  const double d = a.shift[src * N + j];
  if (live && a.src && j == 0) a.src[s] = src;
  const int nrow = (a.B - s0) < kWave ? (int)(a.B - s0) : kWave;
  const int64_t rstride = (int64_t)N * P;
  double zq[4], xl = 0.0, xn = 0.0;
  // beads in descending order, in chunks [kb, ke) aligned to multiples of CHUNK, and within
  // a chunk quad by quad. One formula for every bead: the host stores sub[k] = 0 for
  // k >= P-2 and last[P-1] = 0, and x_{P-1} (xl) and x_{k+1} (xn) start at 0, so bead P-1
  // gives z dinv and bead P-2 (z - last xl) dinv exactly.
  // Lanes past the block's end (the last group only) run the same uniform loop on the
  // group's first sample; their rows are never written out.
  for (int kb = ((P - 1) / CHUNK) * CHUNK; kb >= 0; kb -= CHUNK) {
    const int ke = kb + CHUNK < P ? kb + CHUNK : P;
#pragma unroll 2
    for (int m = (ke - 1) >> 2; m >= (kb >> 2); --m) {
      double cd[4], cs[4], cl[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int k = 4 * m + e < P ? 4 * m + e : P - 1;  // the top quad may be partial
        cd[e] = dinv[k];
        cs[e] = sub[k];
        cl[e] = last[k];
      }
      normal_quad(grow, m, a.key0, a.key1, zq);
#pragma unroll
      for (int e = 3; e >= 0; --e) {
        const int k = 4 * m + e;
        if (k < ke) {  // uniform over the wave
          const double x = fma(-cl[e], xl, fma(-cs[e], xn, zq[e])) * cd[e];
          if (k == P - 1) xl = x;
          xn = x;
          stage[lane * ld + (k - kb)] = x + d;
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // write out: row rr (sample s0 + rr, mode j) has its beads contiguous in q
    const int w_ = ke - kb;
    double* __restrict__ qj = a.q + (s0 * N + j) * (int64_t)P + kb;
    if (w_ == CHUNK && nrow == kWave) {  // full chunk: no divisions
#pragma unroll 4
      for (int it = 0; it < CHUNK; ++it) {
        const int e = lane + kWave * it, rr = e / CHUNK, kk = e % CHUNK;
        qj[rr * rstride + kk] = stage[rr * ld + kk];
      }
    } else {
      for (int e = lane; e < nrow * w_; e += kWave) {
        const int rr = e / w_, kk = e - rr * w_;
        qj[rr * rstride + kk] = stage[rr * ld + kk];
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

template <int CHUNK>
__global__ void __launch_bounds__(kWave * kSampleWaves) k_sample_fp64(const SampleArgs a) {
  __shared__ double stage_all[kSampleWaves][kWave * (CHUNK + 1)];
  const int64_t units = (a.B + kWave - 1) / kWave * a.N;  // (sample group, mode) pairs
  const int lane = threadIdx.x & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);  // wave-uniform
  const int64_t offset = a.step ? a.offset + *a.step * a.B : a.offset;
  for (int64_t u = (int64_t)blockIdx.x * kSampleWaves + w; u < units; u += (int64_t)gridDim.x * kSampleWaves)
    sample_unit<CHUNK>(a, u, offset, lane, stage_all[w]);
}

// The samplers of several problems (the temperatures of a batch) in one launch: one problem's
// rows alone leave the chip mostly waiting on each wave's serial walk over the beads. Sixteen
// temperatures of A = 6, N = 12, P = 52..256, 16,384 samples each (MI355X): 1.69 ms as sixteen
// launches with half-line write-out, 1.33 as one with 32 beads (3.9 GB written; a fill reaches 6.7 TB/s).
// The caller puts the longest rows first, so that the short ones fill the tail.
template <int CHUNK>
__global__ void __launch_bounds__(kWave * kSampleWaves) k_sample_batched(const SampleBatch b) {
  __shared__ double stage_all[kSampleWaves][kWave * (CHUNK + 1)];
  const int lane = threadIdx.x & (kWave - 1);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  int64_t u = (int64_t)blockIdx.x * kSampleWaves + w;
  for (int i = 0; i < b.n; ++i) {  // wave-uniform
    const SampleArgs& a = b.p[i];
    const int64_t units = (a.B + kWave - 1) / kWave * a.N;
    if (u < units) {
      sample_unit<CHUNK>(a, u, a.step ? a.offset + *a.step * a.B : a.offset, lane, stage_all[w]);
      return;
    }
    u -= units;
  }
}

hipError_t launch_sample_fp64(const SampleArgs& a, hipStream_t s) {
  const int64_t units = (a.B + kWave - 1) / kWave * a.N;  // one wave each
  int64_t groups = (units + kSampleWaves - 1) / kSampleWaves;
  if (groups > 65536) groups = 65536;
  if (groups < 1) groups = 1;
  const dim3 grid((unsigned)groups), block(kWave * kSampleWaves);
  switch (chunk_for(&a, 1)) {
    case 8: hipLaunchKernelGGL(k_sample_fp64<8>, grid, block, 0, s, a); break;
    case 16: hipLaunchKernelGGL(k_sample_fp64<16>, grid, block, 0, s, a); break;
    default: hipLaunchKernelGGL(k_sample_fp64<32>, grid, block, 0, s, a);
  }
  return hipGetLastError();
}

hipError_t launch_sample_batch(const SampleArgs* args, int n, hipStream_t s) {
  for (int i0 = 0; i0 < n; i0 += kSampleBatchProbs) {
    SampleBatch b{};
    b.n = std::min(kSampleBatchProbs, n - i0);
    int64_t units = 0;
    for (int i = 0; i < b.n; ++i) {
      b.p[i] = args[i0 + i];
      units += (b.p[i].B + kWave - 1) / kWave * b.p[i].N;
    }
    const int64_t groups = (units + kSampleWaves - 1) / kSampleWaves;
    if (groups > 65536 * kSampleBatchProbs) {  // beyond one launch's grid: the strided launches
      for (int i = 0; i < b.n; ++i)
        if (hipError_t e = launch_sample_fp64(b.p[i], s)) return e;
      continue;
    }
    const dim3 grid((unsigned)groups), block(kWave * kSampleWaves);
    switch (chunk_for(b.p, b.n)) {
      case 8: hipLaunchKernelGGL(k_sample_batched<8>, grid, block, 0, s, b); break;
      case 16: hipLaunchKernelGGL(k_sample_batched<16>, grid, block, 0, s, b); break;
      default: hipLaunchKernelGGL(k_sample_batched<32>, grid, block, 0, s, b);
    }
    if (hipError_t e = hipGetLastError()) return e;
  }
  return hipSuccess;
}

}  // namespace pib
