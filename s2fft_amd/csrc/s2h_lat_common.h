// Device helpers shared by the latitudinal (Wigner-d) kernels.
//
// Start values: d^{l0}_{m,n}(theta) = K cos(theta/2)^ecos sin(theta/2)^esin
// evaluated as (mantissa, exponent) so that sin^a cos^b cannot underflow at
// high m; the result is split into a stored double and an integer scale index
// lscale <= 0 with true value = stored * 2^(512 lscale).  A lane contributes
// only while lscale == 0 (earlier terms are below 2^-256 of the O(1) ones).
#pragma once

#include "s2h_internal.h"
#include "s2h_kernels.h"

namespace s2h {
namespace lat {

struct Ext {
  double m;
  int e;
};

__device__ __forceinline__ Ext ext_of(double v) {
  int e;
  const double m = frexp(v, &e);
  return {m, e};
}
__device__ __forceinline__ Ext ext_mul(Ext a, Ext b) {
  int e;
  const double m = frexp(a.m * b.m, &e);
  return {m, a.e + b.e + e};
}
__device__ __forceinline__ Ext ext_pow(double base, int k) {
  Ext r = {0.5, 1};
  Ext x = ext_of(base);
  while (k) {
    if (k & 1) r = ext_mul(r, x);
    k >>= 1;
    if (k) x = ext_mul(x, x);
  }
  return r;
}

// Start value d^{l0}_{m,n}(theta) split into (stored, lscale).
__device__ __forceinline__ void start_value(const MStart& st, double c2, double s2, double& d,
                                            int& lscale) {
  Ext v = {st.kmant, st.kexp};
  if (st.ecos) v = ext_mul(v, ext_pow(c2, st.ecos));
  if (st.esin) v = ext_mul(v, ext_pow(s2, st.esin));
  if (v.m == 0.0) {
    d = 0.0;
    lscale = 0;
    return;
  }
  int ls = -((256 - v.e) >> 9);
  if (ls > 0) ls = 0;
  lscale = ls;
  d = ldexp(v.m, v.e - 512 * ls);
}

// (hi + lo) 2^e: a factor with its rounding error, |hi| in [1/2, 1) or zero.
struct ExtD {
  double hi, lo;
  int e;
};
__device__ __forceinline__ ExtD extd_of(double v, double rel) {
  int e;
  const double hi = frexp(v, &e);
  return {hi, hi * rel, e};
}
// a *= b, not normalised: hundreds of factors in [1/4, 1) fit
__device__ __forceinline__ void extd_mul(ExtD& a, const ExtD& b) {
  const double p = a.hi * b.hi;
  a.lo = fma(a.hi, b.lo, fma(a.lo, b.hi, fma(a.hi, b.hi, -p)));
  a.hi = p;
  a.e += b.e;
}
// a *= x^k by squarings of x, each brought back to [1/2, 1)
__device__ __forceinline__ void extd_mul_pow(ExtD& a, ExtD x, int k) {
  while (k) {
    if (k & 1) extd_mul(a, x);
    k >>= 1;
    if (k) {
      const double p = x.hi * x.hi;
      const double lo = fma(2.0 * x.hi, x.lo, fma(x.hi, x.hi, -p));
      int e;
      x.hi = frexp(p, &e);
      x.lo = ldexp(lo, -e);
      x.e = 2 * x.e + e;
    }
  }
}

// start_value for the FP64 kernels.  c2 and s2 rounded to FP64 and multiplied
// up carry a relative error of about j eps into every d of their ring and m
// (the largest error of the transforms: 5e-14 at L = 512); here the rounding
// errors of c2, s2 and of every product are kept.  One power of c2 s2 and one
// of the difference of the exponents (at most 2 |n|) in place of two powers.
__device__ __forceinline__ void start_value_fp64(const MStart& st, const LatRing& rg, double& d,
                                                 int& lscale) {
  const ExtD c = extd_of(rg.c2, rg.c2r), s = extd_of(rg.s2, rg.s2r);
  const int k = st.ecos < st.esin ? st.ecos : st.esin;
  ExtD v = {st.kmant, 0.0, st.kexp};
  if (k) {
    ExtD cs = c;  // in [1/4, 1)
    extd_mul(cs, s);
    extd_mul_pow(v, cs, k);
  }
  if (st.ecos > k) extd_mul_pow(v, c, st.ecos - k);
  if (st.esin > k) extd_mul_pow(v, s, st.esin - k);
  if (v.hi == 0.0) {
    d = 0.0;
    lscale = 0;
    return;
  }
  int ve;
  v.hi = frexp(v.hi, &ve);
  v.lo = ldexp(v.lo, -ve);
  ve += v.e;
  int ls = -((256 - ve) >> 9);
  if (ls > 0) ls = 0;
  lscale = ls;
  d = ldexp(v.hi + v.lo, ve - 512 * ls);
}

// Moves (d, dm1) down by 2^512 once |d| passes 2^256.  The recursion grows
// by less than 2.5 per step, so checks every 32 steps cannot overflow.
__device__ __forceinline__ void rescale(double& d, double& dm1, int& lscale) {
  const bool big = fabs(d) > 0x1p256;
  const double f = big ? 0x1p-512 : 1.0;
  d *= f;
  dm1 *= f;
  lscale += big ? 1 : 0;
}

// Blocks go to the 8 XCDs in turn and there to the 32 CUs in turn, the longest
// columns first; every second row of 32 in reverse evens out what the CUs get
// (forward at L = 1024 173 -> 165 us).
__device__ __forceinline__ int balanced_block(int i, int n) {
  const int j = i >> 3;
  return ((j >> 5) & 1) && (j | 31) < (n >> 3) ? ((j ^ 31) << 3) | (i & 7) : i;
}

// blockIdx.x -> m: c adjacent m per XCD in a row (workgroups are dealt to the
// 8 XCDs round-robin), heaviest (smallest |m|) first, every second row over the
// XCDs in reverse.  For m_lo < 0 the order is 0, -1, 1, -2, 2, ...: two runs of c / 2
// columns, and the matrix-core kernels, bound by their 16-byte accesses to the
// spectra, take c = 16 so that an XCD's L2 sees whole lines (MW L = 512, spin 2, 64
// maps: BF16 inverse, which wrote 1.05 GB for 0.54 GB of spectra, 825 us with c = 4,
// 735 with 16; HEALPix L = 512, spin 2, 16 maps, forward 660 and 620); 4 spread the
// work more evenly (VALU forward, GL L = 400, spin 1, 3 maps 97 us and 100).
__device__ __forceinline__ int m_of_block(int i, int nm, int m_lo, int cfull = 16) {
  const int c = m_lo == 0 ? 4 : cfull;
  const int nfull = nm & ~(8 * c - 1);  // the remap is a bijection on [0, nfull)
  int idx = i;
  if (i < nfull) {
    const int k = i >> 3, r = k / c;
    const int xcd = r & 1 ? 7 - (i & 7) : i & 7;
    idx = r * 8 * c + xcd * c + k % c;
  }
  if (m_lo == 0) return idx;
  return (idx & 1) ? -((idx + 1) >> 1) : (idx >> 1);
}

// Block i of a launch over nm m-values x G ring groups (grid.x = nm G) ->
// (m, ring group g).  Blocks are dispatched round-robin over the 8 XCDs by
// linear index, so i & 7 is the XCD and i >> 3 the order on it: the G groups
// of one m are consecutive blocks of one XCD.  They run together and read the
// m's harmonic and recursion coefficients through that XCD's L2, not HBM.  The m-values
// follow m_of_block.  A bijection of [0, nm G) onto [0, nm) x [0, G).
__device__ __forceinline__ int m_group_of_block(int i, int nm, int G, int m_lo, int& g,
                                                int cfull = 16) {
  const int nm8 = nm & ~7;
  int ip;
  if (i < nm8 * G) {
    const int xcd = i & 7, j = i >> 3;
    const int k = j / G;
    g = j - k * G;
    ip = 8 * k + xcd;
  } else {
    const int r = i - nm8 * G;
    const int k = r / G;
    g = r - k * G;
    ip = nm8 + k;
  }
  return m_of_block(ip, nm, m_lo, cfull);
}

// Recursion coefficients of one 32-step chunk, staged in LDS so that every
// step reads them with a broadcast LDS load instead of a dependent global or
// scalar load: (a', -b' * bsign, sigma) for l = blk + i; a' and b' are zero from
// l = L - 1 on, which makes the steps past the band-limit produce zeros.
struct ChunkCoef {
  double a, nb, c, pad;
};
constexpr int kChunk = 32;

__device__ __forceinline__ ChunkCoef finish_coef(const Coef& c, double bsign) {
  return {c.a, -c.b * bsign, c.c, 0.0};
}

// Chunk `blk`'s coefficient for lane i (< 32) as stored, zero past l = L - 1.  A
// prefetch keeps it in this form until it is written to LDS (finish_coef
// there): arithmetic on the loaded value right after the load would make the
// wave wait for the memory latency at once.
__device__ __forceinline__ Coef load_ucoef_raw(const Coef* __restrict__ cf, int blk, int i, int L) {
  const int l = blk + i;
  Coef v = {0.0, 0.0, 0.0, 0.0};
  if (l < L) v = cf[l];
  return v;
}

// One recursion step with staged coefficients: e_{l+1}.
__device__ __forceinline__ double rec_step_unit(const ChunkCoef& c, double x, double e, double em1) {
  return fma(fma(c.a, x, c.nb), e, -em1);
}

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The part of the conjugate-gradient dot <Y, A(Y)> over the ring rows
// [a.dot_row_lo, a.dot_row_hi), fused into a synthesis epilogue: those rows
// have no aliasing and one w n = a.dot_wn, so A(Y) = w n Y and a stored value
// v adds c_m w n v^2 (c_m = 2 for m > 0 of real maps).  dacc[t]: the lane's
// sum of v^2 for its map tile t (map 8 t + (lane % 16) / 2 of the workgroup,
// both components).  The workgroup adds the lanes up in a fixed order
// (component, lane group, wave) into a.dot_part[map * a.dot_part_stride +
// blockIdx.x].  red: 2 NW 64 doubles of LDS no longer read by any thread;
// every thread calls this.
template <int NW>
__device__ void synth_dot_partials(const LatArgs& a, int m, int b0, const double (&dacc)[2],
                                   double* red) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  red[(wave * 64 + lane) * 2] = dacc[0];
  red[(wave * 64 + lane) * 2 + 1] = dacc[1];
  __syncthreads();
  if (threadIdx.x < 16) {
    const int mi = threadIdx.x, t = mi >> 3, j = mi & 7;
    double s = 0.0;
    for (int w = 0; w < NW; ++w)
      for (int kg = 0; kg < 4; ++kg)
        for (int c = 0; c < 2; ++c) s += red[(w * 64 + 16 * kg + 2 * j + c) * 2 + t];
    if (b0 + mi < a.batch)
      a.dot_part[(int64_t)(b0 + mi) * a.dot_part_stride + blockIdx.x] =
          (m > 0 ? 2.0 : 1.0) * a.dot_wn * s;
  }
}

typedef double v4d __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

// 16x16x4 matrix-core products.  Operand layouts (both types): A[i][k] in
// lane i + 16k, B[k][j] in lane j + 16k.  The result layouts differ:
// FP64 holds C[i][j] in lane j + 16 (i%4), register i/4; FP32 holds it in
// lane j + 16 (i/4), register i%4.  row_of(r, kq) is the row held in
// register r by lanes 16 kq .. 16 kq + 15.
template <typename T>
struct Mma;
template <>
struct Mma<double> {
  typedef v4d acc;
  __device__ static acc run(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  __device__ static int row_of(int r, int kq) { return 4 * r + kq; }
};
template <>
struct Mma<float> {
  typedef v4f acc;
  __device__ static acc run(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  __device__ static int row_of(int r, int kq) { return 4 * kq + r; }
};

}  // namespace lat
}  // namespace s2h
