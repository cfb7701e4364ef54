// Ragged ring FFTs, every ring in the registers of its threads.
//
// Forward  (s2fft/utils/healpix_ffts.py:187-226 + spherical.py:533-546):
//   out[row, col] = w_t * exp(-i m phi0_t) * F_t[m mod nphi_t],  m = m_first + col
//   with F_t the unnormalised DFT of the ring; the periodic extension, the
//   quadrature weight and the ring phase are fused into the store.
// Inverse  (healpix_ffts.py:335-371 + spherical.py:183-200):
//   F_t[q] = sum_{m = q mod nphi} exp(+i m phi0_t) c(m), f_t[p] = sum_q F_t[q] e^{2 pi i q p/nphi}
//   the folding and the phase are fused into the load.
//
// Three kinds of rings: the grid's one power-of-two length as such (from 64 points on),
// other powers of two in passes through LDS, every other length by Bluestein's chirp-z
// (Bluestein 1970).  Lengths with small prime factors too: with a mixed-radix LDS
// kernel for those the grid of nside 192, five maps, took 109 us and 62 without it.
// RMS error of a ring against extended precision, the former LDS kernels (radix 8, odd
// primes to 13, convolutions) beside it: powers of two 1.9e-16 at 256 points (2.6e-16)
// and 2.4e-16 at 4096 (4.5e-16); other lengths 3.5e-16 below 64 points (4.5e-16 and
// more), 4.4e-16 below 1100 (smooth lengths 13.8e-16, others 7.3e-16) and 4.9e-16 above
// (18.8e-16, 8.8e-16).  Powers of two as convolutions would have 2 to 4 times theirs.
// Two real maps share one complex transform (z = x + i y, split by the
// conjugate symmetry of the spectra), halving the transforms for real data.
//
// T = N / 16 threads per ring hold 16 points each, p = t + T e in the first pass
// (coalesced loads straight into it), and run radix-16 passes with one LDS
// exchange between passes: N = 4096: 16 x 16 x 16, 2048, 1024, 512: 16 x 16 x
// 8, 4, 2, 256: 16 x 16, 128, 64: 16 x 8, 16 x 4.  An exchange writes the
// positions its thread read last, so it needs one barrier.
//
// Powers of two: the last pass takes the sub-transforms so that thread t ends
// up with X[t + T e]: coalesced stores, no exchange into natural order.
//
// Bluestein: X[k] = c_k sum_p (x_p c_p) conj(c_{k-p}), c_k = e^{-i pi k^2/n}, the
// convolution by two FFTs of M >= 2n - 1 points (M = 8192: 16 x 16 x 16 x 2, the
// radix 2 between neighbouring lanes).  Decimation in frequency forward and in
// time back, so nothing is put into natural order in between: FFT(chirp) is
// stored in the order of the registers.  Four barriers per convolution; the
// zero upper half of the input and the unwanted upper half of the output are
// left out of the first and last pass.
// Chirps, FFT(chirp) and twiddles come from the plan's table, every one rounded from its
// own evaluation: FFT(chirp) from a transform with multiplied-up twiddles, and twiddles
// multiplied up here, left 1.6 times the error.
//
// What bounds it: the large grids their HBM traffic (64 maps of L = 512 MW, 1.07
// GB: 0.38 ms forward and 0.40 inverse, 2.8 TB/s; the former LDS kernels with
// one barrier pair per radix-8 pass took 2.14 and 2.29), with two waves per SIMD
// (the 16 points and their twiddles); single maps the latency of the passes (L =
// 128, one map: 10 us, was 18; nside 512: 45, was 119; inverse 57, was 147).
//
// HEALPix ring phases are e^{-i m phi0} with phi0 = 0 or pi / n, so the phase of
// column m = k + j n is (-1)^j e^{-i pi k / n}: one product per residue and a
// sign per column, in both directions.
#include <algorithm>

#include "s2h_fft_lds.h"
#include "s2h_kernels.h"
#include "s2h_lat_common.h"

namespace s2h {

namespace {

constexpr double kC8 = 0.92387953251128675613, kS8 = 0.38268343236508977173;  // cos, sin pi/8
constexpr double kR2 = 0.70710678118654752440;

__device__ __forceinline__ cplx cconj(cplx a) { return {a.x, -a.y}; }
// a * w (INV: a * conj w)
template <bool INV>
__device__ __forceinline__ cplx tmul(cplx a, cplx w) {
  return INV ? cplx{fma(a.x, w.x, a.y * w.y), fma(a.y, w.x, -(a.x * w.y))}
             : cplx{fma(a.x, w.x, -(a.y * w.y)), fma(a.x, w.y, a.y * w.x)};
}
// -i a (INV: i a)
template <bool INV>
__device__ __forceinline__ cplx mul_mi(cplx a) {
  return INV ? cplx{-a.y, a.x} : cplx{a.y, -a.x};
}

template <bool INV>
__device__ __forceinline__ void dft2(cplx& a, cplx& b) {
  const cplx t = a;
  a = cadd(t, b);
  b = csub(t, b);
}
template <bool INV>
__device__ __forceinline__ void dft4(cplx& a, cplx& b, cplx& c, cplx& d) {
  const cplx s0 = cadd(a, c), d0 = csub(a, c), s1 = cadd(b, d), d1 = mul_mi<INV>(csub(b, d));
  a = cadd(s0, s1);
  b = cadd(d0, d1);
  c = csub(s0, s1);
  d = csub(d0, d1);
}
// w16^k a for the twiddles inside radix 8 and 16
template <bool INV, int K>
__device__ __forceinline__ cplx w16(cplx a) {
  if constexpr (K == 0) return a;
  if constexpr (K == 1) return tmul<INV>(a, cplx{kC8, -kS8});
  if constexpr (K == 2) {
    const cplx t = mul_mi<INV>(a);
    return {kR2 * (a.x + t.x), kR2 * (a.y + t.y)};
  }
  if constexpr (K == 3) return tmul<INV>(a, cplx{kS8, -kC8});
  if constexpr (K == 4) return mul_mi<INV>(a);
  if constexpr (K == 6) {
    const cplx t = mul_mi<INV>(a);
    return {kR2 * (t.x - a.x), kR2 * (t.y - a.y)};
  }
  if constexpr (K == 9) return tmul<INV>(a, cplx{-kC8, kS8});
  return a;
}
template <bool INV>
__device__ __forceinline__ void dft8(cplx* v) {
  dft4<INV>(v[0], v[2], v[4], v[6]);
  dft4<INV>(v[1], v[3], v[5], v[7]);
  const cplx o1 = w16<INV, 2>(v[3]), o2 = mul_mi<INV>(v[5]), o3 = w16<INV, 6>(v[7]);
  const cplx e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6], o0 = v[1];
  v[0] = cadd(e0, o0);
  v[4] = csub(e0, o0);
  v[1] = cadd(e1, o1);
  v[5] = csub(e1, o1);
  v[2] = cadd(e2, o2);
  v[6] = csub(e2, o2);
  v[3] = cadd(e3, o3);
  v[7] = csub(e3, o3);
}
// 16 points, natural order in and out.  HALF_IN: v[8..15] are zero (not read);
// HALF_OUT: only v[0..7] are wanted.
template <bool INV, bool HALF_IN, bool HALF_OUT>
__device__ __forceinline__ void dft16(cplx* v) {
  // columns j: points j, j + 4, j + 8, j + 12 -> y[j][k]
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if constexpr (HALF_IN) {
      const cplx a = v[j], b = v[j + 4], t = mul_mi<INV>(b);
      v[j] = cadd(a, b);
      v[j + 4] = cadd(a, t);
      v[j + 8] = csub(a, b);
      v[j + 12] = csub(a, t);
    } else {
      dft4<INV>(v[j], v[j + 4], v[j + 8], v[j + 12]);
    }
  }
  v[5] = w16<INV, 1>(v[5]);
  v[6] = w16<INV, 2>(v[6]);
  v[7] = w16<INV, 3>(v[7]);
  v[9] = w16<INV, 2>(v[9]);
  v[10] = w16<INV, 4>(v[10]);
  v[11] = w16<INV, 6>(v[11]);
  v[13] = w16<INV, 3>(v[13]);
  v[14] = w16<INV, 6>(v[14]);
  v[15] = w16<INV, 9>(v[15]);
  // rows k: X[k + 4 m]
  cplx x[16];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    cplx a = v[4 * k], b = v[4 * k + 1], c = v[4 * k + 2], d = v[4 * k + 3];
    dft4<INV>(a, b, c, d);
    x[k] = a;
    x[k + 4] = b;
    x[k + 8] = c;
    x[k + 12] = d;
  }
#pragma unroll
  for (int k = 0; k < (HALF_OUT ? 8 : 16); ++k) v[k] = x[k];
}

// w, w^2, w^4 and w^8 of w = e^{-2 pi i t / 2^LOG}, t < T = 2^LOG / 16, from the
// plan's table (ring_twiddles), each rounded once.
struct Tw16 {
  cplx w, w2, w4, w8;
};
__device__ __forceinline__ Tw16 load_tw16(const cplx* __restrict__ tab, int T, int t) {
  const cplx* p = tab + 4 * (T - 2) + t;
  return {p[0], p[T], p[2 * T], p[3 * T]};
}

// v[k] *= w^k (INV: conj w^k), the other powers by products of depth 2 at most.
// Squared up from w alone they carry up to 15 times its rounding error: rings of 256
// points had 3.6e-16 of RMS error instead of 1.9e-16, of 4096 5.2e-16 instead of 2.4e-16
// (MW L = 512, 64 maps, inverse rings 434 -> 443 us; nside 512, one map, unchanged).
template <bool INV>
__device__ __forceinline__ void twiddle16(cplx* v, const Tw16& q) {
  const cplx w = q.w, w2 = q.w2, w4 = q.w4, w8 = q.w8;
  v[1] = tmul<INV>(v[1], w);
  v[2] = tmul<INV>(v[2], w2);
  v[4] = tmul<INV>(v[4], w4);
  v[8] = tmul<INV>(v[8], w8);
  const cplx w3 = cmul(w2, w), w5 = cmul(w4, w), w6 = cmul(w4, w2), w9 = cmul(w8, w);
  v[3] = tmul<INV>(v[3], w3);
  v[5] = tmul<INV>(v[5], w5);
  v[6] = tmul<INV>(v[6], w6);
  v[9] = tmul<INV>(v[9], w9);
  v[7] = tmul<INV>(v[7], cmul(w4, w3));
  v[10] = tmul<INV>(v[10], cmul(w8, w2));
  v[11] = tmul<INV>(v[11], cmul(w8, w3));
  v[12] = tmul<INV>(v[12], cmul(w8, w4));
  v[13] = tmul<INV>(v[13], cmul(w8, w5));
  v[14] = tmul<INV>(v[14], cmul(w8, w6));
  v[15] = tmul<INV>(v[15], cmul(w8, cmul(w4, w3)));
}

template <int LOGM>
struct Shape {
  static constexpr int M = 1 << LOGM, T = M / 16;
  static constexpr int S = T >= 16 ? T / 16 : T;  // points per sub-transform of the last stage
  static constexpr int LDS = M + (LOGM <= 9 ? M / 8 + 32 : 0);  // complex per ring
  // LDS place of point q.  8 neighbouring lanes take 128 bytes per cycle: the
  // passes access runs of consecutive q or one q per lane S apart, spread over
  // the banks by an exclusive-or within each aligned group of 8 (no room for
  // padding at the large M), by padding at the small ones.
  __device__ static int at(int q) {
    if constexpr (LOGM >= 13) return q ^ (((q >> 5) & 3) << 1);
    if constexpr (LOGM == 12) return q ^ ((q >> 4) & 7);
    if constexpr (LOGM == 11) return q ^ ((q >> 3) & 7);
    if constexpr (LOGM == 10) return q ^ ((q >> 3) & 3) ^ (((q >> 6) & 1) << 2);
    if constexpr (LOGM == 9) return q + (q >> 3) + (q >> 5) * 2;
    if constexpr (LOGM == 8) return q + (q >> 4);
    return q + (q >> 3);
  }
};

// A value the compiler takes for new: what is computed from it again (twiddle
// powers, LDS places) is computed again and not held in registers meanwhile.
__device__ __forceinline__ int renew(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

__device__ __forceinline__ double swap_lane1(double x) {
  // lane ^ 1 by a quad permute (1, 0, 3, 2)
  const long long v = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_mov_dpp((int)(v & 0xffffffff), 0xB1, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(v >> 32), 0xB1, 0xF, 0xF, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// e^{-2 pi i k / 32}
__device__ __constant__ const double kW32[16][2] = {
    {1.0, 0.0},
    {0.98078528040323044913, -0.19509032201612826785},
    {0.92387953251128675613, -0.38268343236508977173},
    {0.83146961230254523708, -0.55557023301960222474},
    {0.70710678118654752440, -0.70710678118654752440},
    {0.55557023301960222474, -0.83146961230254523708},
    {0.38268343236508977173, -0.92387953251128675613},
    {0.19509032201612826785, -0.98078528040323044913},
    {0.0, -1.0},
    {-0.19509032201612826785, -0.98078528040323044913},
    {-0.38268343236508977173, -0.92387953251128675613},
    {-0.55557023301960222474, -0.83146961230254523708},
    {-0.70710678118654752440, -0.70710678118654752440},
    {-0.83146961230254523708, -0.55557023301960222474},
    {-0.92387953251128675613, -0.38268343236508977173},
    {-0.98078528040323044913, -0.19509032201612826785}};

template <int S, bool INV>
__device__ __forceinline__ void dft_groups(cplx* v) {
#pragma unroll
  for (int g = 0; g < 16; g += S) {
    if constexpr (S == 2) dft2<INV>(v[g], v[g + 1]);
    if constexpr (S == 4) dft4<INV>(v[g], v[g + 1], v[g + 2], v[g + 3]);
    if constexpr (S == 8) dft8<INV>(v + g);
    if constexpr (S == 16) dft16<INV, false, false>(v + g);
  }
}

// v[e], e < 8: the chirped input at p = t + T e -> the convolution there.
template <int LOGM>
__device__ __forceinline__ void blue_conv(cplx* v, cplx* lds, int t0, const cplx* __restrict__ bhat,
                                          const cplx* __restrict__ tw) {
  typedef Shape<LOGM> P;
  constexpr int T = P::T, S = P::S;
  int t = t0;
  const Tw16 w1 = load_tw16(tw, T, t);  // of e^{-2 pi i t / M}
  dft16<false, true, false>(v);
  twiddle16<false>(v, w1);
#pragma unroll
  for (int k = 0; k < 16; ++k) lds[P::at(k * T + t)] = v[k];
  __syncthreads();
  if constexpr (T < 16) {
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = lds[P::at((t + T * (i / S)) * S + i % S)];
    dft_groups<S, false>(v);
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = cmul(v[i], bhat[i * T + t]);
    dft_groups<S, true>(v);
    t = renew(t);
#pragma unroll
    for (int i = 0; i < 16; ++i) lds[P::at((t + T * (i / S)) * S + i % S)] = v[i];
  } else {
    int nn = t % S, base = (t / S) * T + nn;
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = lds[P::at(base + i * S)];
    dft16<false, false, false>(v);
    if constexpr (S == 1) {
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = cmul(v[i], bhat[i * T + t]);
    } else {
      twiddle16<false>(v, load_tw16(tw, S, nn));  // of e^{-2 pi i nn / T}
#pragma unroll
      for (int i = 0; i < 16; ++i) lds[P::at(base + i * S)] = v[i];
      __syncthreads();
      if constexpr (S <= 16) {
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = lds[P::at((t + T * (i / S)) * S + i % S)];
        dft_groups<S, false>(v);
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = cmul(v[i], bhat[i * T + t]);
        dft_groups<S, true>(v);
        t = renew(t);
#pragma unroll
        for (int i = 0; i < 16; ++i) lds[P::at((t + T * (i / S)) * S + i % S)] = v[i];
      } else {
        // S = 32: 16 x 2, the radix 2 between lanes t and t ^ 1
        const int odd = t & 1, b3 = (t >> 1) * 32 + odd;
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = lds[P::at(b3 + 2 * i)];
        dft16<false, false, false>(v);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const cplx w = odd ? cplx{kW32[i][0], kW32[i][1]} : cplx{1.0, 0.0};
          const cplx a = cmul(v[i], w);
          const cplx o = {swap_lane1(a.x), swap_lane1(a.y)};
          // X = (even + odd, even - odd); times FFT(chirp); and back
          cplx y = odd ? csub(o, a) : cadd(a, o);
          y = cmul(y, bhat[i * T + t]);
          const cplx q = {swap_lane1(y.x), swap_lane1(y.y)};
          y = odd ? csub(q, y) : cadd(y, q);
          v[i] = tmul<true>(y, w);
        }
        dft16<true, false, false>(v);
        t = renew(t);
#pragma unroll
        for (int i = 0; i < 16; ++i) lds[P::at((t >> 1) * 32 + (t & 1) + 2 * i)] = v[i];
      }
      nn = t % S;
      base = (t / S) * T + nn;
      const Tw16 w2 = load_tw16(tw, S, nn);
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = lds[P::at(base + i * S)];
      twiddle16<true>(v, w2);
    }
    dft16<true, false, false>(v);
    base = renew(base);
#pragma unroll
    for (int i = 0; i < 16; ++i) lds[P::at(base + i * S)] = v[i];
  }
  t = renew(t);
  const Tw16 w3 = load_tw16(tw, T, t);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 16; ++k) v[k] = lds[P::at(k * T + t)];
  twiddle16<true>(v, w3);
  dft16<true, false, true>(v);
}

// ------------------------------------------------------------- powers of two
template <int LOGN>
struct Pow2Shape {
  static constexpr int N = 1 << LOGN, T = N / 16, LOGT = LOGN - 4;
  static constexpr int S = T >= 16 ? T / 16 : T;
  // LDS place of point q: an exclusive-or with the row q / T, bits reversed,
  // keeps all three access patterns (runs of lanes, runs of S, one row per
  // lane) free of bank conflicts
  __device__ static int at(int q) {
    if constexpr (LOGT == 2) return q ^ ((q >> 3) & 3);
    const int r = q >> LOGT;
    return q ^ (((r & 1) << 2) | (r & 2) | ((r >> 2) & 1));
  }
};

// v[e] = x[t + T e] -> X[t + T e] (INV: the unnormalised inverse).
template <int LOGN, bool INV>
__device__ __forceinline__ void pow2_fft(cplx* v, cplx* lds, int t, const cplx* __restrict__ tw) {
  typedef Pow2Shape<LOGN> P;
  constexpr int T = P::T, S = P::S;
  const Tw16 w1 = load_tw16(tw, T, t);
  dft16<INV, false, false>(v);
  twiddle16<INV>(v, w1);
#pragma unroll
  for (int k = 0; k < 16; ++k) lds[P::at(k * T + t)] = v[k];
  __syncthreads();
  if constexpr (T >= 16) {
    const int nn = t % S, base = (t / S) * T + nn;
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = lds[P::at(base + i * S)];
    dft16<INV, false, false>(v);
    if constexpr (S > 1) {
      twiddle16<INV>(v, load_tw16(tw, S, nn));
#pragma unroll
      for (int i = 0; i < 16; ++i) lds[P::at(base + i * S)] = v[i];
      __syncthreads();
    }
  }
  if constexpr (S > 1) {
    // sub-transforms g = t + T i: k = g + R s, R = 256 (T < 16: 16)
    constexpr int G = 16 / S;
    cplx u[16];
#pragma unroll
    for (int i = 0; i < G; ++i) {
      const int g = t + T * i;
      const int q0 = T >= 16 ? (g & 15) * T + (g >> 4) * S : g * T;
#pragma unroll
      for (int s = 0; s < S; ++s) u[i * S + s] = lds[P::at(q0 + s)];
    }
    dft_groups<S, INV>(u);
#pragma unroll
    for (int i = 0; i < G; ++i)
#pragma unroll
      for (int s = 0; s < S; ++s) v[i + G * s] = u[i * S + s];
  }
}

// ------------------------------------------------------------- rings in and out
__device__ __forceinline__ double ring_scale(int mode, int n) {
  return mode == 1 ? 1.0 / (double)n : mode == 2 ? 1.0 / sqrt((double)n) : 1.0;
}
__device__ __forceinline__ bool ring_phase(int apply, const RingJob& job) {
  return apply && rint(job.nphi * job.phi0_over_pi) != 0.0;
}

// Loads through these take unconditional loads from clamped places (one basic
// block: all of them in flight together) and drop the unwanted values afterwards.

// v[e] = pixel t + T e of the ring (z = x + i y for a pair of real maps), zero
// from n on.
template <int E>
__device__ __forceinline__ void load_pixels(const int T, cplx* v, const RingFwdArgs& a, const RingJob& job,
                                            int t, int64_t b0, int paired, bool two) {
  const int n = job.nphi;
  const int64_t off = b0 * a.map_stride + job.pix_offset;
  const int64_t next = two ? a.map_stride : 0;
  const auto at = [&](int e) { return t + T * e < n ? t + T * e : 0; };
  bool real = a.real_only_all || (a.real_only_2L && n == 2 * a.L);
  if (paired && !a.f_complex) {
    const double* s0 = reinterpret_cast<const double*>(a.f) + off;
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = {s0[at(e)], s0[next + at(e)]};
    real = !two;
  } else if (paired) {
    const cplx* s0 = reinterpret_cast<const cplx*>(a.f) + off;
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = {s0[at(e)].x, s0[next + at(e)].x};
    real = !two;
  } else if (a.in_single) {
    const float2* s0 = reinterpret_cast<const float2*>(a.f) + off;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const float2 x = s0[at(e)];
      v[e] = {(double)x.x, (double)x.y};
    }
  } else {
    const cplx* s0 = reinterpret_cast<const cplx*>(a.f) + off;
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = s0[at(e)];
  }
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const bool in = t + T * e < n;
    v[e] = {in ? v[e].x : 0.0, in && !real ? v[e].y : 0.0};
  }
}

// Stores a ring whose residues have at most one column each, from registers:
// residue p = t + T e (phased) is column m = p or p - n.
template <int E>
__device__ __forceinline__ void store_direct(const int T, const cplx* v, const RingFwdArgs& a,
                                             const RingJob& job, int t, int64_t b0, bool ph) {
  const int n = job.nphi;
  cplx* d0 = a.out + b0 * a.out_map_stride + (int64_t)job.row * a.ncol;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int p = t + T * e;
    int col = p - a.m_first;
    const bool wrap = col >= n;
    if (wrap) col -= n;
    const double sg = wrap && ph ? -1.0 : 1.0;
    if (p < n && col < a.ncol) d0[col] = {sg * v[e].x, sg * v[e].y};
  }
}

// Stores a ring's columns from its residues in LDS: [0, n), real pairs the
// second map's at [n, 2n).  Column m = k + j n is (-1)^j times residue k (ph).
__device__ __forceinline__ void store_columns(const int T, const cplx* lds, const RingFwdArgs& a,
                                              const RingJob& job, int t, int64_t b0, bool two,
                                              bool ph) {
  const int n = job.nphi;
  const int64_t o0 = b0 * a.out_map_stride + (int64_t)job.row * a.ncol;
  cplx* d0 = a.out + o0;
  float2* d0s = reinterpret_cast<float2*>(a.out) + o0;
  int k = (a.m_first + t) % n;
  if (k < 0) k += n;
  int j = (a.m_first + t - k) / n;
  const int dj = T / n, dk = T - dj * n;
  for (int col = t; col < a.ncol; col += T) {
    const bool zero = a.zero_neg_2L && n == 2 * a.L && a.m_first + col < 0;
    const double sg = zero ? 0.0 : ph && (j & 1) ? -1.0 : 1.0;
    const cplx z = lds[k];
    if (a.out_single)
      d0s[col] = make_float2((float)(sg * z.x), (float)(sg * z.y));
    else
      d0[col] = {sg * z.x, sg * z.y};
    if (two) {
      const cplx y = lds[n + k];
      d0[a.out_map_stride + col] = {sg * y.x, sg * y.y};
    }
    k += dk;
    j += dj;
    if (k >= n) {
      k -= n;
      ++j;
    }
  }
}

// Natural-order residues v[e] (t + T e) into LDS for store_columns, times
// phase(p); real pairs split into X = (z + conj z')/2, Y = (z - conj z')/(2i),
// z' the residue n - p.  Called by every thread; ends on a barrier.
template <int E, typename Phase>
__device__ __forceinline__ void residues_to_lds(const int T, cplx* v, cplx* lds, int n, int t, int paired,
                                                Phase phase) {
  __syncthreads();
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int p = t + T * e;
    if (p < n) lds[p] = paired ? v[e] : phase(e, v[e]);
  }
  __syncthreads();
  if (!paired) return;
  cplx zc[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int p = t + T * e;
    zc[e] = p < n ? lds[p == 0 ? 0 : n - p] : cplx{0.0, 0.0};
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int p = t + T * e;
    if (p >= n) continue;
    const cplx X = {0.5 * (v[e].x + zc[e].x), 0.5 * (v[e].y - zc[e].y)};
    const cplx Y = {0.5 * (v[e].y + zc[e].y), -0.5 * (v[e].x - zc[e].x)};
    lds[p] = phase(e, X);
    lds[n + p] = phase(e, Y);
  }
  __syncthreads();
}

// The folded spectrum F[q] = sum_{m = q mod n} (-1)^j c(m), m = q + j n in [lo, hi]
// (the sign for ph), of a map or of z = c_x + i c_y of a pair of real maps.
struct FoldIn {
  const cplx* x;
  const cplx* y;      // second map of a pair, or null
  const float2* xs;   // complex64 spectra instead of x, or null
  int m_first, lo, hi, n;
  bool herm, ph;

  __device__ FoldIn(const RingInvArgs& a, const RingJob& job, int64_t b0, bool two) {
    const int64_t in0 = b0 * a.in_map_stride + (int64_t)job.row * a.ncol;
    n = job.nphi;
    herm = a.herm_mode == 1 || (a.herm_mode == 2 && n == 2 * a.L);
    lo = herm ? -(a.L - 1) : a.m_lo;
    hi = herm ? (a.L - 1) : a.m_hi;
    x = a.in + in0;
    y = two ? x + a.in_map_stride : nullptr;
    xs = a.in_single ? reinterpret_cast<const float2*>(a.in) + in0 : nullptr;
    m_first = a.m_first;
    ph = ring_phase(a.apply_phase, job);
  }
  // u[e] = c(m), or c_x(m) + i c_y(m), for m = at(e), zero where m is outside
  // [lo, hi]; m < 0 of Hermitian spectra from conj c(-m), m = 0 without its
  // imaginary part: a map alone drops it with the imaginary part of the ring, in a
  // pair it would be the partner's (at(e) = 0 for an e < N0 at most)
  template <int E, int N0, typename At>
  __device__ __forceinline__ void gather(cplx* u, At at) const {
    // The m once, and only uniform branches from here on: with && and the m computed
    // again at each use, the compiler (ROCm 7.2) branched around the selections, and in
    // one instance lost the imaginary part of every m >= 0 of the second map.
    int m[E], place[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      m[e] = at(e);
      const int am = herm & (m[e] < 0) ? -m[e] : m[e];
      place[e] = (m[e] < lo) | (m[e] > hi) ? 0 : am - m_first;
    }
    if (xs) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const float2 r = xs[place[e]];
        u[e] = {(double)r.x, (double)r.y};
      }
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e) u[e] = x[place[e]];
    }
#pragma unroll
    for (int e = 0; e < N0; ++e) u[e].y = herm & (m[e] == 0) ? 0.0 : u[e].y;
    if (y) {
      cplx r[E];
#pragma unroll
      for (int e = 0; e < E; ++e) r[e] = y[place[e]];
#pragma unroll
      for (int e = 0; e < N0; ++e) r[e].y = herm & (m[e] == 0) ? 0.0 : r[e].y;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const double sg = herm & (m[e] < 0) ? -1.0 : 1.0;
        u[e] = {fma(-sg, r[e].y, u[e].x), fma(sg, u[e].y, r[e].x)};
      }
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e) u[e].y = herm & (m[e] < 0) ? -u[e].y : u[e].y;
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const bool in = (m[e] >= lo) & (m[e] <= hi);
      u[e] = {in ? u[e].x : 0.0, in ? u[e].y : 0.0};
    }
  }
  __device__ static int floor_div(int p, int q) { return p >= 0 ? p / q : -((q - 1 - p) / q); }

  // v[e] = F[t + T e], for rings longer than T
  template <int E>
  __device__ __forceinline__ void owned(const int T, cplx* v, int t) const {
    if (hi - lo < n) {  // one m per residue
#pragma unroll
      for (int e0 = 0; e0 < E; e0 += 8)
        gather<8, 1>(v + e0, [&](int e) {
          const int q = t + T * (e0 + e);
          return q >= n ? hi + 1 : q <= hi ? q : q - n;
        });
      if (ph) {
#pragma unroll
        for (int e = 0; e < E; ++e)
          if (t + T * e > hi) v[e] = {-v[e].x, -v[e].y};
      }
      return;
    }
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = {0.0, 0.0};
    if (E == 8 && n <= 2 * T) {
      aliases<2, 0>(T, v, t);
    } else {
      aliases<8, 0>(T, v, t);
      if constexpr (E > 8) aliases<8, 8>(T, v, t);
    }
  }
  // v[E0 + e] += the sum over j of c(q + j n), q = t + T (E0 + e), e < EV, in batches of
  // eight loads, of 8 / EV values of j: a batch waits out one memory latency, and a ring
  // just longer than T, with 16 columns per thread, would need 14 of one j each (nside 64,
  // one map, back: 17.1 -> 11.7 us, nside 256, 4 maps 49 -> 42)
  template <int EV, int E0>
  __device__ __forceinline__ void aliases(const int T, cplx* v, int t) const {
    constexpr int JV = 8 / EV;
    const int j1 = floor_div(hi, n);
    for (int j = floor_div(lo, n); j <= j1; j += JV) {
      cplx u[8];
      gather<8, JV == 1 ? 1 : 8>(u, [&](int k) {
        const int q = t + T * (E0 + k % EV);
        return (q < n) & (j + k / EV <= j1) ? q + (j + k / EV) * n : hi + 1;
      });
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const double sg = ph && ((j + k / EV) & 1) ? -1.0 : 1.0;
        cplx& x = v[E0 + k % EV];
        x = {fma(sg, u[k].x, x.x), fma(sg, u[k].y, x.y)};
      }
    }
  }
  // a thread's share of residue t % n, for rings of at most T points: the
  // G = T / n threads of a residue take j = j0 + g, j0 + g + G, ...
  __device__ __forceinline__ cplx shared(const int T, int t) const {
    cplx part = {0.0, 0.0};
    const int G = T / n, q = t % n, g = t / n;
    if (g >= G) return part;
    const int j1 = floor_div(hi, n);
    for (int jb = floor_div(lo, n) + g; jb <= j1; jb += 8 * G) {
      cplx u[8];
      gather<8, 8>(u, [&](int i) { return q + (jb + i * G) * n; });
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const double sg = ph && ((jb + i * G) & 1) ? -1.0 : 1.0;
        part = {fma(sg, u[i].x, part.x), fma(sg, u[i].y, part.y)};
      }
    }
    return part;
  }
  // v[e] = F[t + T e], e < 8.  Called by every thread, with one barrier inside;
  // another before lds is written again.
  __device__ __forceinline__ void residues(const int T, cplx* v, cplx* lds, int t) const {
    cplx part = {0.0, 0.0};
    if (n > T) {
      owned<8>(T, v, t);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = {0.0, 0.0};
      part = shared(T, t);
    }
    lds[t] = part;
    __syncthreads();
    if (n <= T && t < n) {
      for (int g = 0; g < T / n; ++g) v[0] = cadd(v[0], lds[g * n + t]);
    }
  }
};

// Stores pixel t + T e from v[e]; with sub_from the result is subtracted from it.
template <int E>
__device__ __forceinline__ void store_pixels(const int T, cplx* v, const RingInvArgs& a, const RingJob& job,
                                             int t, int64_t b0, int paired, bool two, bool herm) {
  const int n = job.nphi;
  const int64_t off = b0 * a.map_stride + job.pix_offset;
  if (paired || !a.f_complex) {
    double* d0 = reinterpret_cast<double*>(a.f) + off;
    if (a.sub_from) {
      const double* u0 = reinterpret_cast<const double*>(a.sub_from) + off;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int p = t + T * e;
        if (p < n) v[e] = {u0[p] - v[e].x, two ? u0[a.map_stride + p] - v[e].y : 0.0};
      }
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int p = t + T * e;
      if (p >= n) continue;
      d0[p] = v[e].x;
      if (two) d0[a.map_stride + p] = v[e].y;
    }
  } else if (a.f_single) {
    float2* d0 = reinterpret_cast<float2*>(a.f) + off;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int p = t + T * e;
      if (p < n) d0[p] = make_float2((float)v[e].x, herm ? 0.0f : (float)v[e].y);
    }
  } else {
    cplx* d0 = reinterpret_cast<cplx*>(a.f) + off;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if (herm) v[e].y = 0.0;
    }
    if (a.sub_from) {
      const cplx* u0 = reinterpret_cast<const cplx*>(a.sub_from) + off;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int p = t + T * e;
        if (p < n) v[e] = csub(u0[p], v[e]);
      }
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int p = t + T * e;
      if (p < n) d0[p] = v[e];
    }
  }
}

// Consecutive jobs of one kind within a launch: blocks [block0, ...) hold
// blockDim / T rings each.
struct RingSeg {
  int body;      // log2 of the convolution (Bluestein), kPow2Body + log2 n, or
                 // kSubBody + log2 of the convolution whose threads it takes
  int job0, count, block0;
  int direct;    // forward: every residue has at most one column (ring_direct)
  int lds_ring;  // complex of LDS per ring
};
constexpr int kPow2Body = 32, kSubBody = 64;
constexpr int kMaxSegs = 2 * kBlueClasses + 1;
constexpr int kRingLdsMax = 160 * 1024;
struct RingSegs {
  RingSeg s[kMaxSegs];
  int n;
};

// the ring of this thread, and its place in it
struct RingOf {
  int t, sub;
  bool valid, two;
  int64_t b0;
  RingJob job;
  cplx* lds;
  __device__ RingOf(const int T, const RingJob* jobs, const RingSeg& seg, int paired, int batch, void* raw) {
    t = threadIdx.x % T;
    sub = threadIdx.x / T;
    const int r = (blockIdx.x - seg.block0) * (blockDim.x / T) + sub;
    valid = r < seg.count;
    job = jobs[seg.job0 + (valid ? r : seg.count - 1)];
    b0 = paired ? 2 * (int64_t)blockIdx.y : (int64_t)blockIdx.y;
    two = paired && b0 + 1 < batch;
    lds = reinterpret_cast<cplx*>(raw) + sub * seg.lds_ring;
  }
};

template <int LOGM>
__device__ __forceinline__ void blue_fwd(const RingFwdArgs& a, const RingSeg& seg, int paired,
                                         void* raw) {
  typedef Shape<LOGM> P;
  constexpr int T = P::T;
  const RingOf ring(T, a.jobs, seg, paired, a.batch, raw);
  const RingJob& job = ring.job;
  cplx* lds = ring.lds;
  const int n = job.nphi;
  int t = ring.t;
  const cplx* __restrict__ bhat = a.chirp_pool + job.chirp_off;
  const cplx* __restrict__ chirp = bhat + P::M;
  const cplx* __restrict__ phase = chirp + n;

  cplx v[16];
  load_pixels<8>(T, v, a, job, t, ring.b0, paired, ring.two);
  cplx c[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int p = t + T * e;
    c[e] = p < n ? chirp[p] : cplx{0.0, 0.0};
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = cmul(v[e], c[e]);
  blue_conv<LOGM>(v, lds, t, bhat, a.chirp_pool);

  const double w = (a.apply_weight ? job.weight : 1.0) * ring_scale(a.norm_mode, n);
  t = renew(t);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int p = t + T * e;
    const cplx ch = p < n ? chirp[p] : cplx{0.0, 0.0};
    v[e] = cmul(v[e], cplx{w * ch.x, w * ch.y});
  }
  const bool ph = ring_phase(a.apply_phase, job);
  if (seg.direct) {
    if (ring.valid) store_direct<8>(T, v, a, job, t, ring.b0, false);
    return;
  }
  residues_to_lds<8>(T, v, lds, n, t, paired, [&](int e, cplx z) {
    return ph ? cmul(z, phase[t + T * e]) : z;
  });
  if (ring.valid) store_columns(T, lds, a, job, t, ring.b0, ring.two, ph);
}

template <int LOGM>
__device__ __forceinline__ void blue_inv(const RingInvArgs& a, const RingSeg& seg, int paired,
                                         void* raw) {
  typedef Shape<LOGM> P;
  constexpr int T = P::T;
  const RingOf ring(T, a.jobs, seg, paired, a.batch, raw);
  const RingJob& job = ring.job;
  cplx* lds = ring.lds;
  const int n = job.nphi;
  int t = ring.t;
  const cplx* __restrict__ bhat = a.chirp_pool + job.chirp_off;
  const cplx* __restrict__ chirp = bhat + P::M;
  const cplx* __restrict__ phase = chirp + n;
  const FoldIn in(a, job, ring.b0, ring.two);

  cplx v[16];
  in.residues(T, v, lds, t);
  const double w = (a.apply_weight ? job.weight : 1.0) * ring_scale(a.norm_mode, n);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int p = t + T * e;
    if (p < n) {
      const cplx ch = chirp[p];
      // conj(F e^{i pi p / n}) c_p
      cplx f = {w * v[e].x, -w * v[e].y};
      if (in.ph) f = cmul(f, phase[p]);
      v[e] = cmul(f, ch);
    }
  }
  __syncthreads();  // the partial sums are read
  blue_conv<LOGM>(v, lds, t, bhat, a.chirp_pool);
  if (!ring.valid) return;
  t = renew(t);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int p = t + T * e;
    const cplx z = cmul(v[e], p < n ? chirp[p] : cplx{0.0, 0.0});
    v[e] = {z.x, -z.y};
  }
  store_pixels<8>(T, v, a, job, t, ring.b0, paired, ring.two, in.herm);
}

// Rings of another power of two, on the threads of a Bluestein ring (half of its points
// at most): all T threads load, fold and store; the transform runs in self-sorting
// passes through LDS, the first of radix 2, 4, 8 or 16 without twiddles, the others of
// radix 16.  A HEALPix grid has two rings of each.
template <int R, bool INV>
__device__ __forceinline__ void sub_pass(const cplx* src, cplx* dst, const int T, int t, int n,
                                         int Ns, const cplx* __restrict__ tw) {
  const int nb = n / R;
  for (int j = t; j < nb; j += T) {
    cplx u[16];
#pragma unroll
    for (int r = 0; r < R; ++r) u[r] = src[j + r * nb];
    const int jl = j & (Ns - 1);
    if constexpr (R == 16) {
      if (Ns > 1) twiddle16<INV>(u, load_tw16(tw, Ns, jl));
      dft16<INV, false, false>(u);
    }
    if constexpr (R == 8) dft8<INV>(u);
    if constexpr (R == 4) dft4<INV>(u[0], u[1], u[2], u[3]);
    if constexpr (R == 2) dft2<INV>(u[0], u[1]);
#pragma unroll
    for (int k = 0; k < R; ++k) dst[(j - jl) * R + jl + k * Ns] = u[k];
  }
}
// v[e] = x[t + T e] -> X[t + T e], e < 8, n <= 8 T <= 2048 points in 2 n of LDS.
// Called by every thread; another barrier before lds is written again.
template <bool INV>
__device__ __forceinline__ void sub_fft(cplx* v, cplx* lds, const int T, int t, int n,
                                        const cplx* __restrict__ tw) {
#pragma unroll
  for (int e = 0; e < 8; ++e)
    if (t + T * e < n) lds[t + T * e] = v[e];
  __syncthreads();
  const int odd = (31 - __clz(n)) & 3;  // log2 of the first radix, 0: 16
  cplx* src = lds;
  cplx* dst = lds + n;
  const int passes = T <= 32 ? 2 : 3;  // the same for every ring of the workgroup
  int Ns = 1;
#pragma unroll 1
  for (int pass = 0; pass < passes; ++pass) {
    if (Ns < n) {
      const int lr = pass == 0 && odd ? odd : 4;
      if (lr == 4)
        sub_pass<16, INV>(src, dst, T, t, n, Ns, tw);
      else if (lr == 3)
        sub_pass<8, INV>(src, dst, T, t, n, Ns, tw);
      else if (lr == 2)
        sub_pass<4, INV>(src, dst, T, t, n, Ns, tw);
      else
        sub_pass<2, INV>(src, dst, T, t, n, Ns, tw);
      cplx* x = src;
      src = dst;
      dst = x;
      Ns <<= lr;
    }
    __syncthreads();
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = t + T * e < n ? src[t + T * e] : cplx{0.0, 0.0};
}

__device__ __forceinline__ void sub_fwd(const RingFwdArgs& a, const RingSeg& seg, int paired,
                                        void* raw) {
  const int T = 1 << ((seg.body & (kPow2Body - 1)) - 4);
  const RingOf ring(T, a.jobs, seg, paired, a.batch, raw);
  const RingJob& job = ring.job;
  const int n = job.nphi, t = ring.t;
  const cplx* __restrict__ phase = a.chirp_pool + job.chirp_off;
  cplx v[8];
  load_pixels<8>(T, v, a, job, t, ring.b0, paired, ring.two);
  sub_fft<false>(v, ring.lds, T, t, n, a.chirp_pool);
  const double w = (a.apply_weight ? job.weight : 1.0) * ring_scale(a.norm_mode, n);
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = {w * v[e].x, w * v[e].y};
  const bool ph = ring_phase(a.apply_phase, job);
  residues_to_lds<8>(T, v, ring.lds, n, t, paired, [&](int e, cplx z) {
    return ph ? cmul(z, phase[t + T * e]) : z;
  });
  if (ring.valid) store_columns(T, ring.lds, a, job, t, ring.b0, ring.two, ph);
}

__device__ __forceinline__ void sub_inv(const RingInvArgs& a, const RingSeg& seg, int paired,
                                        void* raw) {
  const int T = 1 << ((seg.body & (kPow2Body - 1)) - 4);
  const RingOf ring(T, a.jobs, seg, paired, a.batch, raw);
  const RingJob& job = ring.job;
  const int n = job.nphi, t = ring.t;
  const cplx* __restrict__ phase = a.chirp_pool + job.chirp_off;
  const FoldIn in(a, job, ring.b0, ring.two);
  cplx v[8], f[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int p = t + T * e;
    f[e] = in.ph && p < n ? phase[p] : cplx{1.0, 0.0};
  }
  in.residues(T, v, ring.lds, t);
  const double w = (a.apply_weight ? job.weight : 1.0) * ring_scale(a.norm_mode, n);
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = tmul<true>(cplx{w * v[e].x, w * v[e].y}, f[e]);
  __syncthreads();  // the partial sums are read
  sub_fft<true>(v, ring.lds, T, t, n, a.chirp_pool);
  if (ring.valid) store_pixels<8>(T, v, a, job, t, ring.b0, paired, ring.two, in.herm);
}

// e^{-i pi (t + T e) / N} of a power-of-two ring: e^{-i pi t / N} from the
// twiddle table times e^{-i pi e / 16}
template <int LOGN>
__device__ __forceinline__ cplx pow2_phase(cplx base, int e) {
  return cmul(base, cplx{kW32[e][0], kW32[e][1]});
}

// direct, real pairs: the columns m in [0, n / 2)
template <int LOGN>
__device__ __forceinline__ void pow2_fwd(const RingFwdArgs& a, const RingSeg& seg, int paired,
                                         void* raw) {
  typedef Pow2Shape<LOGN> P;
  constexpr int T = P::T, N = P::N;
  const RingOf ring(T, a.jobs, seg, paired, a.batch, raw);
  const RingJob& job = ring.job;
  cplx* lds = ring.lds;
  const int t = ring.t;
  const cplx* __restrict__ tw = a.chirp_pool;
  cplx v[16];
  load_pixels<16>(T, v, a, job, t, ring.b0, paired, ring.two);
  pow2_fft<LOGN, false>(v, lds, t, tw);
  const double w = (a.apply_weight ? job.weight : 1.0) * ring_scale(a.norm_mode, N);
#pragma unroll
  for (int e = 0; e < 16; ++e) v[e] = {w * v[e].x, w * v[e].y};
  const bool ph = ring_phase(a.apply_phase, job);
  const cplx base = load_tw16(tw, 2 * T, t).w;
  if (seg.direct && paired) {
    // X and Y of the residues below N / 2 from z and the upper half's z'
    __syncthreads();
#pragma unroll
    for (int e = 8; e < 16; ++e) lds[T * e + t] = v[e];
    __syncthreads();
    if (!ring.valid) return;
    cplx* d0 = a.out + ring.b0 * a.out_map_stride + (int64_t)job.row * a.ncol;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int p = t + T * e;
      const cplx z = v[e], zc = p == 0 ? z : lds[N - p];
      cplx X = {0.5 * (z.x + zc.x), 0.5 * (z.y - zc.y)};
      cplx Y = {0.5 * (z.y + zc.y), -0.5 * (z.x - zc.x)};
      if (ph) {
        const cplx f = pow2_phase<LOGN>(base, e);
        X = cmul(X, f);
        Y = cmul(Y, f);
      }
      if (p < a.ncol) {
        d0[p] = X;
        if (ring.two) d0[a.out_map_stride + p] = Y;
      }
    }
    return;
  }
  if (seg.direct) {
    if (ph) {
#pragma unroll
      for (int e = 0; e < 16; ++e) v[e] = cmul(v[e], pow2_phase<LOGN>(base, e));
    }
    if (ring.valid) store_direct<16>(T, v, a, job, t, ring.b0, ph);
    return;
  }
  residues_to_lds<16>(T, v, lds, N, t, paired, [&](int e, cplx z) {
    return ph ? cmul(z, pow2_phase<LOGN>(base, e)) : z;
  });
  if (ring.valid) store_columns(T, lds, a, job, t, ring.b0, ring.two, ph);
}

template <int LOGN>
__device__ __forceinline__ void pow2_inv(const RingInvArgs& a, const RingSeg& seg, int paired,
                                         void* raw) {
  typedef Pow2Shape<LOGN> P;
  constexpr int T = P::T, N = P::N;
  const RingOf ring(T, a.jobs, seg, paired, a.batch, raw);
  const RingJob& job = ring.job;
  cplx* lds = ring.lds;
  const int t = ring.t;
  const cplx* __restrict__ tw = a.chirp_pool;
  const FoldIn in(a, job, ring.b0, ring.two);
  cplx v[16];
  in.owned<16>(T, v, t);
  const double w = (a.apply_weight ? job.weight : 1.0) * ring_scale(a.norm_mode, N);
#pragma unroll
  for (int e = 0; e < 16; ++e) v[e] = {w * v[e].x, w * v[e].y};
  if (in.ph) {
    const cplx base = load_tw16(tw, 2 * T, t).w;
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = tmul<true>(v[e], pow2_phase<LOGN>(base, e));
  }
  pow2_fft<LOGN, true>(v, lds, t, tw);
  if (ring.valid) store_pixels<16>(T, v, a, job, t, ring.b0, paired, ring.two, in.herm);
}

// Runs the body of this block's segment: those whose rings of T threads fit WG.
template <int WG, int DIR, typename Args>
__device__ __forceinline__ void ring_body(const Args& a, const RingSeg& seg, int paired,
                                          void* raw) {
#define S2H_BLUE(L)                                                             \
  case L:                                                                       \
    if constexpr (Shape<L>::T <= WG && Shape<L>::T * kSpan >= WG) {             \
      if constexpr (DIR == 0) blue_fwd<L>(a, seg, paired, raw);                 \
      else blue_inv<L>(a, seg, paired, raw);                                    \
    }                                                                           \
    break;
#define S2H_POW2(L)                                                             \
  case kPow2Body + L:                                                           \
    if constexpr (Pow2Shape<L>::T <= WG && Pow2Shape<L>::T * kSpan >= WG) {     \
      if constexpr (DIR == 0) pow2_fwd<L>(a, seg, paired, raw);                 \
      else pow2_inv<L>(a, seg, paired, raw);                                    \
    }                                                                           \
    break;
  constexpr int kSpan = WG == 64 ? 16 : 8;
  if (seg.body >= kSubBody) {
    if constexpr (DIR == 0) sub_fwd(a, seg, paired, raw);
    else sub_inv(a, seg, paired, raw);
    return;
  }
  switch (seg.body) {
    S2H_BLUE(6) S2H_BLUE(7) S2H_BLUE(8) S2H_BLUE(9) S2H_BLUE(10) S2H_BLUE(11) S2H_BLUE(12)
    S2H_BLUE(13)
    S2H_POW2(6) S2H_POW2(7) S2H_POW2(8) S2H_POW2(9) S2H_POW2(10) S2H_POW2(11) S2H_POW2(12)
    default: break;
  }
#undef S2H_BLUE
#undef S2H_POW2
}

__device__ __forceinline__ RingSeg seg_of_block(const RingSegs& g) {
  int i = 0;
  while (i + 1 < g.n && (int)blockIdx.x >= g.s[i + 1].block0) ++i;
  return g.s[i];
}

}  // namespace

// gridDim.y: maps (complex input) or map pairs (real input, `paired`).
template <int WG>
__global__ void __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(2)))
ring_reg_fwd_kernel(RingFwdArgs a, RingSegs g, int paired) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  ring_body<WG, 0>(a, seg_of_block(g), paired, lds_raw);
  if (a.pad_rows && blockIdx.x == gridDim.x - 1) {
    const int maps = paired ? 2 : 1;
    for (int b = maps * blockIdx.y; b < min(a.batch, maps * ((int)blockIdx.y + 1)); ++b) {
      cplx* pad = a.out + (int64_t)b * a.out_map_stride + (int64_t)a.pad_row0 * a.ncol;
      for (int i = threadIdx.x; i < a.pad_rows * a.ncol; i += WG) pad[i] = {0.0, 0.0};
    }
  }
}
template <int WG>
__global__ void __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(2)))
ring_reg_inv_kernel(RingInvArgs a, RingSegs g, int paired) {
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  ring_body<WG, 1>(a, seg_of_block(g), paired, lds_raw);
}

// ------------------------------------------------------------------ launchers
namespace {

// Whether every residue of an n-point ring has at most one column.
bool ring_direct(const RingFwdArgs& a, int n, int paired) {
  if (a.out_single || a.zero_neg_2L) return false;
  if (paired) return a.m_first == 0 && a.ncol <= n / 2;
  return a.ncol <= n && a.m_first <= 0 && -a.m_first < n;
}

int shape_lds(int logm) { return (1 << logm) + (logm <= 9 ? (1 << logm) / 8 + 32 : 0); }
int seg_threads(const RingSeg& s) { return 1 << ((s.body & (kPow2Body - 1)) - 4); }

// The segments of a job set, longest convolutions first.
RingSegs ring_segs(const JobSet& js) {
  RingSegs g{};
  int j0 = js.n_pow2;
  for (int c = kBlueClasses - 1; c >= 0; --c) {
    const int lg = c + kBlueLogMin;
    if (js.blue[c]) g.s[g.n++] = RingSeg{lg, j0, js.blue[c], 0, 0, shape_lds(lg)};
    j0 += js.blue[c];
    if (js.sub[c]) g.s[g.n++] = RingSeg{kSubBody + lg, j0, js.sub[c], 0, 0, shape_lds(lg)};
    j0 += js.sub[c];
  }
  if (js.n_pow2)
    g.s[g.n++] = RingSeg{kPow2Body + js.log_pow2, 0, js.n_pow2, 0, 0, 1 << js.log_pow2};
  return g;
}

// Launches segments [i0, i1) together at the workgroup size of the largest.
template <int DIR, typename Args>
hipError_t launch_segs(const Args& a, const RingSegs& all, int i0, int i1, unsigned gy, int paired,
                       hipStream_t s) {
  RingSegs g{};
  int wg = 64, lds = 0, blocks = 0;
  for (int i = i0; i < i1; ++i) wg = std::max(wg, seg_threads(all.s[i]));
  for (int i = i0; i < i1; ++i) {
    RingSeg q = all.s[i];
    const int rings = wg / seg_threads(q);
    q.block0 = blocks;
    blocks += (q.count + rings - 1) / rings;
    lds = std::max(lds, rings * q.lds_ring * (int)sizeof(cplx));
    g.s[g.n++] = q;
  }
  const dim3 grid(blocks, gy);
#define S2H_LAUNCH(WG)                                                                     \
  if constexpr (DIR == 0)                                                                  \
    hipLaunchKernelGGL((ring_reg_fwd_kernel<WG>), grid, dim3(WG), lds, s, a, g, paired);   \
  else                                                                                     \
    hipLaunchKernelGGL((ring_reg_inv_kernel<WG>), grid, dim3(WG), lds, s, a, g, paired);
  switch (wg) {
    case 64: S2H_LAUNCH(64) break;
    case 128: S2H_LAUNCH(128) break;
    case 256: S2H_LAUNCH(256) break;
    default: S2H_LAUNCH(512) break;
  }
#undef S2H_LAUNCH
  return hipGetLastError();
}

// One launch for a whole ragged grid while it has at most kMergeBlocks
// workgroups, else one per segment (each at its own workgroup size).  Together
// against one launch per segment: nside 512, one map 44 against 75 us, four
// maps 90 against 129, nside 1024, 16 maps (25 600 workgroups) 1434 against 1330.
constexpr int kMergeBlocks = 16384;
template <int DIR, typename Args>
hipError_t launch_rings(const Args& a, const RingSegs& g, unsigned gy, int paired, hipStream_t s) {
  int wg = 64, narrow = 512;
  int64_t threads = 0;
  for (int i = 0; i < g.n; ++i) {
    wg = std::max(wg, seg_threads(g.s[i]));
    narrow = std::min(narrow, seg_threads(g.s[i]));
    threads += (int64_t)g.s[i].count * seg_threads(g.s[i]);
  }
  int lds = 0;
  for (int i = 0; i < g.n; ++i)
    lds = std::max(lds, wg / seg_threads(g.s[i]) * g.s[i].lds_ring * (int)sizeof(cplx));
  const bool together = threads * gy <= (int64_t)kMergeBlocks * wg &&
                        narrow * (wg == 64 ? 16 : 8) >= wg && lds <= kRingLdsMax;
  if (together) return launch_segs<DIR>(a, g, 0, g.n, gy, paired, s);
  for (int i = 0, i1; i < g.n; i = i1) {
    // the powers of two among the rings of one convolution length go with them
    for (i1 = i + 1; i1 < g.n && g.s[i1].body == kSubBody + g.s[i].body;) ++i1;
    const hipError_t e = launch_segs<DIR>(a, g, i, i1, gy, paired, s);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// real pairs: two maps share a complex transform
bool fwd_paired(const RingFwdArgs& a) { return !a.f_complex || a.real_only_all; }
// float64 maps only: complex128 ones stay alone.  In a pair the smaller map takes the
// rounding of the larger one (a partner 1e8 times larger leaves 1e-8 of it), and a NaN
// or infinity reaches both.  What it costs, HEALPix real, 4 maps: nside 256, L = 512 120
// us instead of 113 in pairs, nside 512, L = 1024 446 instead of 417.
bool inv_paired(const RingInvArgs& a) { return a.herm_mode == 1 && !a.f_complex; }
unsigned grid_y(int batch, int paired) { return (unsigned)(paired ? (batch + 1) / 2 : batch); }

}  // namespace

hipError_t launch_ring_fft_forward(const RingFwdArgs& a0, const JobSet& js, int batch,
                                   hipStream_t s) {
  if (batch == 0 || js.n_pow2 + js.n_rest == 0) return hipSuccess;
  RingFwdArgs a = a0;
  a.jobs = js.jobs;
  a.batch = batch;
  const int paired = fwd_paired(a) ? 1 : 0;
  RingSegs g = ring_segs(js);
  for (int i = 0; i < g.n; ++i) {
    RingSeg& q = g.s[i];
    if (q.body & kPow2Body) {
      q.direct = ring_direct(a, 1 << js.log_pow2, paired);
      if (!q.direct && paired) q.lds_ring *= 2;  // the residues of both maps
    } else {
      q.direct = !paired && !a.apply_phase && ring_direct(a, js.min_rest, 0);
    }
  }
  return launch_rings<0>(a, g, grid_y(batch, paired), paired, s);
}

hipError_t launch_ring_fft_inverse(const RingInvArgs& a0, const JobSet& js, int batch,
                                   hipStream_t s) {
  if (batch == 0 || js.n_pow2 + js.n_rest == 0) return hipSuccess;
  RingInvArgs a = a0;
  a.jobs = js.jobs;
  a.batch = batch;
  const int paired = inv_paired(a) ? 1 : 0;
  return launch_rings<1>(a, ring_segs(js), grid_y(batch, paired), paired, s);
}

hipError_t allow_large_lds_rings() {
  const int bytes = kRingLdsMax;
  const void* fns[] = {(const void*)ring_reg_fwd_kernel<64>,  (const void*)ring_reg_fwd_kernel<128>,
                       (const void*)ring_reg_fwd_kernel<256>, (const void*)ring_reg_fwd_kernel<512>,
                       (const void*)ring_reg_inv_kernel<64>,  (const void*)ring_reg_inv_kernel<128>,
                       (const void*)ring_reg_inv_kernel<256>, (const void*)ring_reg_inv_kernel<512>};
  for (const void* f : fns) {
    const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace s2h
