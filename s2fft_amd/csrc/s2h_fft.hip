// Bluestein chirp tables, the DFT over gamma of the Wigner transforms and the
// reality fill of Wigner coefficients.  (The ring FFTs live in
// s2h_ring_fft.hip.)
#include "s2h_fft_lds.h"
#include "s2h_kernels.h"

namespace s2h {

constexpr int kFftMax = kMaxConvLen;

// The chirp pool's tables of one length per workgroup (ChirpEntry).
__global__ void __launch_bounds__(kThreads) chirp_setup_kernel(const ChirpEntry* entries,
                                                               cplx* pool) {
  extern __shared__ double smem[];
  const ChirpEntry en = entries[blockIdx.x];
  const int n = en.n, M = en.M;
  double* re = smem;
  double* im = smem + M;
  if (blockIdx.x == 0) {
    for (int j = threadIdx.x; j < kRingTwiddles; j += kThreads) {
      const TwiddleOf w = ring_twiddle(j);
      pool[j] = expi_pi(-2 * w.num, w.N);
    }
  }
  if (en.ring == 2) {
    for (int k = threadIdx.x; k < n; k += kThreads) pool[en.off + k] = expi_pi(-k, n);
    return;
  }
  for (int j = threadIdx.x; j < M; j += kThreads) {
    cplx v = {0.0, 0.0};
    if (j < n)
      v = expi_pi((int64_t)j * j, n);
    else if (j > M - n)
      v = expi_pi((int64_t)(M - j) * (M - j), n);
    re[j] = v.x;
    im[j] = v.y;
  }
  __syncthreads();
  fft_mixed<kFftMax, true>(re, im, M, -1);
  cplx* dst = pool + en.off;
  const double s = 1.0 / M;
  for (int j = threadIdx.x; j < M; j += kThreads)
    dst[en.ring ? blue_place(j, M) : j] = {re[j] * s, im[j] * s};
  if (!en.ring) return;
  for (int k = threadIdx.x; k < n; k += kThreads) {
    dst[M + k] = expi_pi(-(int64_t)k * k, n);
    dst[M + n + k] = expi_pi(-k, n);
  }
}

// Direct DFT over gamma (G = 2N-1 <= 15 points) for every (beta, alpha)
// sample.  Modes: 0 forward from complex f, 2 forward from real f (both give
// fban[k], k = n + N-1, n in [-(N-1), N-1]), 1 inverse to complex f from all
// 2N-1 rows, 3 inverse to real f from the rows n >= 0 only (Hermitian),
// 4 Re of the inverse sum over the rows n >= 0 only (the adjoint of mode 2
// restricted to n >= 0: Re sum_{n >= 0} x_n e^{+2 pi i n g / G}), 5 the
// adjoint of mode 3: from real f, the N rows n >= 0 of the forward sum, the
// rows n >= 1 doubled.
// A sample's inputs sit in registers (N a template parameter), the G roots of
// unity in LDS; blockIdx.y takes every gridDim.y-th output.  Bound by its
// launch at the sizes of a Wigner transform: MW L = 64, N = 4 22 -> 3.4 us (before,
// a root evaluated for every term and the inputs in scratch memory).
template <int N>
__global__ void __launch_bounds__(kThreads) gamma_dft_kernel(int64_t npix, int mode, double scale,
                                                             const void* in_, void* out_) {
  constexpr int G = 2 * N - 1;
  __shared__ cplx w[G];  // e^{2 pi i j / G}
  if (threadIdx.x < G) w[threadIdx.x] = expi_pi(2 * (int64_t)threadIdx.x, G);
  __syncthreads();
  const int64_t p = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (p >= npix) return;
  cplx x[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    x[g] = {0.0, 0.0};
    if (mode == 2 || mode == 5)
      x[g].x = static_cast<const double*>(in_)[(int64_t)g * npix + p];
    else if (mode < 2 || g < N)  // modes 3, 4: the N rows n >= 0
      x[g] = static_cast<const cplx*>(in_)[(int64_t)g * npix + p];
  }
  const auto wrap = [](int j) { return j >= G ? j - G : j; };
  const int nout = mode == 5 ? N : G;
  for (int k = blockIdx.y; k < nout; k += gridDim.y) {
    cplx* out = static_cast<cplx*>(out_) + (int64_t)k * npix + p;
    if (mode == 3 || mode == 4) {  // sample g = k from x[n]
      const double wn = mode == 3 ? 2.0 : 1.0;
      double acc = x[0].x;
      int j = 0;
#pragma unroll
      for (int n = 1; n < N; ++n) {
        j = wrap(j + k);
        acc += wn * cmul(x[n], w[j]).x;
      }
      static_cast<double*>(out_)[(int64_t)k * npix + p] = acc * scale;
      continue;
    }
    // row n from the samples: root -n g; sample k from the rows: root (i - (N - 1)) k
    const int n = mode == 5 ? k : k - (N - 1);
    const int step = mode == 1 ? k : n > 0 ? G - n : -n;
    int j = mode == 1 ? (N * k) % G : 0;  // -(N - 1) = N modulo G
    cplx acc = {0.0, 0.0};
#pragma unroll
    for (int i = 0; i < G; ++i) {
      acc = cadd(acc, cmul(x[i], w[j]));
      j = wrap(j + step);
    }
    const double f = mode == 5 && n ? 2.0 * scale : scale;
    *out = {acc.x * f, acc.y * f};
  }
}

// flmn[N-1-n][l][L-1+m] = (-1)^(m+n) conj(flmn[N-1+n][l][L-1-m]) for n >= 1
// (s2fft/transforms/wigner.py:523-526).
__global__ void __launch_bounds__(kThreads) wigner_fill_kernel(cplx* flmn, int L, int N) {
  const int n = blockIdx.z + 1;
  const int l = blockIdx.y;
  const int c = blockIdx.x * kThreads + threadIdx.x;
  if (c >= 2 * L - 1) return;
  const int m = c - (L - 1);
  const int64_t plane = (int64_t)L * (2 * L - 1);
  const cplx v = flmn[(N - 1 + n) * plane + (int64_t)l * (2 * L - 1) + (L - 1 - m)];
  const double s = ((m + n) & 1) ? -1.0 : 1.0;
  flmn[(N - 1 - n) * plane + (int64_t)l * (2 * L - 1) + c] = {s * v.x, -s * v.y};
}

// Adjoint of wigner_fill_kernel for a real-valued loss: the cotangent of
// each filled entry flmn[N-1-n][l][L-1+m] flows back to its source
// flmn[N-1+n][l][L-1-m] as (-1)^(m+n) conj(.): g[N-1+n][l][L-1+m] +=
// (-1)^(m+n) conj(g[N-1-n][l][L-1-m]) for n >= 1 (in place).
__global__ void __launch_bounds__(kThreads) wigner_fill_adjoint_kernel(cplx* g, int L, int N) {
  const int n = blockIdx.z + 1;
  const int l = blockIdx.y;
  const int c = blockIdx.x * kThreads + threadIdx.x;
  if (c >= 2 * L - 1) return;
  const int m = c - (L - 1);
  const int64_t plane = (int64_t)L * (2 * L - 1);
  const cplx v = g[(N - 1 - n) * plane + (int64_t)l * (2 * L - 1) + (L - 1 - m)];
  const double s = ((m + n) & 1) ? -1.0 : 1.0;
  cplx* o = g + (N - 1 + n) * plane + (int64_t)l * (2 * L - 1) + c;
  o->x += s * v.x;
  o->y -= s * v.y;
}

// ------------------------------------------------------------ launchers
hipError_t launch_chirp_setup(const ChirpEntry* entries, cplx* pool, int count, int max_conv,
                              hipStream_t s) {
  if (count == 0) return hipSuccess;
  const size_t lds = 2 * sizeof(double) * (size_t)max_conv;
  hipLaunchKernelGGL(chirp_setup_kernel, dim3(count), dim3(kThreads), lds, s, entries, pool);
  return hipGetLastError();
}

hipError_t launch_gamma_dft(int N, int64_t npix, int mode, double scale, const void* in,
                            void* out, hipStream_t s) {
  if (npix == 0) return hipSuccess;
  const int64_t blocks = (npix + kThreads - 1) / kThreads;
  // few samples: one output per thread
  const dim3 grid((unsigned)blocks, blocks < 512 ? 2 * N - 1 : 1), block(kThreads);
  switch (N) {
#define S2H_GAMMA(n)                                                                              \
  case n:                                                                                         \
    hipLaunchKernelGGL(gamma_dft_kernel<n>, grid, block, 0, s, npix, mode, scale, in, out);       \
    break;
    S2H_GAMMA(1) S2H_GAMMA(2) S2H_GAMMA(3) S2H_GAMMA(4)
    S2H_GAMMA(5) S2H_GAMMA(6) S2H_GAMMA(7) S2H_GAMMA(8)
#undef S2H_GAMMA
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_wigner_fill(cplx* flmn, int L, int N, hipStream_t s) {
  if (N < 2) return hipSuccess;
  hipLaunchKernelGGL(wigner_fill_kernel, dim3((2 * L - 1 + kThreads - 1) / kThreads, L, N - 1),
                     dim3(kThreads), 0, s, flmn, L, N);
  return hipGetLastError();
}

hipError_t allow_large_lds() {
  hipError_t e = allow_large_lds_rings();
  if (e == hipSuccess) e = allow_large_lds_alias();
  if (e == hipSuccess) e = allow_large_lds_lat();
  if (e != hipSuccess) return e;
  const int bytes = 2 * sizeof(double) * kFftMax;
  return hipFuncSetAttribute((const void*)chirp_setup_kernel,
                             hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
}

}  // namespace s2h

namespace s2h {
__global__ void __launch_bounds__(kThreads) real_to_complex_kernel(const double* in, cplx* out,
                                                                   int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i < n) out[i] = {in[i], 0.0};
}

hipError_t launch_real_to_complex(const double* in, cplx* out, int64_t n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(real_to_complex_kernel, dim3((unsigned)((n + kThreads - 1) / kThreads)),
                     dim3(kThreads), 0, s, in, out, n);
  return hipGetLastError();
}

hipError_t launch_wigner_fill_adjoint(cplx* g, int L, int N, hipStream_t s) {
  if (N < 2) return hipSuccess;
  hipLaunchKernelGGL(wigner_fill_adjoint_kernel,
                     dim3((2 * L - 1 + kThreads - 1) / kThreads, L, N - 1), dim3(kThreads), 0, s,
                     g, L, N);
  return hipGetLastError();
}
}  // namespace s2h
