// Stored Wigner-d tables and the dense contractions of the precompute path.
//
// The reference's precompute path builds a kernel K[t][l][m] =
// d^l_{m,-spin}(theta_t) sqrt((2l+1)/4pi) (x forward quadrature weights, x
// HEALPix ring phases) once (s2fft/precompute_transforms/construct.py:16-161)
// and applies it as einsum "tlm,tm->lm" (forward) or "tlm,lm->tm" (inverse)
// (s2fft/precompute_transforms/spherical.py:87-149, 314-380); its
// compute_all_slices (s2fft/recursions/price_mcewen.py:377-643) returns the
// bare d-values dl[L-1+m][t][l].  Both tables come from one builder here: a
// lane per (m, theta) walks the l-recursion of the latitudinal kernels with a
// plan's own coefficient tables and writes every l of its (m, theta) through
// arbitrary strides; for the kernel layout [t][l][m] consecutive lanes (m)
// store consecutive addresses.  The contractions are FP64 VALU (one
// small product per m, m the fastest index), bound by the table reads, which is
// what this path trades for its O(L^3) memory.
#include "s2h_fft_lds.h"
#include "s2h_kernels.h"
#include "s2h_lat_common.h"

namespace s2h {

namespace {

constexpr int kPcRows = 4;    // rows per lane in the contractions
constexpr int kPcM = 16;      // m values per wave
constexpr int kPcWaves = 16;  // waves per workgroup at most
constexpr int kRescale = 8;  // steps between rescale checks

__global__ void __launch_bounds__(kThreads) dtable_kernel(DTableArgs a) {
  const int mi = blockIdx.x * kThreads + threadIdx.x;
  const int t = blockIdx.y;
  if (mi >= a.nm) return;
  const int m = a.m_lo + mi;
  const int am = m < 0 ? -m : m;
  const double th = a.theta[t];
  double x = cos(th), c2 = cos(0.5 * th), s2 = sin(0.5 * th);
  // the poles exactly (cos(pi/2) rounds to 6e-17, not 0): d^l_{mn}(0) and
  // d^l_{mn}(pi) vanish unless m = n or m = -n
  if (fabs(th) < 1e-14) {
    x = 1.0;
    c2 = 1.0;
    s2 = 0.0;
  } else if (fabs(th - M_PI) < 1e-14) {
    x = -1.0;
    c2 = 0.0;
    s2 = 1.0;
  }
  const MStart st = a.mstart[mi];
  const Coef* __restrict__ cf = a.coef + (int64_t)am * a.L;
  const double bsign = m < 0 ? -1.0 : 1.0;
  double fac = a.scale * (a.wt ? a.wt[t] : 1.0);
  double pre = 0.0, pim = 0.0;  // e^{i phase_sign m phi0}
  if (a.cplx) {
    const double ang = a.phi0 ? a.phase_sign * (double)m * a.phi0[t] : 0.0;
    sincos(ang, &pim, &pre);
  }
  const int64_t base = (int64_t)mi * a.sm + (int64_t)t * a.st;
  const auto put = [&](int l, double v) {
    const int64_t o = base + (int64_t)l * a.sl;
    if (a.cplx) {
      cplx* out = static_cast<cplx*>(a.out);
      out[o] = {v * pre, v * pim};
    } else {
      static_cast<double*>(a.out)[o] = v;
    }
  };
  const int l0 = st.ell0 < a.L ? st.ell0 : a.L;
  for (int l = 0; l < l0; ++l) put(l, 0.0);
  double d, dm1 = 0.0;
  int lscale;
  lat::start_value(st, c2, s2, d, lscale);
  for (int l = l0; l < a.L; ++l) {
    const lat::ChunkCoef c = lat::finish_coef(cf[l], bsign);  // d: e_l, d_l = sigma_l e_l
    put(l, lscale == 0 ? c.c * d * fac * (a.lw ? a.lw[l] : 1.0) : 0.0);
    const double dn = lat::rec_step_unit(c, x, d, dm1);
    dm1 = d;
    d = dn;
    if (((l - l0) % kRescale) == kRescale - 1) lat::rescale(d, dm1, lscale);
  }
}

template <typename K>
__device__ __forceinline__ cplx kval(const K* k, int64_t i);
template <>
__device__ __forceinline__ cplx kval<double>(const double* k, int64_t i) {
  return {k[i], 0.0};
}
template <>
__device__ __forceinline__ cplx kval<cplx>(const cplx* k, int64_t i) {
  return k[i];
}

// acc += k x, k real or complex
__device__ __forceinline__ void pc_fma(const double*, cplx k, cplx x, cplx& acc) {
  acc = {fma(k.x, x.x, acc.x), fma(k.x, x.y, acc.y)};
}
__device__ __forceinline__ void pc_fma(const cplx*, cplx k, cplx x, cplx& acc) {
  acc = {fma(k.x, x.x, fma(-k.y, x.y, acc.x)), fma(k.x, x.y, fma(k.y, x.x, acc.y))};
}

// out[b][o][mi] = scale sum_c K(o, c, mi) x[b][c][mi]: forward o = l, c = theta,
// inverse o = theta, c = l.  One product per m, with m the fastest index of every
// array: lanes hold 16 adjacent m by 4 rows o, so that loads of K and x are
// 256-byte runs and the four rows share those of x; kRows further rows and NB
// maps per lane in registers use each loaded value 4 times.  The waves of a
// workgroup take c in turn and are added up through LDS, in a fixed order.
// Bound by the loads, which every value passes 4 times on the way from L2: 4 maps
// and 4 rows per lane are the balance, as K and x weigh the same then.  Measured:
// HEALPix nside 64, L = 128, real, 16 maps (a kernel of 67 MB, 268 million complex
// multiply-adds): 530 -> 26 us (a thread per output and 8 maps, one load at a time).
struct PcGemm {
  const void* k;
  int64_t k_row, k_step;    // strides of o and c
  const cplx* x;
  int64_t x_map, x_step;    // strides of maps and c
  cplx* out;
  int64_t o_map, o_row;     // strides of maps and o
  int rows, steps, nm, batch;
  int mirror;               // real maps: also out[-m] = (-1)^m conj(out[m])
  double scale;
};

template <typename K, int NB>
__global__ void __launch_bounds__(64 * kPcWaves) pc_kernel(PcGemm a) {
  extern __shared__ __attribute__((aligned(16))) unsigned char pc_raw[];
  cplx* red = reinterpret_cast<cplx*>(pc_raw);  // [wave][map][lane]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwave = blockDim.x >> 6;
  // blocks i, i + 8, ... run on one XCD: the map chunks of a tile (the same K) in
  // turn, and of the tiles every eighth, with the same m where the m tiles divide
  const int chunks = (a.batch + NB - 1) / NB, mtiles = (a.nm + kPcM - 1) / kPcM;
  const int otiles = (a.rows + 4 * kPcRows - 1) / (4 * kPcRows);
  const int j = blockIdx.x >> 3;
  const int tile = j / chunks * 8 + (blockIdx.x & 7), b0 = j % chunks * NB;
  if (tile >= mtiles * otiles) return;
  const int m0 = tile % mtiles * kPcM, o0 = tile / mtiles * 4 * kPcRows;
  // past the ends: the last m, row and map again, not stored
  const int mi = min(m0 + (lane & 15), a.nm - 1), os = o0 + (lane >> 4);
  const K* __restrict__ kk = static_cast<const K*>(a.k) + mi;
  const cplx* __restrict__ xx = a.x + mi;
  int64_t ko[kPcRows];
#pragma unroll
  for (int r = 0; r < kPcRows; ++r) ko[r] = min(os + 4 * r, a.rows - 1) * a.k_row;
  cplx acc[kPcRows][NB];
#pragma unroll
  for (int r = 0; r < kPcRows; ++r)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[r][b] = {0.0, 0.0};
#pragma unroll 2
  for (int c = wave; c < a.steps; c += nwave) {
    cplx k[kPcRows], x[NB];
#pragma unroll
    for (int r = 0; r < kPcRows; ++r) k[r] = kval<K>(kk, ko[r] + c * a.k_step);
#pragma unroll
    for (int b = 0; b < NB; ++b) x[b] = xx[min(b0 + b, a.batch - 1) * a.x_map + c * a.x_step];
#pragma unroll
    for (int r = 0; r < kPcRows; ++r)
#pragma unroll
      for (int b = 0; b < NB; ++b) pc_fma(kk, k[r], x[b], acc[r][b]);
  }
#pragma unroll
  for (int r = 0; r < kPcRows; ++r) {
#pragma unroll
    for (int b = 0; b < NB; ++b) red[(wave * NB + b) * 64 + lane] = acc[r][b];
    __syncthreads();
    for (int e = threadIdx.x; e < 64 * NB; e += blockDim.x) {
      cplx s = red[e];
      for (int w = 1; w < nwave; ++w) s = cadd(s, red[w * 64 * NB + e]);
      const int b = b0 + (e >> 6), o = o0 + ((e & 63) >> 4) + 4 * r, m = m0 + (e & 15);
      if (b < a.batch && o < a.rows && m < a.nm) {
        cplx* out = a.out + (int64_t)b * a.o_map + o * a.o_row;
        s = {a.scale * s.x, a.scale * s.y};
        out[m] = s;
        if (a.mirror && m > 0) out[-m] = m & 1 ? cplx{-s.x, s.y} : cplx{s.x, -s.y};
      }
    }
    __syncthreads();
  }
}

}  // namespace

hipError_t launch_dtable(const DTableArgs& a, hipStream_t s) {
  if (a.nm == 0 || a.T == 0 || a.L == 0) return hipSuccess;
  hipLaunchKernelGGL(dtable_kernel, dim3((a.nm + kThreads - 1) / kThreads, a.T), dim3(kThreads),
                     0, s, a);
  return hipGetLastError();
}

namespace {

template <typename K, int NB>
hipError_t launch_pc_nb(const PcGemm& a, hipStream_t s) {
  const int tiles = (a.nm + kPcM - 1) / kPcM * ((a.rows + 4 * kPcRows - 1) / (4 * kPcRows));
  const int chunks = (a.batch + NB - 1) / NB;
  // at least four steps per wave
  int waves = 1;
  while (waves < kPcWaves && 8 * waves <= a.steps) waves *= 2;
  hipLaunchKernelGGL((pc_kernel<K, NB>), dim3((tiles + 7) / 8 * 8 * chunks), dim3(64 * waves),
                     sizeof(cplx) * 64 * NB * waves, s, a);
  return hipGetLastError();
}

// The fewest maps per lane that hold the batch, up to 4: a lone map with 4 would
// load and multiply the same map 4 times.  Whole forward, HEALPix nside 64, 1 / 2 / 16
// maps: 132 / 194 / 631 -> 31 / 31 / 41 us, inverse 88 / 122 / 413 -> 43 / 50 / 68 us.
hipError_t launch_pc(const PcGemm& a, bool kernel_complex, hipStream_t s) {
  if (a.batch == 0 || a.nm == 0 || a.rows == 0) return hipSuccess;
  if (kernel_complex) {
    if (a.batch == 1) return launch_pc_nb<cplx, 1>(a, s);
    if (a.batch == 2) return launch_pc_nb<cplx, 2>(a, s);
    return launch_pc_nb<cplx, 4>(a, s);
  }
  if (a.batch == 1) return launch_pc_nb<double, 1>(a, s);
  if (a.batch == 2) return launch_pc_nb<double, 2>(a, s);
  return launch_pc_nb<double, 4>(a, s);
}

}  // namespace

hipError_t launch_pc_forward(const PcArgs& a, hipStream_t s) {
  PcGemm g{};
  g.k = a.kernel;
  g.k_row = a.nm;
  g.k_step = (int64_t)a.L * a.nm;
  g.x = a.y;
  g.x_map = a.y_map_stride;
  g.x_step = a.nm;
  g.out = a.flm + (a.L - 1 + a.m_lo);
  g.o_map = a.flm_map_stride;
  g.o_row = 2 * a.L - 1;
  g.rows = a.L;
  g.steps = a.T;
  g.nm = a.nm;
  g.batch = a.batch;
  g.mirror = a.m_lo == 0;
  g.scale = a.scale;
  return launch_pc(g, a.kernel_complex, s);
}

hipError_t launch_pc_inverse(const PcArgs& a, hipStream_t s) {
  PcGemm g{};
  g.k = a.kernel;
  g.k_row = (int64_t)a.L * a.nm;
  g.k_step = a.nm;
  g.x = a.flm + (a.L - 1 + a.m_lo);
  g.x_map = a.flm_map_stride;
  g.x_step = 2 * a.L - 1;
  g.out = a.y;
  g.o_map = a.y_map_stride;
  g.o_row = a.nm;
  g.rows = a.T;
  g.steps = a.L;
  g.nm = a.nm;
  g.batch = a.batch;
  g.scale = a.scale;
  return launch_pc(g, a.kernel_complex, s);
}

}  // namespace s2h
