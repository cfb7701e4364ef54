// Latitudinal (Wigner-d) steps of small batches: the ell-recursion per (ring, m)
// in registers, fused with the synthesis (inverse) or the projection (forward).
//
// Replaces s2fft/transforms/otf_recursions.py, which recurses over m at fixed
// (theta, ell) with log-space renormalisation (price_mcewen.py:118-255).  Here
// each lane owns R rings (or ring pairs theta, pi-theta for spin 0) and walks
//   e^{l+1} = (a'_l x - b'_l) e^l - e^{l-1},   d^l = sigma_l e^l
// from l0 = max(|m|, |spin|): two FP64 operations per step (the plan's unit
// coefficients, which fold the normalisation sqrt((2l+1)/4pi) or the Wigner
// one).  Underflow of the boundary value sin^a cos^b at high m is handled with
// an integer scale index: true value = stored * 2^(512 * lscale), lscale <= 0; a
// ring only contributes once lscale reaches 0 (earlier terms are below 2^-256
// of the O(1) ones).
//
// What bounds them: one map needs 4 FP64 operations per ring, m and l (the
// recursion and a complex multiply-add), 16 cycles of a SIMD, but everything
// that is the same for all rings (coefficients, the inverse's flm, the
// forward's sums over rings) goes through LDS, one pipe for the four SIMDs.
// Several rings per lane share each of those accesses (rings_per_lane).  Paired
// rings (spin 0) have no b' and read 8 bytes of coefficients per step.
// Measured, one map: HEALPix nside 512, L = 1024, real: forward 229 -> 165 us,
// inverse 240 -> 112 us (55 us of FP64 operations each at the card's rate; the
// vector units are 62 % and 78 % busy); MW L = 128 forward 23 -> 12 us; GL L = 256
// 41 -> 22 us and 19 -> 13 us; GL L = 400, spin 1, 3 maps 182 -> 97 us and 114 ->
// 64 us (before: one ring per lane and three operations per step, the forward
// adding ring groups up with atomics onto a cleared flm).
#include <algorithm>

#include "s2h_fft_lds.h"
#include "s2h_kernels.h"
#include "s2h_lat_common.h"

namespace s2h {

namespace {

constexpr int kChunk = 128;  // l per staged chunk
constexpr int kLive = 32;    // l between two looks at the scale index
constexpr int kGroup = 8;    // steps unrolled together (inverse)
constexpr int kSum = 16;     // l whose sums over the rings are formed together
constexpr int kWaveLds = 512 + kChunk;  // complex values of LDS per wave of the forward
constexpr int kFwdWaves = 8;     // waves of a forward workgroup at most
constexpr int kFwdRingsMax = 8;  // rings per lane of the forward at most
// a grid has at most kMaxRingLen rings (DH: 2 L, HEALPix: 4 nside - 1)
static_assert(64 * kFwdRingsMax * kFwdWaves >= kMaxRingLen, "rings of one workgroup");

using lat::rescale;
using lat::start_value_fp64;

// by value: a conditional over array elements would keep the array in memory
__device__ __forceinline__ cplx sel(bool c, cplx a, cplx b) {
  return {c ? a.x : b.x, c ? a.y : b.y};
}

// One chunk of recursion coefficients (a', -b' bsign) in LDS: a' alone where b'
// vanishes.
template <bool PAIRED>
struct StepCoef;
template <>
struct StepCoef<true> {
  double a;
  __device__ __forceinline__ double factor(double x) const { return a * x; }
};
template <>
struct StepCoef<false> {
  double a, nb;
  __device__ __forceinline__ double factor(double x) const { return fma(a, x, nb); }
};
template <bool PAIRED>
__device__ __forceinline__ StepCoef<PAIRED> step_coef(const Coef& c, double bsign) {
  if constexpr (PAIRED)
    return {c.a};
  else
    return {c.a, -c.b * bsign};
}

// One step: (d, dm1) = (e^l, e^{l-1}) -> (e^{l+1}, e^l).
template <bool PAIRED>
__device__ __forceinline__ void step(const StepCoef<PAIRED>& c, double x, double& d, double& dm1) {
  const double dn = fma(c.factor(x), d, -dm1);
  dm1 = d;
  d = dn;
}

// Sum of the two halves of a's lanes in lanes 0 .. 31 and of b's in 32 .. 63.
__device__ __forceinline__ double half_sum(double a, double b) {
  const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
  return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}
// Rows of 16 lanes: (a0 + a1, b0 + b1, a2 + a3, b2 + b3).
__device__ __forceinline__ double row_sum(double a, double b) {
  const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
  return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}
__device__ __forceinline__ cplx half_sum(cplx a, cplx b) {
  return {half_sum(a.x, b.x), half_sum(a.y, b.y)};
}
__device__ __forceinline__ cplx row_sum(cplx a, cplx b) {
  return {row_sum(a.x, b.x), row_sum(a.y, b.y)};
}

// The tables of map b: the plan's, or its own in a multi-plane launch.
struct MapTables {
  const MStart* mstart;
  const Coef* ucoef;
  int lmin;
  __device__ MapTables(const LatArgs& a, int64_t b) {
    const LatPlane* pl = a.planes ? a.planes + b : nullptr;
    mstart = pl ? pl->mstart : a.mstart;
    ucoef = pl ? pl->ucoef : a.ucoef;
    lmin = pl ? pl->lmin_out : a.lmin_out;
  }
};

// The pole rows' spin and first l for map b.
__device__ __forceinline__ int pole_spin_of(const LatPole& p, int64_t b) {
  return p.spin + p.spin_step * (int)b;
}
__device__ __forceinline__ int pole_lmin_of(const LatPole& p, int64_t b) {
  const int s = pole_spin_of(p, b), as = s < 0 ? -s : s;
  return p.lmin_spin && as > p.lmin ? as : p.lmin;
}

}  // namespace

// ------------------------------------------------------------------ inverse
// NB maps per workgroup share each d-value.  The coefficients and the NB maps'
// flm (times sigma_l) of a chunk are loaded one chunk ahead and staged in a
// double-buffered LDS array, one barrier per chunk; every step reads them with
// broadcast loads.  The sums of a ring that starts to contribute are cleared
// (what came before is below 2^-256 of it).
template <int R, int NB, bool PAIRED>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2)))
lat_inverse_kernel(LatArgs a) {
  constexpr int P = PAIRED ? 2 : 1;  // sums per ring: both parities of l - l0, or one
  __shared__ StepCoef<PAIRED> cs[2][kChunk];
  __shared__ cplx fs[2][NB][kChunk];
  int g;
  const int m = lat::m_group_of_block(lat::balanced_block(blockIdx.x, gridDim.x), a.nm, a.groups,
                                      a.m_lo, g, 4);
  const int am = m < 0 ? -m : m;
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int b0 = blockIdx.z * NB;
  const MapTables tab(a, b0);  // multi-plane launches have NB = 1
  const MStart st = tab.mstart[m - a.m_lo];
  const double bsign = m < 0 ? -1.0 : 1.0;
  const Coef* __restrict__ cf = tab.ucoef + (int64_t)am * a.L;
  const int L = a.L, l0 = st.ell0;
  const int nb = min(NB, a.batch - b0);
  const int64_t frow = flm_row(a);
  const cplx* __restrict__ flm = a.flm + (int64_t)b0 * a.flm_map_stride + flm_col(a, m);

  // staging, one chunk ahead: kStage elements of (map, l) and kCoef
  // coefficients per thread of the smallest workgroup (64)
  constexpr int kStage = NB * kChunk / 64, kCoef = kChunk / 64;
  cplx fv[kStage];
  Coef cv[kCoef];
  const auto load = [&](int blk) {
#pragma unroll
    for (int k = 0; k < kStage; ++k) {
      const int e = tid + k * nthr, j = e / kChunk, l = blk + e % kChunk;
      const bool in = e < NB * kChunk && j < nb && l >= tab.lmin && l < L;
      fv[k] = {0.0, 0.0};
      if (in) {
        const cplx f = flm[(int64_t)j * a.flm_map_stride + (int64_t)l * frow];
        const double sigma = cf[l].c;
        fv[k] = {f.x * sigma, f.y * sigma};
      }
    }
#pragma unroll
    for (int k = 0; k < kCoef; ++k) {
      const int i = tid + k * nthr;
      cv[k] = Coef{0.0, 0.0, 0.0, 0.0};
      if (i < kChunk && blk + i + 1 < L) cv[k] = cf[blk + i];
    }
  };
  const auto stage = [&](int buf) {
#pragma unroll
    for (int k = 0; k < kStage; ++k) {
      const int e = tid + k * nthr;
      if (e < NB * kChunk) fs[buf][e / kChunk][e % kChunk] = fv[k];
    }
#pragma unroll
    for (int k = 0; k < kCoef; ++k) {
      const int i = tid + k * nthr;
      if (i < kChunk) cs[buf][i] = step_coef<PAIRED>(cv[k], bsign);
    }
  };
  load(l0);

  double x[R], d[R], dm1[R];
  int ls[R];
  cplx acc[R][NB][P];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int p = (g * R + r) * nthr + tid;
    x[r] = d[r] = dm1[r] = 0.0;
    ls[r] = 0;
    if (p < a.nrings) {
      const LatRing rg = a.rings[p];
      x[r] = rg.x;
      start_value_fp64(st, rg, d[r], ls[r]);
    }
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int q = 0; q < P; ++q) acc[r][j][q] = {0.0, 0.0};
  }
  stage(0);
  __syncthreads();

  int buf = 0;
  for (int blk = l0; blk < L; blk += kChunk, buf ^= 1) {
    const bool more = blk + kChunk < L;
    if (more) load(blk + kChunk);
    const int nsub = min(kChunk, L - blk);
    for (int s0 = 0; s0 < nsub; s0 += kLive) {
      const StepCoef<PAIRED>* c = cs[buf] + s0;
#pragma unroll 1
      for (int i0 = 0; i0 < kLive; i0 += kGroup) {
#pragma unroll
        for (int i = 0; i < kGroup; ++i) {
          const StepCoef<PAIRED> ci = c[i0 + i];
          cplx f[NB];
#pragma unroll
          for (int j = 0; j < NB; ++j) f[j] = fs[buf][j][s0 + i0 + i];
#pragma unroll
          for (int r = 0; r < R; ++r) {
#pragma unroll
            for (int j = 0; j < NB; ++j) {
              cplx& s = acc[r][j][PAIRED ? (i & 1) : 0];
              s.x = fma(d[r], f[j].x, s.x);
              s.y = fma(d[r], f[j].y, s.y);
            }
            step(ci, x[r], d[r], dm1[r]);
          }
        }
      }
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const bool was = ls[r] == 0;
        rescale(d[r], dm1[r], ls[r]);
        if (!was && ls[r] == 0) {
#pragma unroll
          for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int q = 0; q < P; ++q) acc[r][j][q] = {0.0, 0.0};
        }
      }
    }
    if (more) stage(buf ^ 1);
    __syncthreads();
  }

  // paired rings: ring b takes (-1)^(l + m) d, i.e. the parity of l - ell0,
  // with the roles swapped when ell0 + m is odd
  const bool flip = ((l0 + m) & 1) != 0;
  cplx* out = a.ftm + (int64_t)b0 * a.ftm_map_stride +
              (int64_t)(m - a.ftm_m_first) * spec_cstride(a.ftm_tiled);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int p = (g * R + r) * nthr + tid;
    if (p >= a.nrings) continue;
    const int2 tt = *reinterpret_cast<const int2*>(&a.rings[p].ta);
    const bool live = ls[r] == 0;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      if (j >= nb) continue;
      cplx* o = out + (int64_t)j * a.ftm_map_stride;
      const cplx zero = {0.0, 0.0};
      if constexpr (PAIRED) {
        const cplx ae = sel(live, sel(flip, acc[r][j][1], acc[r][j][0]), zero);
        const cplx ao = sel(live, sel(flip, acc[r][j][0], acc[r][j][1]), zero);
        o[spec_row(tt.x, a.ftm_ncol, a.ftm_tiled)] = cadd(ae, ao);
        if (tt.y >= 0 && tt.y != tt.x) o[spec_row(tt.y, a.ftm_ncol, a.ftm_tiled)] = csub(ae, ao);
      } else {
        o[spec_row(tt.x, a.ftm_ncol, a.ftm_tiled)] = sel(live, acc[r][j][0], zero);
      }
    }
  }
  if (g != 0) return;
  for (int e = tid; e < a.pad_rows * nb; e += nthr)
    out[(int64_t)(e / a.pad_rows) * a.ftm_map_stride +
        spec_row(a.pad_row0 + e % a.pad_rows, a.ftm_ncol, a.ftm_tiled)] = {0.0, 0.0};
  if (a.pole.south < 0 && a.pole.north < 0) return;
  // the pole rows' column m (spherical.py:166-177): the south row holds only m =
  // spin, sum_l (-1)^|l-spin| flm[l, spin], the north row only m = -spin, sum_l
  // flm[l, -spin] (both with the normalisation); the first wave sums over l
  if (tid >= 64) return;
  for (int j = 0; j < nb; ++j) {
    const int spin = pole_spin_of(a.pole, b0 + j);
    const cplx* f = flm + (int64_t)j * a.flm_map_stride;
    cplx* o = out + (int64_t)j * a.ftm_map_stride;
#pragma unroll
    for (int side = 0; side < 2; ++side) {
      const int row = side == 0 ? a.pole.south : a.pole.north;
      if (row < 0) continue;
      cplx s = {0.0, 0.0};
      if (m == (side == 0 ? spin : -spin)) {
        for (int l = pole_lmin_of(a.pole, b0 + j) + tid; l < L; l += 64) {
          const double w = a.pole.norm[l], sw = side == 0 && ((l - spin) & 1) ? -w : w;
          const cplx v = f[(int64_t)l * frow];
          s = {fma(sw, v.x, s.x), fma(sw, v.y, s.y)};
        }
        for (int k = 32; k > 0; k >>= 1) {
          s.x += __shfl_xor(s.x, k);
          s.y += __shfl_xor(s.y, k);
        }
      }
      if (tid == 0) o[(int64_t)row * a.ftm_ncol] = s;
    }
  }
}

// ------------------------------------------------------------------ forward
// One workgroup covers every ring of its (m, map), R per lane.  A step's terms are
// added up over the lane's rings, then over the lanes four l together: a swap of
// lane halves turns two l of 64 partial sums into one register of 2 x 32, a swap
// of rows two of these into one of 4 x 16; 16 l of them go through the wave's LDS
// (places skewed by (row, l), so that neither direction has bank conflicts), lane 16
// q + i adds four of l = i, and the four quarters meet by lane swaps.  The waves'
// sums of a chunk of l stay in LDS until its end, where they meet and are stored:
// one owner per element, no atomics, no zeroing pass; one barrier pair per chunk.
// The owner also writes the zeros below the first l, the m < 0 half of real maps
// and the pole terms, and has loaded the values that it adds to a chunk ahead.
template <int R, bool PAIRED>
__global__ void __launch_bounds__(64 * kFwdWaves) __attribute__((amdgpu_waves_per_eu(2)))
lat_forward_kernel(LatArgs a) {
  // per wave: 4 x 64 partial sums (double-buffered), then the sums of the chunk's l
  extern __shared__ __attribute__((aligned(16))) unsigned char fwd_raw[];
  __shared__ StepCoef<PAIRED> cs[2][kChunk];
  __shared__ double sg[2][kChunk];
  const int m = lat::m_of_block(lat::balanced_block(blockIdx.x, gridDim.x), a.nm, a.m_lo, 4);
  const int am = m < 0 ? -m : m;
  const int64_t b = blockIdx.z;
  const int tid = threadIdx.x, nthr = blockDim.x, lane = tid & 63, wave = tid >> 6;
  const int nwave = nthr >> 6;
  cplx* red = reinterpret_cast<cplx*>(fwd_raw) + wave * kWaveLds;
  cplx* tot = red + 512;  // [l - blk]
  const MapTables tab(a, b);
  const MStart st = tab.mstart[m - a.m_lo];
  const double bsign = m < 0 ? -1.0 : 1.0;
  const Coef* __restrict__ cf = tab.ucoef + (int64_t)am * a.L;
  const int L = a.L, l0 = st.ell0;
  const cplx* ftm = a.ftm + b * a.ftm_map_stride +
                    (int64_t)(m - a.ftm_m_first) * spec_cstride(a.ftm_tiled);

  constexpr int kCoef = kChunk / 64;
  Coef cv[kCoef];
  const auto load = [&](int blk) {
#pragma unroll
    for (int k = 0; k < kCoef; ++k) {
      const int i = tid + k * nthr;
      cv[k] = Coef{0.0, 0.0, 0.0, 0.0};
      if (i < kChunk && blk + i < L) cv[k] = cf[blk + i];  // a', b' are zero at L - 1
    }
  };
  const auto stage = [&](int buf) {
#pragma unroll
    for (int k = 0; k < kCoef; ++k) {
      const int i = tid + k * nthr;
      if (i < kChunk) {
        cs[buf][i] = step_coef<PAIRED>(cv[k], bsign);
        sg[buf][i] = cv[k].c;
      }
    }
  };
  load(l0);

  // ring-side data of ring r by the parity of l - ell0: the pair's sum where l +
  // m is even, else its difference; zero until the ring contributes
  const bool flip = PAIRED && ((l0 + m) & 1) != 0;
  double x[R], d[R], dm1[R];
  int ls[R];
  cplx u[R][PAIRED ? 2 : 1];
  const auto load_u = [&](int r) {
    const int p = (wave * R + r) * 64 + lane;
    const int2 tt = *reinterpret_cast<const int2*>(&a.rings[p].ta);
    const cplx fa = ftm[spec_row(tt.x, a.ftm_ncol, a.ftm_tiled)];
    if constexpr (PAIRED) {
      cplx fb = {0.0, 0.0};
      if (tt.y >= 0 && tt.y != tt.x) fb = ftm[spec_row(tt.y, a.ftm_ncol, a.ftm_tiled)];
      u[r][0] = flip ? csub(fa, fb) : cadd(fa, fb);
      u[r][1] = flip ? cadd(fa, fb) : csub(fa, fb);
    } else {
      u[r][0] = fa;
    }
  };
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int p = (wave * R + r) * 64 + lane;
    x[r] = d[r] = dm1[r] = 0.0;
    ls[r] = 0;
#pragma unroll
    for (int q = 0; q < (PAIRED ? 2 : 1); ++q) u[r][q] = {0.0, 0.0};
    if (p < a.nrings) {
      const LatRing rg = a.rings[p];
      x[r] = rg.x;
      start_value_fp64(st, rg, d[r], ls[r]);
      if (ls[r] == 0) load_u(r);
    }
  }

  cplx* out = a.flm + b * a.flm_map_stride + flm_col(a, m);
  const int64_t frow = flm_row(a);
  const double msgn = (m & 1) ? -1.0 : 1.0;
  const int mirror = m > 0 ? a.mirror : 0;  // 1: conjugate half, 2: zeros there
  const double scale = m > 0 ? a.pos_scale : 1.0;
  // pole terms (spherical.py:562-571): flm[l, spin] takes (-1)^|l-spin| of the
  // south row, flm[l, -spin] the north row
  const int pspin = pole_spin_of(a.pole, b), plmin = pole_lmin_of(a.pole, b);
  const bool south = a.pole.south >= 0 && m == pspin, north = a.pole.north >= 0 && m == -pspin;
  cplx ps = {0.0, 0.0}, pn = {0.0, 0.0};
  if (south) ps = ftm[spec_row(a.pole.south, a.ftm_ncol, a.ftm_tiled)];
  if (north) pn = ftm[spec_row(a.pole.north, a.ftm_ncol, a.ftm_tiled)];
  // rows below the first l (the packed layout holds none)
  if (!a.flm_packed) {
    for (int l = tid; l < min(l0, L); l += nthr) {
      if ((south || north) && l >= plmin) continue;  // below
      cplx* o = out + (int64_t)l * frow;
      if (!a.accumulate) *o = {0.0, 0.0};
      if (mirror) {
        const cplx v = a.accumulate ? *o : cplx{0.0, 0.0};
        o[-2 * m] = mirror == 1 ? cplx{msgn * v.x, -msgn * v.y} : cplx{0.0, 0.0};
      }
    }
  }
  // one element, by its owner; old: what it adds to
  const auto finish = [&](int l, cplx v, cplx old) {
    if (l < tab.lmin) v = {0.0, 0.0};
    if ((south || north) && l >= plmin) {
      const double w = a.pole.norm[l];
      if (south) {
        const double s = ((l - pspin) & 1) ? -w : w;
        v = {fma(s, ps.x, v.x), fma(s, ps.y, v.y)};
      }
      if (north) v = {fma(w, pn.x, v.x), fma(w, pn.y, v.y)};
    }
    cplx* o = out + (int64_t)l * frow;
    v = {fma(scale, v.x, old.x), fma(scale, v.y, old.y)};
    *o = v;
    if (mirror) o[-2 * m] = mirror == 1 ? cplx{msgn * v.x, -msgn * v.y} : cplx{0.0, 0.0};
  };
  // pole rows below the first l of the projection (l < |spin|)
  if ((south || north) && tid == 0 && !a.flm_packed)
    for (int l = plmin; l < min(l0, L); ++l)
      finish(l, {0.0, 0.0}, a.accumulate ? out[(int64_t)l * frow] : cplx{0.0, 0.0});

  stage(0);
  __syncthreads();
  // place of (t, lane) in the wave's partial sums, and of l = i's four of quarter q
  const int li = lane & 15, q = lane >> 4;
  const int rt = li >> 2, rrow = ((li & 1) << 1) | ((li >> 1) & 1);
  const auto place = [&](int k) { return rt * 64 + 16 * rrow + ((4 * q + k + 4 * rt + rrow) & 15); };
  const auto quarters = [&](const cplx (&v)[4], int s0) {
    const cplx w = cadd(cadd(v[0], v[1]), cadd(v[2], v[3]));
    const cplx h = half_sum(w, w), z = row_sum(h, h);
    if (lane < kSum) tot[s0 + lane] = z;
  };
  int buf = 0;
  for (int blk = l0; blk < L; blk += kChunk, buf ^= 1) {
    const bool more = blk + kChunk < L;
    if (more) load(blk + kChunk);
    cplx old[kCoef];
#pragma unroll
    for (int k = 0; k < kCoef; ++k) {
      const int l = blk + tid + k * nthr;
      old[k] = {0.0, 0.0};
      if (a.accumulate && tid + k * nthr < kChunk && l < L) old[k] = out[(int64_t)l * frow];
    }
    const int nsub = min(kChunk, L - blk);
    for (int s0 = 0; s0 < nsub; s0 += kSum) {
      const StepCoef<PAIRED>* c = cs[buf] + s0;
      // the partial sums of the group before: loaded here, needed after the steps
      const cplx* rp = red + (s0 & kSum ? 0 : 256);
      cplx v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = rp[place(k)];
      cplx* rw = red + (s0 & kSum ? 256 : 0);
      cplx p[4];
#pragma unroll
      for (int i = 0; i < kSum; ++i) {
        const StepCoef<PAIRED> ci = c[i];
        double px = 0.0, py = 0.0;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const cplx ur = u[r][PAIRED ? (i & 1) : 0];
          px = fma(d[r], ur.x, px);
          py = fma(d[r], ur.y, py);
          step(ci, x[r], d[r], dm1[r]);
        }
        p[i & 3] = {px, py};
        if ((i & 3) == 3) {
          const cplx h0 = half_sum(p[0], p[1]), h1 = half_sum(p[2], p[3]);
          const int t = i >> 2;
          rw[t * 64 + (lane & 48) + ((lane + 4 * t + q) & 15)] = row_sum(h0, h1);
        }
      }
      if (s0 > 0) quarters(v, s0 - kSum);
      lat::wave_sync();
      if ((s0 & kSum) || s0 + kSum >= nsub) {  // every kLive = 2 kSum steps
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const bool was = ls[r] == 0;
          rescale(d[r], dm1[r], ls[r]);
          if (!was && ls[r] == 0) load_u(r);
        }
      }
    }
    {
      const int last = (nsub - 1) & ~(kSum - 1);
      const cplx* rp = red + (last & kSum ? 256 : 0);
      cplx v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) v[k] = rp[place(k)];
      quarters(v, last);
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kCoef; ++k) {
      const int e = tid + k * nthr, l = blk + e;
      if (e < kChunk && l < L) {
        cplx s = (reinterpret_cast<const cplx*>(fwd_raw) + 512)[e];
        for (int w = 1; w < nwave; ++w)
          s = cadd(s, (reinterpret_cast<const cplx*>(fwd_raw) + w * kWaveLds + 512)[e]);
        const double sigma = sg[buf][e];  // e_l -> d_l
        finish(l, {sigma * s.x, sigma * s.y}, old[k]);
      }
    }
    if (more) stage(buf ^ 1);
    __syncthreads();
  }
}

// ------------------------------------------------------------------ launchers
namespace {

// Rings per lane: the fewest (1, 2, 4, up to rmax) with which a launch of
// `columns` (m, map) pairs has at most 4096 waves, four per SIMD: few columns need
// the waves, many are better off with shared LDS reads and sums.  Measured: 1024
// columns of 1024 pairs, forward 2 / 4 / 8 rings per lane 184 / 172 / 204 us, inverse
// 1 / 4 122 / 111 us; 2397 columns of 400 rings, forward 1 / 4 / 8 151 / 101 / 97 us,
// inverse 1 / 4 82 / 67 us; 511 columns of 256 rings, forward 1 / 2 22 / 21.5 us,
// inverse 1 / 2 13 / 14 us.
int rings_per_lane(int nrings, int64_t columns, int rmax) {
  int R = 1;
  while (R < rmax && columns * ((nrings + 64 * R - 1) / (64 * R)) > 4096) R *= 2;
  return R;
}

template <int R, int NB, bool PAIRED>
hipError_t lat_inv_r(LatArgs a, hipStream_t s) {
  // as many waves per workgroup (up to 4) as the rings fill
  const int waves = std::min(4, (a.nrings + 64 * R - 1) / (64 * R));
  a.groups = (a.nrings + 64 * R * waves - 1) / (64 * R * waves);
  const dim3 grid(a.nm * a.groups, 1, (a.batch + NB - 1) / NB), block(64 * waves);
  hipLaunchKernelGGL((lat_inverse_kernel<R, NB, PAIRED>), grid, block, 0, s, a);
  return hipGetLastError();
}
// Sums of 4 rings of 3 or 4 maps in two parities would not fit the registers.
template <int NB>
hipError_t lat_inv_nb(const LatArgs& a, bool paired, hipStream_t s) {
  const int64_t columns = (int64_t)a.nm * ((a.batch + NB - 1) / NB);
  switch (rings_per_lane(a.nrings, columns, paired && NB > 2 ? 2 : 4)) {
    case 1: return paired ? lat_inv_r<1, NB, true>(a, s) : lat_inv_r<1, NB, false>(a, s);
    case 2: return paired ? lat_inv_r<2, NB, true>(a, s) : lat_inv_r<2, NB, false>(a, s);
    default: return paired ? lat_inv_r<(NB > 2 ? 2 : 4), NB, true>(a, s) : lat_inv_r<4, NB, false>(a, s);
  }
}

template <int R>
hipError_t lat_fwd_r(const LatArgs& a, bool paired, hipStream_t s) {
  const int waves = (a.nrings + 64 * R - 1) / (64 * R);
  const dim3 grid(a.nm, 1, a.batch), block(64 * waves);
  const size_t lds = sizeof(cplx) * kWaveLds * waves;
  if (paired)
    hipLaunchKernelGGL((lat_forward_kernel<R, true>), grid, block, lds, s, a);
  else
    hipLaunchKernelGGL((lat_forward_kernel<R, false>), grid, block, lds, s, a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_lat_inverse(const LatArgs& a, bool paired, hipStream_t s) {
  if (a.nm == 0 || a.nrings == 0 || a.batch == 0) return hipSuccess;
  // up to 4 maps per workgroup (a multi-plane launch: one), evenly
  const int chunks = a.planes ? a.batch : (a.batch + 3) / 4;
  switch ((a.batch + chunks - 1) / chunks) {
    case 1: return lat_inv_nb<1>(a, paired, s);
    case 2: return lat_inv_nb<2>(a, paired, s);
    case 3: return lat_inv_nb<3>(a, paired, s);
    default: return lat_inv_nb<4>(a, paired, s);
  }
}

hipError_t launch_lat_forward(const LatArgs& a, bool paired, hipStream_t s) {
  if (a.nm == 0 || a.nrings == 0 || a.batch == 0) return hipSuccess;
  int R = rings_per_lane(a.nrings, (int64_t)a.nm * a.batch, kFwdRingsMax);
  while (a.nrings > 64 * R * kFwdWaves) R *= 2;
  switch (R) {
    case 1: return lat_fwd_r<1>(a, paired, s);
    case 2: return lat_fwd_r<2>(a, paired, s);
    case 4: return lat_fwd_r<4>(a, paired, s);
    case 8: return lat_fwd_r<8>(a, paired, s);
    default: return hipErrorInvalidValue;  // more rings than a plan has
  }
}

hipError_t allow_large_lds_lat() {
  const int bytes = (int)(sizeof(cplx) * kWaveLds * kFwdWaves);
  const void* fns[] = {
      (const void*)lat_forward_kernel<1, true>,  (const void*)lat_forward_kernel<1, false>,
      (const void*)lat_forward_kernel<2, true>,  (const void*)lat_forward_kernel<2, false>,
      (const void*)lat_forward_kernel<4, true>,  (const void*)lat_forward_kernel<4, false>,
      (const void*)lat_forward_kernel<8, true>,  (const void*)lat_forward_kernel<8, false>};
  for (const void* f : fns) {
    const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace s2h
