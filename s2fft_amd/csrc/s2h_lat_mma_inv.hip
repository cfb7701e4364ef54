// Batched inverse latitudinal step on the matrix cores.
//
// ftm[b, t, m] = sum_l d_l(t) flm[b, l, m]: for one m a (rings x l) . (l x maps)
// product whose left factor is generated by the ell-recursion.  Each wave owns
// 64 ring pairs (one recursion per lane); per 16-l chunk the d-values pass
// through a padded LDS tile into the A-operand layout (A[i][k]: lane i + 16k,
// i = pair within a 16-pair tile, k = l within a 4-l step), the flm values of
// the chunk are staged once per workgroup as B operands (B[k][j]: lane
// j + 16k, j = (map, re/im)), and each lane's accumulator owns whole outputs
// (C[i][j]: lane j + 16 (i%4), register i/4 for FP64; lane j + 16 (i/4),
// register i%4 for FP32), so no reduction is needed.  Even
// and odd l + m accumulate separately to serve the pair theta / pi - theta.
//
// Software pipeline: the d tile and the flm tile are double-buffered, and one
// loop body runs the 16 recursion steps of chunk k+1 between the 32 matrix
// products of chunk k (two products per step), so the vector ALUs and the
// matrix cores work at the same time within one wave; one barrier per chunk.
// T = double (plain FP64, V_MFMA_F64_16X16X4F64) or float (mixed precision,
// V_MFMA_F32_16X16X4F32, FP32 products accumulated in FP32 within a 16-l
// chunk and in FP64 across chunks).
#include "s2h_fft_lds.h"
#include "s2h_kernels.h"
#include "s2h_lat_common.h"

namespace s2h {

namespace {

constexpr int kIW = 4;       // waves per workgroup
constexpr int kIT = kIW * 64;
constexpr int kChunkL = 16;  // l per chunk
constexpr int kDPad = 17;    // LDS row stride (elements) of the d tile
constexpr int kMaps = 16;    // maps per workgroup (two 8-map column tiles)

using lat::Mma;
using lat::m_of_block;
using lat::start_value;
using lat::v4d;
using lat::v4f;

// unit-c coefficients of steps blk .. blk + 15 (lane i < 16), as stored
__device__ __forceinline__ Coef coef16(const Coef* cf, int blk, int i, int L) {
  return lat::load_ucoef_raw(cf, blk, i, L);
}

}  // namespace

// TILED: the spectra layout (spec_row) as a compile-time choice
template <typename T, bool PAIRED, bool TILED>
__global__ void __launch_bounds__(kIT, 2) lat_inverse_mma_kernel(LatArgs a) {
  typedef typename Mma<T>::acc acc_t;
  __shared__ __attribute__((aligned(16))) T dtile[kIW][2][64 * kDPad];  // [wave][buffer][pair][l_local]
  __shared__ T btile[2][kChunkL][2][16];          // [buffer][l_local][map tile][map*2 + comp]
  __shared__ lat::ChunkCoef ccs[2][kChunkL];      // recursion coefficients, double-buffered
  int grp;
  const int m = lat::m_group_of_block(blockIdx.x, a.nm, (a.nrings + kIT - 1) / kIT, a.m_lo, grp);
  const int am = m < 0 ? -m : m;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row = lane & 15, kq = lane >> 4;
  const int b0 = blockIdx.z * kMaps;
  const int L = a.L;
  const MStart st = a.mstart[m - a.m_lo];
  const double bsign = m < 0 ? -1.0 : 1.0;
  const Coef* __restrict__ cf = a.ucoef + (int64_t)am * L;  // unit-c: d_l = sigma_l e_l

  const int pbase = (grp * kIW + wave) * 64;
  const int p = pbase + lane;
  double x = 0.0, d = 0.0, dm1 = 0.0;
  int ls = 0;
  if (p < a.nrings) {
    const LatRing rg = a.rings[p];
    x = rg.x;
    if constexpr (sizeof(T) == 8)
      lat::start_value_fp64(st, rg, d, ls);
    else
      start_value(st, rg.c2, rg.s2, d, ls);
  }

  // accumulators: [map tile][16-pair tile q], even / odd l + m
  acc_t ae[2][4], ao[2][4];
  v4d se[2][4], so[2][4];  // FP64 accumulation across chunks (float path)
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      ae[t][q] = acc_t{0, 0, 0, 0};
      ao[t][q] = acc_t{0, 0, 0, 0};
      se[t][q] = v4d{0, 0, 0, 0};
      so[t][q] = v4d{0, 0, 0, 0};
    }

  const cplx* flm = a.flm + (int64_t)b0 * a.flm_map_stride + flm_col(a, m);
  // flm chunk staging: thread t holds elements e = t + kIT * j (j < 2) of
  // [l_local 16][column 32]
  constexpr int kStage = kChunkL * 32 / kIT;
  auto load_flm = [&](int blk, double* v) {
#pragma unroll
    for (int j = 0; j < kStage; ++j) {
      const int e = threadIdx.x + kIT * j;
      const int i = e >> 5, col = e & 31;
      const int l = blk + i, bm = col >> 1;
      double x0 = 0.0;
      if (l < L && l >= a.lmin_out && b0 + bm < a.batch) {
        const double* f = reinterpret_cast<const double*>(
            flm + (int64_t)bm * a.flm_map_stride + (int64_t)l * flm_row(a));
        x0 = f[col & 1];
      }
      v[j] = x0;
    }
  };
  // staged scaled by sigma_l (the chunk's coefficients in ccs[buf] hold it):
  // the d tile holds e_l = d_l / sigma_l
  auto store_flm = [&](int buf, const double* v) {
#pragma unroll
    for (int j = 0; j < kStage; ++j) {
      const int e = threadIdx.x + kIT * j;
      const int i = e >> 5, col = e & 31;
      btile[buf][i][col >> 4][col & 15] = T(v[j] * ccs[buf][i].c);
    }
  };
  // one unit-c recursion step of this lane's pair into d tile buffer `buf`;
  // steps past the band-limit produce zeros (zero coefficients from l = L - 1 on)
  auto step = [&](int buf, int i, bool live, const lat::ChunkCoef& c) {
    dtile[wave][buf][lane * kDPad + i] = live ? T(d) : T(0);
    const double dn = lat::rec_step_unit(c, x, d, dm1);
    dm1 = d;
    d = dn;
  };

  // ---- prologue: chunk 0 staged, its recursion done; chunk 1 prefetched
  double fv[kStage];
  Coef cn = {0.0, 0.0, 0.0, 0.0};
  load_flm(st.ell0, fv);
  if (threadIdx.x < kChunkL)
    ccs[0][threadIdx.x] = lat::finish_coef(lat::load_ucoef_raw(cf, st.ell0, threadIdx.x, L), bsign);
  __syncthreads();
  store_flm(0, fv);  // read by the products after the next barrier
  {
    const bool live = ls == 0;
#pragma unroll
    for (int i = 0; i < kChunkL; ++i) step(0, i, live, ccs[0][i]);
    lat::rescale(d, dm1, ls);
  }
  if (st.ell0 + kChunkL < L) {
    load_flm(st.ell0 + kChunkL, fv);
    if (threadIdx.x < kChunkL)
      ccs[1][threadIdx.x] =
          lat::finish_coef(lat::load_ucoef_raw(cf, st.ell0 + kChunkL, threadIdx.x, L), bsign);
  }
  __syncthreads();

  int cur = 0;
  for (int blk = st.ell0; blk < L; blk += kChunkL, cur ^= 1) {
    const int nxt = cur ^ 1;
    const bool has1 = blk + kChunkL < L;      // chunk k+1 exists
    const bool has2 = blk + 2 * kChunkL < L;  // chunk k+2 exists
    if (has1) store_flm(nxt, fv);             // chunk k+1's flm (loaded one chunk ago; its
                                              // coefficients are in ccs[nxt] since the last barrier)
    if (has2) {
      load_flm(blk + 2 * kChunkL, fv);
      if (threadIdx.x < kChunkL) cn = coef16(cf, blk + 2 * kChunkL, threadIdx.x, L);
    }
    const bool live = ls == 0;
    const T* dt = dtile[wave][cur];
    // product i -> (c = i / 8, q = (i / 2) % 4, parity = i % 2) for both map
    // tiles: A = d(pair 16 q + row, l_local le), B = flm(l_local le, column
    // row of map tile t), le = 2 (4 c + kq) + parity.  Each product's operands
    // are read from LDS one step ahead, so the read latency hides behind the
    // previous step instead of stalling the matrix cores.
    auto operands = [&](int i, T& av, T& b0v, T& b1v) {
      const int c = i >> 3, q = (i >> 1) & 3, par = i & 1;
      const int le = 2 * (4 * c + kq) + par;
      av = dt[(16 * q + row) * kDPad + le];
      b0v = btile[cur][le][0][row];
      b1v = btile[cur][le][1][row];
    };
    auto product = [&](int i, T av, T b0v, T b1v) {
      const int q = (i >> 1) & 3;
      if (i & 1) {
        ao[0][q] = Mma<T>::run(av, b0v, ao[0][q]);
        ao[1][q] = Mma<T>::run(av, b1v, ao[1][q]);
      } else {
        ae[0][q] = Mma<T>::run(av, b0v, ae[0][q]);
        ae[1][q] = Mma<T>::run(av, b1v, ae[1][q]);
      }
    };
    T an, b0n, b1n;
    operands(0, an, b0n, b1n);
    // 16 recursion steps of chunk k+1 between the 32 products of chunk k.  On
    // the last chunk the steps run on stale coefficients into the unused
    // buffer: no branch in the loop, and nothing reads their values.
#pragma unroll
    for (int i = 0; i < kChunkL; ++i) {
      const T ac = an, b0c = b0n, b1c = b1n;
      if (i + 1 < kChunkL) operands(i + 1, an, b0n, b1n);
      step(nxt, i, live, ccs[nxt][i]);
      product(i, ac, b0c, b1c);
    }
    lat::rescale(d, dm1, ls);
    if (sizeof(T) == 4) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            se[t][q][r] += (double)ae[t][q][r];
            so[t][q][r] += (double)ao[t][q][r];
          }
          ae[t][q] = acc_t{0, 0, 0, 0};
          ao[t][q] = acc_t{0, 0, 0, 0};
        }
    }
    if (has2 && threadIdx.x < kChunkL) ccs[cur][threadIdx.x] = lat::finish_coef(cn, bsign);  // chunk k+2's coefficients
    // orders: this chunk's reads of dtile[cur] / btile[cur] / ccs[nxt] before the
    // next body overwrites them, and this body's writes before their reads
    __syncthreads();
  }
  if (sizeof(T) == 8) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          se[t][q][r] = (double)ae[t][q][r];
          so[t][q][r] = (double)ao[t][q][r];
        }
  }
  // C[i][j]: pair 16q + row_of(r, kq), column j = row -> map t*8 + row/2, comp row%2.
  // The ring rows are loaded before any store (the stores could alias the
  // ring table, which would serialise the loads).
  int ta[16], tb[16];
#pragma unroll
  for (int q = 0; q < 4; ++q)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int pp = pbase + 16 * q + Mma<T>::row_of(r, kq);
      int ra = -1, rb = -1;
      if (pp < a.nrings) {
        const LatRing rg = a.rings[pp];
        ra = rg.ta;
        if (PAIRED && rg.tb >= 0 && rg.tb != rg.ta) rb = rg.tb;
      }
      ta[4 * q + r] = ra;
      tb[4 * q + r] = rb;
    }
  const bool dot = a.dot_part != nullptr;
  double dacc[2] = {0.0, 0.0};
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int bm = b0 + t * 8 + (row >> 1);
    if (bm >= a.batch) continue;
    double* out = reinterpret_cast<double*>(a.ftm + (int64_t)bm * a.ftm_map_stride +
                                            (int64_t)(m - a.ftm_m_first) * spec_cstride(TILED)) + (row & 1);
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int ra = ta[4 * q + r], rb = tb[4 * q + r];
        const double e = se[t][q][r], o = so[t][q][r];
        if (ra >= 0) {
          out[2 * spec_row(ra, a.ftm_ncol, TILED)] = e + o;
          if (dot && ra >= a.dot_row_lo && ra < a.dot_row_hi) dacc[t] = fma(e + o, e + o, dacc[t]);
        }
        if (rb >= 0) {
          out[2 * spec_row(rb, a.ftm_ncol, TILED)] = e - o;
          if (dot && rb >= a.dot_row_lo && rb < a.dot_row_hi) dacc[t] = fma(e - o, e - o, dacc[t]);
        }
      }
  }
  // the d tiles are no longer read (the loop ended on a barrier)
  if (dot) lat::synth_dot_partials<kIW>(a, m, b0, dacc, reinterpret_cast<double*>(&dtile[0][0][0]));
}

template <typename T>
static hipError_t lat_inv_mma(const LatArgs& a, bool paired, hipStream_t s) {
  dim3 grid(a.nm * ((a.nrings + kIT - 1) / kIT), 1, (a.batch + kMaps - 1) / kMaps);
  if (paired && a.ftm_tiled)
    hipLaunchKernelGGL((lat_inverse_mma_kernel<T, true, true>), grid, dim3(kIT), 0, s, a);
  else if (paired)
    hipLaunchKernelGGL((lat_inverse_mma_kernel<T, true, false>), grid, dim3(kIT), 0, s, a);
  else if (a.ftm_tiled)
    hipLaunchKernelGGL((lat_inverse_mma_kernel<T, false, true>), grid, dim3(kIT), 0, s, a);
  else
    hipLaunchKernelGGL((lat_inverse_mma_kernel<T, false, false>), grid, dim3(kIT), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_lat_inverse_mma(const LatArgs& a, bool paired, bool fp32, hipStream_t s) {
  if (a.nm == 0 || a.nrings == 0 || a.batch == 0) return hipSuccess;
  return fp32 ? lat_inv_mma<float>(a, paired, s) : lat_inv_mma<double>(a, paired, s);
}

// One V_MFMA_F32_16X16X4F32, for checking its lane layouts (as the f64 probe).
__global__ void mfma_f32_probe_kernel(const float* a, const float* b, float* out) {
  const int lane = threadIdx.x;
  v4f acc = {0.f, 0.f, 0.f, 0.f};
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[lane], b[lane], acc, 0, 0, 0);
  for (int r = 0; r < 4; ++r) out[lane * 4 + r] = acc[r];
}

hipError_t launch_mfma_f32_probe(const float* a, const float* b, float* out, hipStream_t s) {
  hipLaunchKernelGGL(mfma_f32_probe_kernel, dim3(1), dim3(64), 0, s, a, b, out);
  return hipGetLastError();
}

}  // namespace s2h
