// Batched forward latitudinal step on the matrix cores.
//
// flm[b, l, m] = sum_p S_par(l)[b, p] d_l(p): for one m this is a
// (maps x rings) . (rings x l) product whose right factor is generated by the
// ell-recursion.  Each wave owns 64 ring pairs per pass (one per lane) and
// walks 32 consecutive l in registers; the d-values go through a padded LDS
// tile into the B-operand layout (B[k][j]: lane j + 16k), and the ring-side
// data S (pair sum / difference of the ring Fourier coefficients, 8 maps x
// re/im = 16 rows) sit in registers as A operands (A[i][k]: lane i + 16k).
// The contraction over rings happens inside the MFMA; the waves of a
// workgroup are summed through LDS in FP64 in a fixed order, workgroups of
// one m with FP64 global atomics (2 per element at nside 1024, so the sum is
// independent of their order).  Even and odd l (relative to m) form separate
// 16-column tiles so that each uses one S (sum or difference).
//
// The recursion runs in its unit-c form (the plan's unit coefficients):
// e_{l+1} = (a'_l x - b'_l) e_l - e_{l-1}, two FP64 operations per step,
// d_l = sigma_l e_l; sigma_l depends on l only and scales the FP64 sums.
//
// T = double: V_MFMA_F64_16X16X4F64, the plain FP64 transform.
// T = float:  V_MFMA_F32_16X16X4F32 on FP32-rounded S and d with FP32
//             accumulation over the ring pairs of a wave; the recursion and
//             every sum beyond one wave stay FP64 (mixed precision).  This
//             arithmetic has its own kernel, lat_forward_f32_kernel: 4 waves
//             of 256 pairs, the d tiles double-buffered so that the recursion
//             of one 64-pair set runs between the products of the previous
//             set (5.8 instead of 6.3 ms at L 2048, 16 maps).  The same form
//             for FP64 fits only one wave per SIMD (LDS and registers) and
//             measured 11.3 instead of 8.7 ms.
#include "s2h_fft_lds.h"
#include "s2h_kernels.h"
#include "s2h_lat_common.h"

namespace s2h {

namespace {

constexpr int kMW = 8;         // waves per workgroup
constexpr int kMT = kMW * 64;  // threads
constexpr int kSets = 2;       // 64-pair sets per wave
constexpr int kTile = 8;       // maps per tile (16 MFMA rows)
constexpr int kPad = 17;       // LDS row stride (elements) of the d tile

using lat::Mma;
using lat::m_of_block;
using lat::start_value;
using lat::wave_sync;

}  // namespace

// FP64: one workgroup per (m, 16-map tile) covers every ring pair of its m.
// Its 8 waves take 512 pairs per pass (64 per wave); a pass walks l from the
// m's first l to L and adds its sums into flm, so no two workgroups write one
// element and nothing needs atomics or a zeroing pass.  The 16 maps form two
// 8-map row tiles of the matrix-core product that share each d-value (B
// operand), so each recursion step feeds 4 products instead of 2.  The first
// pass stores (writing the zeros below the m's first l and, with `mirror`,
// the m < 0 half last pass), later passes add; one thread owns each output
// element in every pass, so each addition reads that thread's own store.
// TILED: the spectra layout (spec_row) as a compile-time choice, so that the
// ring-major gathers carry no layout select in their address arithmetic
template <int MT, bool PAIRED, bool TILED>
__global__ void __launch_bounds__(kMT) lat_forward_f64_kernel(LatArgs a) {
  typedef lat::v4d acc_t;
  static_assert(64 * kPad * sizeof(double) >= MT * 2 * 16 * 16 * sizeof(double), "result tile fits");
  __shared__ double dte[kMW][64 * kPad];
  __shared__ double dto[kMW][64 * kPad];
  __shared__ lat::ChunkCoef ccs[2][lat::kChunk];  // recursion coefficients, double-buffered
  const int m = m_of_block(blockIdx.x, a.nm, a.m_lo);
  const int am = m < 0 ? -m : m;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int b0 = blockIdx.z * (MT * kTile);  // first map of the tile
  const int L = a.L;
  const MStart st = a.mstart[m - a.m_lo];
  const double bsign = m < 0 ? -1.0 : 1.0;
  const Coef* __restrict__ cf = a.ucoef + (int64_t)am * L;  // unit-c: d_l = sigma_l e_l
  double* de = dte[wave];
  double* dodd = dto[wave];
  double* ctw = dte[wave];
  const int row = lane & 15, kq = lane >> 4;
  const int lfirst = st.ell0 < L ? st.ell0 : L;
  cplx* out = a.flm + (int64_t)b0 * a.flm_map_stride + flm_col(a, m);
  const int64_t frow = flm_row(a);
  const bool mirror = a.mirror && m > 0;
  const double msgn = (m & 1) ? -1.0 : 1.0;

  // rows below the first l: zero (or unchanged when accumulating); the packed
  // layout holds no rows l < m
  const int lzero = a.flm_packed ? am : 0;
  const int nz = lfirst - lzero;
  if (!a.accumulate && nz > 0) {
    for (int e = threadIdx.x; e < MT * kTile * 2 * nz; e += kMT) {
      const int bi = e / (2 * nz), r = e - bi * 2 * nz;
      const int l = lzero + (r >> 1), comp = r & 1;
      if (b0 + bi < a.batch) {
        double* o = reinterpret_cast<double*>(out + (int64_t)bi * a.flm_map_stride + (int64_t)l * frow);
        o[comp] = 0.0;
        if (mirror) o[comp - 4 * m] = 0.0;  // flm[l, -m]: 2m complex columns to the left
      }
    }
  }
  const int npass = (a.nrings + kMW * 64 - 1) / (kMW * 64);
  for (int pass = 0; pass < npass; ++pass) {
    const bool first = pass == 0, last = pass + 1 == npass;
    // recursion state: lane owns pair p = (pass * kMW + wave) * 64 + lane
    const int base = (pass * kMW + wave) * 64;
    double x = 0.0, d = 0.0, dm1 = 0.0;
    int ls = 0;
    if (base + lane < a.nrings) {
      const LatRing rg = a.rings[base + lane];
      x = rg.x;
      lat::start_value_fp64(st, rg, d, ls);
    }
    // A operands: tile t, row i = lane % 16 -> (map 8t + i/2, re/im i%2), pair base + 4c + lane/16.
    // The wave's ring rows are staged in LDS (its d tile is free here), then
    // the lane's components of rings ta and tb are gathered 8 pairs at a time
    // with all 16 loads in flight: branch-free, from clamped in-bounds
    // addresses, invalid entries zeroed afterwards (a load per conditional
    // branch would wait out one memory latency each).
    double se[MT][16], so[MT][16];
    {
      int2* rrows = reinterpret_cast<int2*>(de);  // (ta, tb), -1: absent
      int2 tt = {-1, -1};
      if (base + lane < a.nrings) {
        tt = *reinterpret_cast<const int2*>(&a.rings[base + lane].ta);
        if (!PAIRED || tt.y < 0 || tt.y == tt.x) tt.y = -1;
      }
      rrows[lane] = tt;
      wave_sync();
      const int comp = row & 1;
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const int amap = b0 + t * kTile + (row >> 1);
        const bool have_map = amap < a.batch;
        const double* mcol = reinterpret_cast<const double*>(
            a.ftm + (int64_t)(have_map ? amap : 0) * a.ftm_map_stride + (int64_t)(m - a.ftm_m_first) * spec_cstride(TILED)) + comp;
#pragma unroll
        for (int c0 = 0; c0 < 16; c0 += 8) {
          int2 rq[8];
          double va[8], vb[8];
#pragma unroll
          for (int c = 0; c < 8; ++c) rq[c] = rrows[4 * (c0 + c) + kq];
#pragma unroll
          for (int c = 0; c < 8; ++c) {
            va[c] = mcol[2 * spec_row(rq[c].x < 0 ? 0 : rq[c].x, a.ftm_ncol, TILED)];
            vb[c] = mcol[2 * spec_row(rq[c].y < 0 ? 0 : rq[c].y, a.ftm_ncol, TILED)];
          }
#pragma unroll
          for (int c = 0; c < 8; ++c) {
            const double ca = have_map && rq[c].x >= 0 ? va[c] : 0.0;
            const double cb = have_map && rq[c].y >= 0 ? vb[c] : 0.0;
            se[t][c0 + c] = ca + cb;
            so[t][c0 + c] = PAIRED ? ca - cb : ca;
          }
        }
      }
      wave_sync();
    }
    Coef cn = {0.0, 0.0, 0.0, 0.0};
    if (threadIdx.x < lat::kChunk)
      ccs[0][threadIdx.x] = lat::finish_coef(lat::load_ucoef_raw(cf, st.ell0, threadIdx.x, L), bsign);
    __syncthreads();
    int buf = 0;
    for (int blk = st.ell0; blk < L; blk += 32, buf ^= 1) {
      const bool more = blk + 32 < L;
      if (more && threadIdx.x < lat::kChunk) cn = lat::load_ucoef_raw(cf, blk + 32, threadIdx.x, L);
      const lat::ChunkCoef* cs = ccs[buf];
      acc_t acc_e[MT], acc_o[MT];
#pragma unroll
      for (int t = 0; t < MT; ++t) acc_e[t] = acc_o[t] = acc_t{0.0, 0.0, 0.0, 0.0};
      const bool live = ls == 0;
      // 32 steps: even offsets to one tile, odd to the other (zero past the
      // band-limit: zero coefficients from l = L - 1 on); each 4-step group's
      // coefficients are read from LDS while the previous group steps
      double ca[4], cb[4], na[4], nb[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        ca[e] = cs[e].a;
        cb[e] = cs[e].nb;
      }
#pragma unroll
      for (int g = 0; g < 8; ++g) {
        if (g < 7) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            na[e] = cs[4 * (g + 1) + e].a;
            nb[e] = cs[4 * (g + 1) + e].nb;
          }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int i = 4 * g + e;
          const double v = live ? d : 0.0;
          if (i & 1)
            dodd[lane * kPad + (i >> 1)] = v;
          else
            de[lane * kPad + (i >> 1)] = v;
          const double dn = fma(fma(ca[e], x, cb[e]), d, -dm1);
          dm1 = d;
          d = dn;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          ca[e] = na[e];
          cb[e] = nb[e];
        }
      }
      wave_sync();
      // each d tile element (B operand) feeds the MT map tiles; even and odd
      // products alternate, 2 MT accumulation chains in flight
#pragma unroll
      for (int c = 0; c < 16; ++c) {
        const double be = de[(4 * c + kq) * kPad + row];
        const double bo = dodd[(4 * c + kq) * kPad + row];
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          acc_e[t] = Mma<double>::run(se[t][c], be, acc_e[t]);
          acc_o[t] = Mma<double>::run(so[t][c], bo, acc_o[t]);
        }
      }
      wave_sync();
      lat::rescale(d, dm1, ls);
      // the wave's sums: [tile][parity][row][col] over the (now free) even tile
#pragma unroll
      for (int t = 0; t < MT; ++t) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = Mma<double>::row_of(r, kq);
          ctw[t * 512 + i * 16 + row] = acc_e[t][r];
          ctw[t * 512 + 256 + i * 16 + row] = acc_o[t][r];
        }
      }
      if (more && threadIdx.x < lat::kChunk) ccs[buf ^ 1][threadIdx.x] = lat::finish_coef(cn, bsign);
      __syncthreads();
      // sum the waves in a fixed order; element (tile, parity, row, col) ->
      // l = blk + 2 col + parity, map b0 + 8 tile + row/2, component row%2.
      // Thread e owns element e in every pass and chunk.
      for (int e = threadIdx.x; e < MT * 512; e += kMT) {
        const int t = e >> 9, par = (e >> 8) & 1, rr = (e >> 4) & 15, col = e & 15;
        const int l = blk + 2 * col + par;
        const int bi = t * kTile + (rr >> 1);
        if (l < L && b0 + bi < a.batch) {
          double v = dte[0][e];
#pragma unroll
          for (int w = 1; w < kMW; ++w) v += dte[w][e];
          v *= cs[2 * col + par].c;  // sigma_l: e_l -> d_l
          double* o = reinterpret_cast<double*>(out + (int64_t)bi * a.flm_map_stride +
                                                (int64_t)l * frow) + (rr & 1);
          if (l < a.lmin_out) v = 0.0;
          if (!first || a.accumulate) v += *o;
          *o = v;
          // flm[l, -m] = (-1)^m conj(flm[l, m]), 2m complex columns to the left
          if (last && mirror) o[-4 * m] = (rr & 1) ? -msgn * v : msgn * v;
        }
      }
      __syncthreads();
    }
  }
}

namespace {
constexpr int kFW = 4;              // waves per workgroup, FP32 kernel
constexpr int kFT = kFW * 64;       // threads
constexpr int kFSets = 4;           // 64-pair sets per wave
}  // namespace

template <bool PAIRED, bool TILED>
__global__ void __launch_bounds__(kFT) lat_forward_f32_kernel(LatArgs a) {
  typedef typename Mma<float>::acc acc_t;
  // per wave, two buffers of the d tiles [parity][pair][l_local]: set s goes
  // to buffer s % 2.  After the chunk's products buffer 0 holds the wave's
  // results [parity][row][col] (FP64).
  static_assert(2 * 64 * kPad * sizeof(float) >= 2 * 16 * 16 * sizeof(double), "result tile fits");
  __shared__ float dt[2][kFW][2][64 * kPad];
  __shared__ lat::ChunkCoef ccs[2][lat::kChunk];  // recursion coefficients, double-buffered
  const int m = m_of_block(blockIdx.x, a.nm, a.m_lo);
  const int am = m < 0 ? -m : m;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int g = blockIdx.y;
  const int b0 = blockIdx.z * kTile;
  const int L = a.L;
  const MStart st = a.mstart[m - a.m_lo];
  const double bsign = m < 0 ? -1.0 : 1.0;
  const Coef* __restrict__ cf = a.ucoef + (int64_t)am * L;  // unit-c: d_l = sigma_l e_l
  double* ctw = reinterpret_cast<double*>(&dt[0][wave][0][0]);

  // recursion state and A operands as in lat_forward_mfma_kernel
  double x[kFSets], d[kFSets], dm1[kFSets];
  int ls[kFSets];
  float se[kFSets][16], so[kFSets][16];
  const int row = lane & 15, kq = lane >> 4;
  const int amap = b0 + (row >> 1);
  const bool have_map = amap < a.batch;
#pragma unroll
  for (int s = 0; s < kFSets; ++s) {
    const int base = ((g * kFW + wave) * kFSets + s) * 64;
    const int p = base + lane;
    dm1[s] = 0.0;
    if (p < a.nrings) {
      const LatRing rg = a.rings[p];
      x[s] = rg.x;
      start_value(st, rg.c2, rg.s2, d[s], ls[s]);
    } else {
      x[s] = 0.0;
      d[s] = 0.0;
      ls[s] = 0;
    }
    const cplx* ftm = a.ftm + (int64_t)amap * a.ftm_map_stride + (int64_t)(m - a.ftm_m_first) * spec_cstride(TILED);
#pragma unroll
    for (int c = 0; c < 16; ++c) {
      const int q = base + 4 * c + kq;
      double ve = 0.0, vo = 0.0;
      if (have_map && q < a.nrings) {
        const LatRing rq = a.rings[q];
        const cplx fa = ftm[spec_row(rq.ta, a.ftm_ncol, TILED)];
        cplx fb = {0.0, 0.0};
        if (PAIRED && rq.tb >= 0 && rq.tb != rq.ta) fb = ftm[spec_row(rq.tb, a.ftm_ncol, TILED)];
        const double ca = (row & 1) ? fa.y : fa.x;
        const double cb = (row & 1) ? fb.y : fb.x;
        ve = ca + cb;
        vo = PAIRED ? ca - cb : ca;
      }
      se[s][c] = (float)ve;
      so[s][c] = (float)vo;
    }
  }

  cplx* out = a.flm + (int64_t)b0 * a.flm_map_stride + flm_col(a, m);
  Coef cn = {0.0, 0.0, 0.0, 0.0};
  if (threadIdx.x < lat::kChunk)
    ccs[0][threadIdx.x] = lat::finish_coef(lat::load_ucoef_raw(cf, st.ell0, threadIdx.x, L), bsign);
  __syncthreads();
  int buf = 0;
  for (int blk = st.ell0; blk < L; blk += 32, buf ^= 1) {
    const bool more = blk + 32 < L;
    if (more && threadIdx.x < lat::kChunk) cn = lat::load_ucoef_raw(cf, blk + 32, threadIdx.x, L);
    const lat::ChunkCoef* cs = ccs[buf];
    acc_t acc_e[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}}, acc_o[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
    // recursion step i (0..31) of set s into buffer s % 2 (even offsets to
    // one tile, odd to the other)
    auto step = [&](int s, int i) {
      const double ca = cs[i].a, cb = cs[i].nb;
      dt[s & 1][wave][i & 1][lane * kPad + (i >> 1)] = ls[s] == 0 ? (float)d[s] : 0.0f;
      const double dn = fma(fma(ca, x[s], cb), d[s], -dm1[s]);
      dm1[s] = d[s];
      d[s] = dn;
    };
#pragma unroll
    for (int i = 0; i < 32; ++i) step(0, i);
    wave_sync();
    // the products of set s (even and odd alternating over four accumulation
    // chains) with the 32 recursion steps of set s + 1 between them
#pragma unroll
    for (int s = 0; s < kFSets; ++s) {
      const float* te = dt[s & 1][wave][0];
      const float* to = dt[s & 1][wave][1];
#pragma unroll
      for (int c = 0; c < 16; ++c) {
        const float be = te[(4 * c + kq) * kPad + row];
        const float bo = to[(4 * c + kq) * kPad + row];
        acc_e[c & 1] = Mma<float>::run(se[s][c], be, acc_e[c & 1]);
        acc_o[c & 1] = Mma<float>::run(so[s][c], bo, acc_o[c & 1]);
        if (s + 1 < kFSets) {
          step(s + 1, 2 * c);
          step(s + 1, 2 * c + 1);
        }
      }
      wave_sync();
      lat::rescale(d[s], dm1[s], ls[s]);  // set s has made the chunk's 32 steps
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = Mma<float>::row_of(r, kq);
      ctw[i * 16 + row] = (double)acc_e[0][r] + (double)acc_e[1][r];
      ctw[256 + i * 16 + row] = (double)acc_o[0][r] + (double)acc_o[1][r];
    }
    if (more && threadIdx.x < lat::kChunk) ccs[buf ^ 1][threadIdx.x] = lat::finish_coef(cn, bsign);
    __syncthreads();
    // sum the waves in a fixed order (element layout as in the FP64 kernel)
    for (int e = threadIdx.x; e < 2 * 16 * 16; e += kFT) {
      const int par = e >> 8, rr = (e >> 4) & 15, col = e & 15;
      const int l = blk + 2 * col + par;
      const int bm = b0 + (rr >> 1);
      double v = reinterpret_cast<const double*>(&dt[0][0][0][0])[e];
#pragma unroll
      for (int w = 1; w < kFW; ++w) v += reinterpret_cast<const double*>(&dt[0][w][0][0])[e];
      v *= cs[2 * col + par].c;  // sigma_l: e_l -> d_l
      if (l < L && l >= a.lmin_out && bm < a.batch) {
        double* o = reinterpret_cast<double*>(out + (int64_t)(rr >> 1) * a.flm_map_stride +
                                              (int64_t)l * flm_row(a)) + (rr & 1);
        if (a.groups > 1 || a.accumulate)
          atomicAdd(o, v);
        else
          *o = v;
      }
    }
    __syncthreads();
  }
}

static hipError_t lat_fwd_f32(const LatArgs& a0, bool paired, hipStream_t s) {
  LatArgs a = a0;
  const int per_wg = kFW * kFSets * 64;
  a.groups = (a.nrings + per_wg - 1) / per_wg;
  dim3 grid(a.nm, a.groups, (a.batch + kTile - 1) / kTile);
  if (paired && a.ftm_tiled)
    hipLaunchKernelGGL((lat_forward_f32_kernel<true, true>), grid, dim3(kFT), 0, s, a);
  else if (paired)
    hipLaunchKernelGGL((lat_forward_f32_kernel<true, false>), grid, dim3(kFT), 0, s, a);
  else if (a.ftm_tiled)
    hipLaunchKernelGGL((lat_forward_f32_kernel<false, true>), grid, dim3(kFT), 0, s, a);
  else
    hipLaunchKernelGGL((lat_forward_f32_kernel<false, false>), grid, dim3(kFT), 0, s, a);
  return hipGetLastError();
}

template <int MT>
static hipError_t lat_fwd_f64(const LatArgs& a, bool paired, hipStream_t s) {
  dim3 grid(a.nm, 1, (a.batch + MT * kTile - 1) / (MT * kTile));
  if (paired && a.ftm_tiled)
    hipLaunchKernelGGL((lat_forward_f64_kernel<MT, true, true>), grid, dim3(kMT), 0, s, a);
  else if (paired)
    hipLaunchKernelGGL((lat_forward_f64_kernel<MT, true, false>), grid, dim3(kMT), 0, s, a);
  else if (a.ftm_tiled)
    hipLaunchKernelGGL((lat_forward_f64_kernel<MT, false, true>), grid, dim3(kMT), 0, s, a);
  else
    hipLaunchKernelGGL((lat_forward_f64_kernel<MT, false, false>), grid, dim3(kMT), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_lat_forward_mfma(const LatArgs& a, bool paired, bool fp32, hipStream_t s) {
  if (a.nm == 0 || a.nrings == 0 || a.batch == 0) return hipSuccess;
  if (fp32) return lat_fwd_f32(a, paired, s);
  // FP64: 16-map tiles from 9 maps on, 8-map tiles below
  return a.batch > kTile ? lat_fwd_f64<2>(a, paired, s) : lat_fwd_f64<1>(a, paired, s);
}

// One V_MFMA_F64_16X16X4F64 on caller-provided operands, for checking the
// operand and result layouts: out[lane*4 + r] = D register r of lane.
__global__ void mfma_f64_probe_kernel(const double* a, const double* b, double* out) {
  const int lane = threadIdx.x;
  lat::v4d acc = {0.0, 0.0, 0.0, 0.0};
  acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[lane], b[lane], acc, 0, 0, 0);
  for (int r = 0; r < 4; ++r) out[lane * 4 + r] = acc[r];
}

hipError_t launch_mfma_f64_probe(const double* a, const double* b, double* out, hipStream_t s) {
  hipLaunchKernelGGL(mfma_f64_probe_kernel, dim3(1), dim3(64), 0, s, a, b, out);
  return hipGetLastError();
}

// Sustained V_MFMA_F64_16X16X4F64 rate: 8 independent accumulators per wave,
// no memory traffic in the loop (2048 flops per instruction).  The
// latitudinal kernels' FP64 roofline is quoted against the published peak;
// this gives the rate the matrix cores reach on the device at hand.
__global__ void __launch_bounds__(256) mfma_f64_rate_kernel(double* out, int iters, double a0) {
  lat::v4d acc[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = lat::v4d{0.0, 0.0, 0.0, 0.0};
  const double a = a0 + threadIdx.x * 1e-9, b = 1.0;
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc[j], 0, 0, 0);
  }
  double t = 0.0;
#pragma unroll
  for (int j = 0; j < 8; ++j) t += acc[j][0] + acc[j][1] + acc[j][2] + acc[j][3];
  out[(int64_t)blockIdx.x * 256 + threadIdx.x] = t;
}

hipError_t launch_mfma_f64_rate(int blocks, int iters, double* out, hipStream_t s) {
  hipLaunchKernelGGL(mfma_f64_rate_kernel, dim3(blocks), dim3(256), 0, s, out, iters, 1.0);
  return hipGetLastError();
}

}  // namespace s2h
