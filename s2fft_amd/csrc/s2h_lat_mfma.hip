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
// workgroup are summed through LDS in FP64 in a fixed order.  The FP64 kernel
// has one workgroup per m and adds its passes up by itself; the FP32 one adds
// the workgroups of an m with FP64 global atomics (2 per element at nside
// 1024, so the sum is independent of their order).  Even and odd l (relative
// to m) form separate 16-column tiles so that each uses one S (sum or
// difference).
//
// The recursion runs in its unit-c form (the plan's unit coefficients):
// e_{l+1} = (a'_l x - b'_l) e_l - e_{l-1}, two FP64 operations per step,
// d_l = sigma_l e_l; sigma_l depends on l only and scales the FP64 sums.
//
// T = double: V_MFMA_F64_16X16X4F64, the plain FP64 transform.
// T = float:  V_MFMA_F32_16X16X4F32 on FP32-rounded S and d with FP32
//             accumulation over 64 of a wave's rings; the recursion and every
//             sum beyond stay FP64 (mixed precision).  This
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

constexpr int kTile = 8;       // maps per tile (16 MFMA rows)
constexpr int kPad = 17;       // LDS row stride (elements) of the d tile

using lat::Mma;
using lat::m_of_block;
using lat::start_value;
using lat::wave_sync;

}  // namespace

// FP64: one workgroup per (m, tile of 8 MT maps) covers every ring pair of its m.
// A wave takes SETS x 64 pairs per pass, one recursion per lane and set; a pass
// walks l from the m's first l to L, 32 at a time, and adds its sums into flm, so
// no two workgroups write one element and nothing needs atomics or a zeroing pass.
// The first pass stores (writing the zeros below the m's first l and, with
// `mirror`, the m < 0 half last pass), later passes add; one thread owns each
// output element in every pass, so each addition reads that thread's own store,
// loaded at the start of its chunk.
// Bound by the matrix cores (64 cycles per product, one per 4 rings, 16 l and 8
// maps), if the recursion, the sums over waves and the memory stay hidden behind
// them: a wave alternates between the phases, so two workgroups of 4 waves share a
// CU and fill each other's gaps.  The ring-side operands of a wave's rings sit in
// registers for the whole pass: 128 of them hold 2 sets of 16 maps or 4 of 8, of pairs
// (two parities) half that; past 256 pairs one workgroup of 8 waves saves the second
// pass and the second reading of the recursions instead.  Measured: MW L = 512, spin
// 2, 64 maps 1411 -> 1259 us, from spectra in blocks of 8 rows (a column in 128-byte
// runs) 1035 us (0.5 ms of products); GL L = 700, spin 1, 5 maps 575 -> 413 us (all
// 700 rings in one pass); MW L = 256, real, 32 maps 88 -> 64 us.  Pairs on 4 waves of
// 2 sets: HEALPix L = 449, 5 maps 97 us against 74 on 8 waves, L = 512, 16 maps 519
// against 494.
// TILED: the spectra layout (spec_row) as a compile-time choice, so that the
// ring-major gathers carry no layout select in their address arithmetic
template <int W, int MT, int SETS, bool PAIRED, bool TILED>
__global__ void __launch_bounds__(64 * W, 2) lat_forward_f64_kernel(LatArgs a) {
  typedef lat::v4d acc_t;
  constexpr int P = PAIRED ? 2 : 1;  // operands: sum and difference of a pair, or the ring
  static_assert(64 * kPad >= MT * 2 * 16 * 16, "result tile fits");
  __shared__ double dte[W][64 * kPad];
  __shared__ double dto[W][64 * kPad];
  __shared__ lat::ChunkCoef ccs[2][lat::kChunk];  // recursion coefficients, double-buffered
  const int m = m_of_block(lat::balanced_block(blockIdx.x, gridDim.x), a.nm, a.m_lo);
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
    for (int e = threadIdx.x; e < MT * kTile * nz; e += (64 * W)) {
      const int bi = e / nz, l = lzero + e - bi * nz;
      if (b0 + bi < a.batch) {
        cplx* o = out + (int64_t)bi * a.flm_map_stride + (int64_t)l * frow;
        *o = {0.0, 0.0};
        if (mirror) o[-2 * m] = {0.0, 0.0};  // flm[l, -m]: 2m columns to the left
      }
    }
  }
  const int npass = (a.nrings + SETS * W * 64 - 1) / (SETS * W * 64);
  for (int pass = 0; pass < npass; ++pass) {
    const bool first = pass == 0, last = pass + 1 == npass;
    // recursion state: lane owns pair base(s) + lane of each set
    const auto base = [&](int s) { return ((pass * SETS + s) * W + wave) * 64; };
    double x[SETS], d[SETS], dm1[SETS];
    int ls[SETS];
    // A operands: tile t, row i = lane % 16 -> (map 8t + i/2, re/im i%2), pair base + 4c + lane/16.
    // The wave's ring rows are staged in LDS (its d tile is free here), then
    // the lane's components of rings ta and tb are gathered 8 pairs at a time
    // with all 16 loads in flight: branch-free, from clamped in-bounds
    // addresses, invalid entries zeroed afterwards (a load per conditional
    // branch would wait out one memory latency each).
    double sv[SETS][MT][P][16];
#pragma unroll
    for (int s = 0; s < SETS; ++s) {
      x[s] = d[s] = dm1[s] = 0.0;
      ls[s] = 0;
      int2* rrows = reinterpret_cast<int2*>(de);  // (ta, tb), -1: absent
      int2 tt = {-1, -1};
      if (base(s) + lane < a.nrings) {
        const LatRing rg = a.rings[base(s) + lane];
        x[s] = rg.x;
        lat::start_value_fp64(st, rg, d[s], ls[s]);
        tt = *reinterpret_cast<const int2*>(&a.rings[base(s) + lane].ta);
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
            if (PAIRED) vb[c] = mcol[2 * spec_row(rq[c].y < 0 ? 0 : rq[c].y, a.ftm_ncol, TILED)];
          }
#pragma unroll
          for (int c = 0; c < 8; ++c) {
            const double ca = have_map && rq[c].x >= 0 ? va[c] : 0.0;
            if constexpr (PAIRED) {
              const double cb = have_map && rq[c].y >= 0 ? vb[c] : 0.0;
              sv[s][t][0][c0 + c] = ca + cb;
              sv[s][t][1][c0 + c] = ca - cb;
            } else {
              sv[s][t][0][c0 + c] = ca;
            }
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
      // this thread's elements: (tile, l = blk + 2 col + parity, map)
      const int col = threadIdx.x & 15, omap = (threadIdx.x >> 4) & 7, opar = (threadIdx.x >> 7) & 1;
      const int ot = threadIdx.x >> 8;  // first tile (eight waves: two at a time)
      const int ol = blk + 2 * col + opar;
      constexpr int TS = W / 4, NO = (MT + TS - 1) / TS;
      cplx old[NO];
#pragma unroll
      for (int t = 0; t < NO; ++t) {
        const int bi = (t * TS + ot) * kTile + omap;
        old[t] = {0.0, 0.0};
        if ((!first || a.accumulate) && ol < L && t * TS + ot < MT && b0 + bi < a.batch)
          old[t] = out[(int64_t)bi * a.flm_map_stride + (int64_t)ol * frow];
      }
      acc_t acc[2][MT];
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[0][t] = acc[1][t] = acc_t{0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s = 0; s < SETS; ++s) {
        if (base(s) >= a.nrings) break;  // the wave's remaining sets are empty
        const bool live = ls[s] == 0;
        // 32 steps: even offsets to one tile, odd to the other (zero past the
        // band-limit: zero coefficients from l = L - 1 on)
#pragma unroll
        for (int i = 0; i < 32; ++i) {
          const double v = live ? d[s] : 0.0;
          if (i & 1)
            dodd[lane * kPad + (i >> 1)] = v;
          else
            de[lane * kPad + (i >> 1)] = v;
          const double dn = fma(fma(cs[i].a, x[s], cs[i].nb), d[s], -dm1[s]);
          dm1[s] = d[s];
          d[s] = dn;
        }
        lat::rescale(d[s], dm1[s], ls[s]);
        wave_sync();
        // each d tile element (B operand) feeds the MT map tiles; even and odd
        // products alternate, 2 MT accumulation chains in flight
#pragma unroll
        for (int c = 0; c < 16; ++c) {
          const double be = de[(4 * c + kq) * kPad + row];
          const double bo = dodd[(4 * c + kq) * kPad + row];
#pragma unroll
          for (int t = 0; t < MT; ++t) {
            acc[0][t] = Mma<double>::run(sv[s][t][0][c], be, acc[0][t]);
            acc[1][t] = Mma<double>::run(sv[s][t][P - 1][c], bo, acc[1][t]);
          }
        }
        wave_sync();
      }
      // the wave's sums: [tile][parity][row][col] over the (now free) even tile
#pragma unroll
      for (int t = 0; t < MT; ++t) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = Mma<double>::row_of(r, kq);
          ctw[t * 512 + i * 16 + row] = acc[0][t][r];
          ctw[t * 512 + 256 + i * 16 + row] = acc[1][t][r];
        }
      }
      if (more && threadIdx.x < lat::kChunk) ccs[buf ^ 1][threadIdx.x] = lat::finish_coef(cn, bsign);
      __syncthreads();
      // sum the waves in a fixed order; thread e owns its element of each map
      // tile in every pass and chunk
#pragma unroll
      for (int t = 0; t < NO; ++t) {
        const int tile = t * TS + ot, bi = tile * kTile + omap;
        if (ol < L && tile < MT && b0 + bi < a.batch) {
          const int e = tile * 512 + opar * 256 + omap * 32 + col;
          cplx v = {dte[0][e], dte[0][e + 16]};
#pragma unroll
          for (int w = 1; w < W; ++w) v = {v.x + dte[w][e], v.y + dte[w][e + 16]};
          const double sigma = cs[2 * col + opar].c;  // e_l -> d_l
          v = ol < a.lmin_out ? cplx{0.0, 0.0} : cplx{sigma * v.x, sigma * v.y};
          v = cadd(v, old[t]);
          cplx* o = out + (int64_t)bi * a.flm_map_stride + (int64_t)ol * frow;
          *o = v;
          // flm[l, -m] = (-1)^m conj(flm[l, m]), 2m columns to the left
          if (last && mirror) o[-2 * m] = {msgn * v.x, -msgn * v.y};
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
// FP32 sums per parity and element, met in FP64: a chain adds up 64 of the wave's 256
// rings.  With two (128 rings) the L + 1 rows of MW / MWSS left up to 1.86e-7 (L =
// 1024; the 2L + 1 rows of the column FFT chain 1.77e-7), with four 1.34e-7, HEALPix L
// = 2048 1.80e-7 -> 1.27e-7, at 1 % of the time (7.74 -> 7.81 ms for 16 maps).
constexpr int kFChains = 4;
}  // namespace

template <bool PAIRED, bool TILED>
__global__ void __launch_bounds__(kFT, 2) lat_forward_f32_kernel(LatArgs a) {
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

  // recursion state and A operands as in lat_forward_f64_kernel
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
    acc_t acc[2][kFChains];  // even and odd l
#pragma unroll
    for (int q = 0; q < kFChains; ++q) acc[0][q] = acc[1][q] = acc_t{0, 0, 0, 0};
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
        acc[0][c % kFChains] = Mma<float>::run(se[s][c], be, acc[0][c % kFChains]);
        acc[1][c % kFChains] = Mma<float>::run(so[s][c], bo, acc[1][c % kFChains]);
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
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        double v = 0.0;
#pragma unroll
        for (int k = 0; k < kFChains; ++k) v += (double)acc[q][k][r];
        ctw[256 * q + i * 16 + row] = v;
      }
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

template <int W, int MT, int SETS, bool PAIRED>
static hipError_t lat_fwd_f64(const LatArgs& a, hipStream_t s) {
  dim3 grid(a.nm, 1, (a.batch + MT * kTile - 1) / (MT * kTile));
  if (a.ftm_tiled)
    hipLaunchKernelGGL((lat_forward_f64_kernel<W, MT, SETS, PAIRED, true>), grid, dim3(64 * W), 0, s, a);
  else
    hipLaunchKernelGGL((lat_forward_f64_kernel<W, MT, SETS, PAIRED, false>), grid, dim3(64 * W), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_lat_forward_mfma(const LatArgs& a, bool paired, bool fp32, hipStream_t s) {
  if (a.nm == 0 || a.nrings == 0 || a.batch == 0) return hipSuccess;
  if (fp32) return lat_fwd_f32(a, paired, s);
  // FP64: 16-map tiles from 9 maps on
  const bool wide = a.batch > kTile;
  const int sets = (a.nrings + 255) / 256;  // of 64 rings per wave, four waves
  if (paired) {
    if (sets > 1) return wide ? lat_fwd_f64<8, 2, 1, true>(a, s) : lat_fwd_f64<8, 1, 1, true>(a, s);
    return wide ? lat_fwd_f64<4, 2, 1, true>(a, s) : lat_fwd_f64<4, 1, 1, true>(a, s);
  }
  if (wide) return sets > 1 ? lat_fwd_f64<4, 2, 2, false>(a, s) : lat_fwd_f64<4, 2, 1, false>(a, s);
  if (sets > 2) return lat_fwd_f64<4, 1, 4, false>(a, s);
  return sets > 1 ? lat_fwd_f64<4, 1, 2, false>(a, s) : lat_fwd_f64<4, 1, 1, false>(a, s);
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
