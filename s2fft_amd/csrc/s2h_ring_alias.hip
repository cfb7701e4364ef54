// Ring spectra without their FFTs: R = G - alpha A(Y) and the conjugate-gradient
// dot, A = (ring FFT) . (ring iFFT), on ring-major and tiled spectra.
#include "s2h_fft_lds.h"
#include "s2h_kernels.h"

namespace s2h {

namespace {

// for (p = tid; p < n; p += TPB) use(p, load(p)), with the loads of U
// consecutive iterations issued before any of their uses.  Without this each
// iteration waits out one global-memory latency, and a ring workgroup has too
// few waves beside it to hide that.
template <int TPB, int U, typename T, typename Load, typename Use>
__device__ __forceinline__ void batched_for(int n, Load load, Use use) {
  for (int p0 = threadIdx.x; p0 < n; p0 += U * TPB) {
    T v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int p = p0 + u * TPB;
      v[u] = p < n ? load(p) : T{};
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int p = p0 + u * TPB;
      if (p < n) use(p, v[u]);
    }
  }
}

}  // namespace

// ------------------------------------------------------------------ aliasing
// R = G - A(Y) for one (ring, map), A = (ring FFT) . (ring iFFT) with the
// FFTs cancelled: with m = q + j_m n (q = m mod n) and w = e^{i n phi0},
//   A(Y)[m] = w_t n e^{-i m phi0} sum_{m' = q mod n} e^{i m' phi0} c(m')
//           = w_t n w^{-j_m} T[q],   T[q] = sum_j w^j c(q + j n),
// m' = q + j n over [-(L-1), L-1] (c(m') = conj c(-m') for Hermitian spectra).
// On the supported grids n phi0 / pi is an integer, so w = +-1 (sgn).
// Rings with n >= 2L - 1 have one m' per q: R = G - w_t n Y elementwise.
// Otherwise thread t owns the residue q = t (mod n): with n >= TPB it sums
// T[q] itself; with n < TPB the G = TPB / n threads of a residue split the j
// (j = g, g + G, ... from the first) and meet in LDS in order of g.  Each
// thread then writes the outputs of its residue (the same split over j).
__device__ __forceinline__ cplx alias_term(const cplx* y, int m, int m_first, bool herm) {
  if (herm && m < 0) {
    const cplx t = y[-m - m_first];
    return {t.x, -t.y};
  }
  return y[m - m_first];
}

// floor(a / n) by a multiply-high with mag = floor((2^32 - 1) / n) + 1: exact
// for 0 <= a < 2^16 and 0 < n < 2^16 (the error a (n mag - 2^32) / 2^32 n stays
// below 1/n), so one division per thread replaces one per residue
struct FastDiv {
  int n;
  unsigned mag;
  __device__ explicit FastDiv(int n_) : n(n_), mag(n_ > 1 ? 0xFFFFFFFFu / (unsigned)n_ + 1u : 0u) {}
  __device__ __forceinline__ int floor(int a) const {
    if (n == 1) return a;
    return a >= 0 ? (int)__umulhi((unsigned)a, mag) : -(int)__umulhi((unsigned)(n - 1 - a), mag);
  }
};

// DOT: instead of writing R, the workgroup adds up
//   sum_m c_m Re(conj(Y[m]) A(Y)[m]),   c_m = 2 for m > 0 of Hermitian spectra, else 1,
// and stores it in a.part[map * jobs + job]: summed over rings this is
// <p, Lat_fwd(A(Lat_inv p))> for Y = Lat_inv(p) (the latitudinal transforms
// are transposes of each other), the curvature a conjugate-gradient step needs
// without projecting A(Y).  With a.alpha the written residual is
// R = G - alpha[map] A(Y); with a.part in that mode the workgroup also stores
// the sum of squares of the R it wrote (re^2 + im^2 over its columns).
template <int TPB, bool DOT>
__global__ void __launch_bounds__(TPB) ring_alias_kernel(RingAliasArgs a) {
  __shared__ double part[2 * TPB];
  if (!DOT && (int)blockIdx.x == a.jobs_end) {  // the padding rows, one run
    cplx* pad = a.r + (int64_t)blockIdx.y * a.map_stride + (int64_t)a.pad_row0 * a.ncol;
    for (int i = threadIdx.x; i < a.pad_rows * a.ncol; i += TPB) pad[i] = {0.0, 0.0};
    return;
  }
  const RingJob job = a.jobs[blockIdx.x];
  const int n = job.nphi;
  const int64_t off = (int64_t)blockIdx.y * a.map_stride + (int64_t)job.row * a.ncol;
  const cplx* __restrict__ y = a.y + off;
  const cplx* g = a.g + off;
  cplx* r = a.r + off;
  const double wn = job.weight * n * (a.alpha && !DOT ? a.alpha[blockIdx.y] : 1.0);
  const int lo = -(a.L - 1), hi = a.L - 1;
  const bool herm = a.herm != 0;
  const int t = threadIdx.x;
  double dsum = 0.0;
  if (n > hi - lo) {
    // no aliasing: the column's own m is the only term
    if constexpr (DOT) {
      batched_for<TPB, 8, cplx>(
          a.ncol, [&](int col) { return y[col]; },
          [&](int col, cplx yv) {
            const int m = a.m_first + col;
            if (m >= lo && m <= hi)
              dsum += (herm && m > 0 ? 2.0 * wn : wn) * (yv.x * yv.x + yv.y * yv.y);
          });
    } else {
      batched_for<TPB, 8, cplx>(
          a.ncol, [&](int col) { return g[col]; },
          [&](int col, cplx gv) {
            const int m = a.m_first + col;
            cplx v = {0.0, 0.0};
            if (m >= lo && m <= hi) v = alias_term(y, m, a.m_first, herm);
            const cplx rv = {gv.x - wn * v.x, gv.y - wn * v.y};
            r[col] = rv;
            dsum = fma(rv.x, rv.x, fma(rv.y, rv.y, dsum));
          });
      if (!a.part) return;
    }
  } else if (herm && a.m_first == 0 && n >= a.L) {
    // Hermitian spectra stored for m in [0, L) on a ring with L <= n < 2L - 1:
    // the only alias of m is m - n, whose coefficient is conj Y[n - m], so
    // A(Y)[m] = w n (Y[m] + w^{-1} conj Y[n - m]) for m >= n - L + 1, else w n Y[m]
    const int e = (int)rint(n * job.phi0_over_pi);
    const double sgn = (a.apply_phase && (e & 1)) ? -1.0 : 1.0;
    const int m_pair = n - a.L + 1;
    for (int m = t; m < a.ncol; m += TPB) {
      const cplx yv = y[m];
      cplx av = yv;
      if (m >= m_pair) {
        const cplx yp = y[n - m];
        av = {fma(sgn, yp.x, av.x), fma(-sgn, yp.y, av.y)};
      }
      if constexpr (DOT) {
        dsum += (m > 0 ? 2.0 * wn : wn) * (yv.x * av.x + yv.y * av.y);
      } else {
        const cplx gv = g[m];
        const cplx rv = {gv.x - wn * av.x, gv.y - wn * av.y};
        r[m] = rv;
        dsum = fma(rv.x, rv.x, fma(rv.y, rv.y, dsum));
      }
    }
    if (!DOT && !a.part) return;
  } else {
    const int e = (int)rint(n * job.phi0_over_pi);
    const double sgn = (a.apply_phase && (e & 1)) ? -1.0 : 1.0;
    // the division's operands: |q - lo|, |hi - q|, |q - m_first| and
    // |m_last - q| are below n + 2L (the host keeps n + 2L < 2^16)
    const FastDiv dv(n);
    const int G = n >= TPB ? 1 : TPB / n;
    const int nq = n >= TPB ? (n + TPB - 1) / TPB : 1;  // residues per thread
    const int gi = n >= TPB ? 0 : t / n;
    const bool active = gi < G;
    const int m_last = a.m_first + a.ncol - 1;
    for (int qi = 0; qi < nq; ++qi) {
      const int q = n >= TPB ? t + qi * TPB : t % n;
      const bool own = active && q < n;
      // T[q]: j from j0 = ceil((lo - q) / n) to floor((hi - q) / n), this
      // thread's j = j0 + gi + k G
      cplx acc = {0.0, 0.0};
      int j0 = 0;
      if (own) {
        j0 = -dv.floor(q - lo);
        const int j1 = dv.floor(hi - q);
        const int cnt = j1 - j0 + 1;
        for (int k0 = gi; k0 < cnt; k0 += 4 * G) {
          cplx v[4];
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int k = k0 + u * G;
            v[u] = k < cnt ? alias_term(y, q + (j0 + k) * n, a.m_first, herm) : cplx{0.0, 0.0};
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int k = k0 + u * G;
            const double sj = ((j0 + k) & 1) && sgn < 0 ? -1.0 : 1.0;
            acc = {fma(sj, v[u].x, acc.x), fma(sj, v[u].y, acc.y)};
          }
        }
      }
      if (G > 1) {
        if (own) {
          part[2 * t] = acc.x;
          part[2 * t + 1] = acc.y;
        }
        __syncthreads();
        cplx tot = {0.0, 0.0};
        if (own)
          for (int gg = 0; gg < G; ++gg)
            tot = cadd(tot, cplx{part[2 * (gg * n + q)], part[2 * (gg * n + q) + 1]});
        __syncthreads();
        acc = tot;
      }
      if (!own) continue;
      // outputs m = q + j n in [m_first, m_last], this thread's j = jo + gi + k G
      const int jo = -dv.floor(q - a.m_first);
      const int cnt = dv.floor(m_last - q) - jo + 1;
      const cplx* src = DOT ? y : g;
      for (int k0 = gi; k0 < cnt; k0 += 4 * G) {
        cplx gv[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int k = k0 + u * G;
          gv[u] = k < cnt ? src[q + (jo + k) * n - a.m_first] : cplx{0.0, 0.0};
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int k = k0 + u * G;
          if (k < cnt) {
            const double c = (((jo + k) & 1) && sgn < 0 ? -wn : wn);
            if constexpr (DOT) {
              const int m = q + (jo + k) * n;
              dsum += (herm && m > 0 ? 2.0 * c : c) * (gv[u].x * acc.x + gv[u].y * acc.y);
            } else {
              const cplx rv = {gv[u].x - c * acc.x, gv[u].y - c * acc.y};
              r[q + (jo + k) * n - a.m_first] = rv;
              dsum = fma(rv.x, rv.x, fma(rv.y, rv.y, dsum));
            }
          }
        }
      }
    }
  }
  // residue-owned columns: the written values of R in the no-alias branch
  // when a.part is set (write mode) fall through to the same reduction
  if (DOT || a.part) {
    // fixed-order workgroup sum: waves by shuffles, then wave 0 over the waves
    for (int o = 32; o > 0; o >>= 1) dsum += __shfl_xor(dsum, o);
    __syncthreads();
    if ((t & 63) == 0) part[t >> 6] = dsum;
    __syncthreads();
    if (t == 0) {
      double tot = 0.0;
      for (int w = 0; w < TPB / 64; ++w) tot += part[w];
      a.part[(int64_t)blockIdx.y * a.jobs_end + blockIdx.x] = tot;
    }
  }
}

// pq[b] = sum over the rings' partial sums in ring order; alpha[b] = num[b] / pq[b]
__global__ void __launch_bounds__(256) ring_dot_final_kernel(const double* part, int njobs,
                                                             const double* num, double* pq,
                                                             double* alpha) {
  __shared__ double red[4];
  const int b = blockIdx.x;
  double acc = 0.0;
  for (int k = threadIdx.x; k < njobs; k += 256) acc += part[(int64_t)b * njobs + k];
  for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0) {
    const double tot = (red[0] + red[1]) + (red[2] + red[3]);
    if (pq) pq[b] = tot;
    if (alpha) alpha[b] = (num && tot != 0.0) ? num[b] / tot : 0.0;
  }
}

// ------------------------------------------------------------------ aliasing, tiled
// ring_alias_kernel's cases for real maps (Hermitian spectra stored for m in
// [0, L)) on the tiled spectra (spec_row), per row block of 8 rows:
//  * belt blocks (every row n >= 2L - 1, no alias: R = G - w n Y) by
//    ring_alias_belt_kernel: kAliasSplit workgroups per block, lane 8 cg + r
//    on row r and column group v = split NG + cg, so that a wave's access to
//    8 columns of the 8 rows is one contiguous kilobyte;
//  * the other blocks by ring_alias_polar_kernel: RW rows of the block per
//    workgroup, their spectra staged in LDS by whole columns (RW 16 coalesced
//    bytes each), then per row as in ring_alias_kernel:
//      L <= n < 2L - 1: the one alias m - n of m >= n - L + 1, whose
//        coefficient is conj Y[n - m]: A(Y)[m] = w n (Y[m] + sgn conj Y[n - m]);
//      n < L: residue sums T[q] = sum_j s_j c(q + j n) over m' in
//        [-(L-1), L-1] (c(m') = conj Y[-m'] for m' < 0, s_j = -1 for odd j
//        when sgn < 0), then A(Y)[q + j n] = s_j w n T[q];  residues of rows
//        with n below the lanes per row split their j over groups that meet
//        in LDS in group order,
//    A(Y) / (w n) written over the staged Y, and R = G - w n A written back
//    by whole columns.
// Every per-row sum runs in a fixed order, and each workgroup's partial sum
// (dot or |R|^2) is reduced in a fixed order into part[map][block][slot]
// (kAliasSlots slots per block; the unused ones are zeroed): deterministic.
constexpr int kAliasSplit = 4;
constexpr int kAliasSlots = 8;
// polar workgroups: TPB threads staging up to LDSB bytes of spectra (8
// columns per lane): 1024 threads and 128 KB (L <= 8192); the dot up to
// L = 4096 as two workgroups of 512 threads and 64 KB per CU, so that one
// stages while the other sums
constexpr int kAliasPolarTpb = 1024;
constexpr int kAliasPolarLds = 128 * 1024;
constexpr int kAliasDotTpb = 512;
constexpr int kAliasDotLds = 64 * 1024;

// rows of a block per polar workgroup: the largest power of two <= 8 with
// RW L 16 bytes within the LDS budget ldsb
__host__ __device__ inline int alias_polar_rows(int L, int ldsb) {
  int rw = kSpecBlock;
  while (rw > 1 && (int64_t)rw * L * 16 > ldsb) rw >>= 1;
  return rw;
}

// fixed-order workgroup sum of dsum into part[slot]; slot 0's workgroup
// also zeroes the slots >= nslots
template <int TPB>
__device__ __forceinline__ void alias_block_sum(double dsum, double* red, double* part, int slot,
                                                int nslots) {
  const int t = threadIdx.x;
  for (int o = 32; o > 0; o >>= 1) dsum += __shfl_xor(dsum, o);
  __syncthreads();
  if ((t & 63) == 0) red[t >> 6] = dsum;
  __syncthreads();
  if (t == 0) {
    double tot = 0.0;
    for (int w = 0; w < TPB / 64; ++w) tot += red[w];
    part[slot] = tot;
    if (slot == 0)
      for (int k = nslots; k < kAliasSlots; ++k) part[k] = 0.0;
  }
}

template <int TPB, bool DOT>
__global__ void __launch_bounds__(TPB) ring_alias_belt_kernel(RingAliasTiledArgs a) {
  constexpr int NG = TPB / kSpecBlock;  // column groups per workgroup
  constexpr int NV = kAliasSplit * NG;  // column groups per row block
  constexpr int U = 4;                  // loads in flight
  __shared__ double red[TPB / 64];
  const int t = threadIdx.x, r = t & 7, cg = t >> 3;
  const int blk = a.belt_blocks[blockIdx.x], b = blockIdx.y, sp = blockIdx.z;
  const int v = sp * NG + cg;
  const int row = kSpecBlock * blk + r;
  const RingJob job = a.rowjobs[row];
  const int n = job.nphi;
  const int L = a.L;
  const int64_t tile = (int64_t)b * a.map_stride + (int64_t)blk * kSpecBlock * a.ncol;
  const cplx* __restrict__ y = a.y + tile + r;  // column m at y[8 m]
  cplx* rr = a.r + tile + r;
  const cplx* g = a.g_tiled ? a.g + tile + r
                            : a.g + (int64_t)b * a.map_stride + (int64_t)row * a.ncol;
  const int gs = a.g_tiled ? kSpecBlock : 1;
  const double wn = job.weight * n * (a.alpha && !DOT ? a.alpha[b] : 1.0);
  double dsum = 0.0;
  if (n > 0) {
    for (int m0 = v; m0 < L; m0 += U * NV) {
      cplx yv[U], gv[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int m = m0 + u * NV;
        yv[u] = gv[u] = cplx{0.0, 0.0};
        if (m < L) {
          yv[u] = y[kSpecBlock * m];
          if (!DOT) gv[u] = g[gs * m];
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int m = m0 + u * NV;
        if (m >= L) continue;
        if constexpr (DOT) {
          dsum += (m > 0 ? 2.0 * wn : wn) * (yv[u].x * yv[u].x + yv[u].y * yv[u].y);
        } else {
          const cplx rv = {gv[u].x - wn * yv[u].x, gv[u].y - wn * yv[u].y};
          rr[kSpecBlock * m] = rv;
          dsum = fma(rv.x, rv.x, fma(rv.y, rv.y, dsum));
        }
      }
    }
  }
  if (DOT || a.part)
    alias_block_sum<TPB>(dsum, red,
                         a.part + (int64_t)b * a.part_map_stride + a.belt_part_off +
                             (int64_t)blockIdx.x * kAliasSlots,
                         sp, kAliasSplit);
}

template <bool DOT, int TPB, int LDSB>
__global__ void __launch_bounds__(TPB) ring_alias_polar_kernel(RingAliasTiledArgs a) {
  constexpr int kAliasMaxCols = LDSB / 16 / TPB;  // staged columns per lane
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  cplx* ys = reinterpret_cast<cplx*>(lds_raw);  // [column m][row of the workgroup]
  __shared__ double xch[2 * TPB];                // residue groups' partial sums
  __shared__ double red[TPB / 64];
  const int L = a.L;
  const int RW = alias_polar_rows(L, LDSB);
  const int H = kSpecBlock / RW;                 // workgroups per block
  // blockIdx.x -> (block, part z): the H parts of a block on one XCD
  // (workgroups are dealt to the 8 XCDs round-robin), so that they read each
  // 128-byte line of the block through that XCD's L2 at about the same time
  const int i = blockIdx.x;
  const int z = (i >> 3) % H;
  const int bi = ((i >> 3) / H) * 8 + (i & 7);
  if (bi >= a.n_polar) return;
  const int blk = a.polar_blocks[bi], b = blockIdx.y;
  const int t = threadIdx.x;
  const int r0 = z * RW;
  const int64_t tile = (int64_t)b * a.map_stride + (int64_t)blk * kSpecBlock * a.ncol;
  const int ntot = L * RW;  // <= kAliasMaxCols TPB
  // stage Y: element (m, q) of the workgroup's rows at ys[m RW + q]; every
  // load of the thread in flight before the first LDS store (q = t % RW is
  // the thread's own: TPB is a multiple of RW)
  const int qt = t % RW;
  {
    cplx v[kAliasMaxCols];
#pragma unroll
    for (int k = 0; k < kAliasMaxCols; ++k) {
      const int idx = t + k * TPB;
      v[k] = idx < ntot ? a.y[tile + (int64_t)(idx / RW) * kSpecBlock + r0 + qt]
                        : cplx{0.0, 0.0};
    }
#pragma unroll
    for (int k = 0; k < kAliasMaxCols; ++k) {
      const int idx = t + k * TPB;
      if (idx < ntot) ys[idx] = v[k];
    }
  }
  __syncthreads();

  const int LPR = TPB / RW;                      // lanes per row
  const int rq = t / LPR, li = t - rq * LPR;
  const int row = kSpecBlock * blk + r0 + rq;
  const RingJob job = a.rowjobs[row];
  const int n = job.nphi;
  const double wn = job.weight * n * (a.alpha && !DOT ? a.alpha[b] : 1.0);
  const int e = (int)rint(n * job.phi0_over_pi);
  const double sgn = (a.apply_phase && (e & 1)) ? -1.0 : 1.0;
  auto Y = [&](int m) { return ys[m * RW + rq]; };
  const int kind = n == 0 ? 0 : n > 2 * L - 2 ? 1 : n >= L ? 2 : 3;  // none, no alias, pair, fold
  double dsum = 0.0;

  // pair rows: A(Y) / (w n) of columns li + k LPR, fold rows: T of residues
  // q = li + k LPR (n >= LPR) or of the one residue of a split, in registers
  cplx av[kAliasMaxCols];
  cplx* tq = av;
  const bool splitf = kind == 3 && n < LPR;
  const int G = splitf ? LPR / n : 1;
  const int gi = splitf ? li / n : 0;
  const int qs = splitf ? li % n : li;
  const bool owns = kind == 3 && gi < G;
  FastDiv dv(kind == 3 ? n : 1);
#pragma unroll
  for (int k = 0; k < kAliasMaxCols; ++k) av[k] = cplx{0.0, 0.0};
  if (kind == 2) {
    const int m_pair = n - L + 1;
#pragma unroll
    for (int k = 0; k < kAliasMaxCols; ++k) {
      const int m = li + k * LPR;
      if (m < L) {
        const cplx y0 = Y(m);
        cplx v = y0;
        if (m >= m_pair) {
          const cplx yp = Y(n - m);
          v = {fma(sgn, yp.x, v.x), fma(-sgn, yp.y, v.y)};
        }
        av[k] = v;
        if constexpr (DOT) dsum += (m > 0 ? 2.0 * wn : wn) * (y0.x * v.x + y0.y * v.y);
      }
    }
  } else if (owns) {
#pragma unroll
    for (int k = 0; k < kAliasMaxCols; ++k) {
      const int q = qs + k * (splitf ? 0 : LPR);
      if ((splitf && k > 0) || q >= n) continue;
      const int j0 = -dv.floor(q + L - 1);
      const int cnt = dv.floor(L - 1 - q) - j0 + 1;
      cplx acc = {0.0, 0.0};
      for (int kk = gi; kk < cnt; kk += G) {
        const int mp = q + (j0 + kk) * n;
        cplx v = Y(mp < 0 ? -mp : mp);
        if (mp < 0) v.y = -v.y;
        const double sj = ((j0 + kk) & 1) && sgn < 0 ? -1.0 : 1.0;
        acc = {fma(sj, v.x, acc.x), fma(sj, v.y, acc.y)};
      }
      tq[k] = acc;
    }
  }
  // split residues: the groups' partial sums meet in LDS in group order
  xch[2 * t] = tq[0].x;
  xch[2 * t + 1] = tq[0].y;
  __syncthreads();
  if (splitf && owns) {
    cplx T = {0.0, 0.0};
    for (int gg = 0; gg < G; ++gg) {
      const int src = rq * LPR + gg * n + qs;
      T = {T.x + xch[2 * src], T.y + xch[2 * src + 1]};
    }
    tq[0] = T;
  }
  if constexpr (DOT) {
    // a fold row's dot from its residues alone: the sum over m >= 0 of
    // c_m Re(conj Y[m] A[m]) is the sum over all m' in (-L, L) of
    // conj(c(m')) s_j T[q] (A(-m) = conj A(m) for a real ring), i.e.
    // sum_q T[q] conj(sum_j s_j c(q + j n)) = sum_q |T[q]|^2
    if (owns && (!splitf || gi == 0)) {
#pragma unroll
      for (int k = 0; k < kAliasMaxCols; ++k) {
        const int q = qs + k * (splitf ? 0 : LPR);
        if ((splitf && k > 0) || q >= n) continue;
        dsum = fma(wn, tq[k].x * tq[k].x + tq[k].y * tq[k].y, dsum);
      }
    }
  } else {
    __syncthreads();  // every read of the staged Y is done
  }

  // columns of the row's outputs: A / (w n) over the staged Y (write mode),
  // or the dot's terms c_m w n Re(conj Y[m] A[m]) (dot mode)
  auto out = [&](int m, cplx A) {
    if constexpr (DOT) {
      const cplx yv = Y(m);
      dsum += (m > 0 ? 2.0 * wn : wn) * (yv.x * A.x + yv.y * A.y);
    } else {
      ys[m * RW + rq] = A;
    }
  };
  if (kind == 1) {
    if constexpr (DOT)
      for (int m = li; m < L; m += LPR) out(m, Y(m));
  } else if (DOT) {
    // pair and fold rows: summed above
  } else if (kind == 2) {
#pragma unroll
    for (int k = 0; k < kAliasMaxCols; ++k) {
      const int m = li + k * LPR;
      if (m < L) out(m, av[k]);
    }
  } else if (owns) {
#pragma unroll
    for (int k = 0; k < kAliasMaxCols; ++k) {
      const int q = qs + k * (splitf ? 0 : LPR);
      if ((splitf && k > 0) || q >= n) continue;
      const int cnt = dv.floor(L - 1 - q) + 1;
      for (int kk = gi; kk < cnt; kk += G) {
        const double sj = ((kk & 1) && sgn < 0) ? -1.0 : 1.0;
        out(q + kk * n, cplx{sj * tq[k].x, sj * tq[k].y});
      }
    }
  }

  if constexpr (!DOT) {
    __syncthreads();
    // R = G - w n A by whole columns (this thread: row r0 + qt), the G loads
    // in flight together
    const int rw_row = kSpecBlock * blk + r0 + qt;
    const RingJob jq = a.rowjobs[rw_row];
    if (jq.nphi > 0) {
      const double c = jq.weight * jq.nphi * (a.alpha ? a.alpha[b] : 1.0);
      cplx gv[kAliasMaxCols];
#pragma unroll
      for (int k = 0; k < kAliasMaxCols; ++k) {
        const int idx = t + k * TPB;
        const int m = idx / RW;
        gv[k] = idx >= ntot ? cplx{0.0, 0.0}
                : a.g_tiled ? a.g[tile + (int64_t)m * kSpecBlock + r0 + qt]
                            : a.g[(int64_t)b * a.map_stride + (int64_t)rw_row * a.ncol + m];
      }
#pragma unroll
      for (int k = 0; k < kAliasMaxCols; ++k) {
        const int idx = t + k * TPB;
        if (idx >= ntot) continue;
        const cplx A = ys[idx];
        const cplx rv = {gv[k].x - c * A.x, gv[k].y - c * A.y};
        a.r[tile + (int64_t)(idx / RW) * kSpecBlock + r0 + qt] = rv;
        dsum = fma(rv.x, rv.x, fma(rv.y, rv.y, dsum));
      }
    }
  }
  if (DOT || a.part)
    alias_block_sum<TPB>(dsum, red,
                         a.part + (int64_t)b * a.part_map_stride + a.polar_part_off +
                             (int64_t)bi * kAliasSlots,
                         z, H);
}

// ------------------------------------------------------------------ launchers
namespace {

constexpr int kTpbAlias = 256;
}  // namespace

hipError_t launch_ring_alias(const RingAliasArgs& a, const JobSet& js, int batch, hipStream_t s) {
  const int njobs = js.n_pow2 + js.n_rest;
  if (batch == 0 || njobs == 0) return hipSuccess;
  RingAliasArgs b = a;
  b.jobs = js.jobs;
  b.jobs_end = njobs;
  hipLaunchKernelGGL((ring_alias_kernel<kTpbAlias, false>), dim3(njobs + (b.pad_rows > 0), batch),
                     dim3(kTpbAlias), 0, s, b);
  return hipGetLastError();
}

hipError_t launch_ring_alias_sumsq(const RingAliasArgs& a, const JobSet& js, int batch,
                                   double* part, double* sumsq, hipStream_t s) {
  const int njobs = ring_dot_jobs(js);
  if (batch == 0 || njobs == 0) return hipSuccess;
  RingAliasArgs b = a;
  b.jobs = js.jobs;
  b.part = part;
  b.jobs_end = njobs;
  hipLaunchKernelGGL((ring_alias_kernel<kTpbAlias, false>), dim3(njobs + (b.pad_rows > 0), batch),
                     dim3(kTpbAlias), 0, s, b);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(ring_dot_final_kernel, dim3(batch), dim3(256), 0, s, part, njobs, nullptr,
                     sumsq, nullptr);
  return hipGetLastError();
}

int ring_dot_jobs(const JobSet& js) { return js.n_pow2 + js.n_rest; }
int ring_dot_tiled_parts(int nblocks) { return nblocks * kAliasSlots; }
namespace {
// both tiled alias kernels over their blocks (part: null, or the per-block slots)
hipError_t launch_alias_tiled_pair(const RingAliasTiledArgs& a, int batch, bool dot,
                                   hipStream_t s) {
  if (a.n_belt > 0) {
    const dim3 grid(a.n_belt, batch, kAliasSplit);
    if (dot)
      hipLaunchKernelGGL((ring_alias_belt_kernel<kTpbAlias, true>), grid, dim3(kTpbAlias), 0, s,
                         a);
    else
      hipLaunchKernelGGL((ring_alias_belt_kernel<kTpbAlias, false>), grid, dim3(kTpbAlias), 0,
                         s, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (a.n_polar > 0) {
    if ((int64_t)a.L * 16 > kAliasPolarLds) return hipErrorInvalidValue;
    const bool small = dot && (int64_t)a.L * 16 <= kAliasDotLds;
    const int RW = alias_polar_rows(a.L, small ? kAliasDotLds : kAliasPolarLds);
    const int H = kSpecBlock / RW;
    const dim3 grid((unsigned)((a.n_polar + 7) / 8 * 8 * H), batch);
    const size_t lds = (size_t)RW * a.L * sizeof(cplx);
    constexpr int T = kAliasPolarTpb, TD = kAliasDotTpb;
    constexpr int B = kAliasPolarLds, BD = kAliasDotLds;
    if (small)
      hipLaunchKernelGGL((ring_alias_polar_kernel<true, TD, BD>), grid, dim3(TD), lds, s, a);
    else if (dot)
      hipLaunchKernelGGL((ring_alias_polar_kernel<true, T, B>), grid, dim3(T), lds, s, a);
    else
      hipLaunchKernelGGL((ring_alias_polar_kernel<false, T, B>), grid, dim3(T), lds, s, a);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// every row block's slots, polar blocks first
void full_part_layout(RingAliasTiledArgs& b) {
  b.part_map_stride = (int64_t)b.nblocks * kAliasSlots;
  b.polar_part_off = 0;
  b.belt_part_off = b.n_polar * kAliasSlots;
}
}  // namespace

hipError_t launch_ring_alias_tiled(const RingAliasTiledArgs& a, int batch, hipStream_t s) {
  if (batch == 0 || a.nblocks == 0) return hipSuccess;
  RingAliasTiledArgs b = a;
  b.part = nullptr;
  return launch_alias_tiled_pair(b, batch, false, s);
}

hipError_t launch_ring_alias_tiled_sumsq(const RingAliasTiledArgs& a, int batch, double* part,
                                         double* sumsq, hipStream_t s) {
  if (batch == 0 || a.nblocks == 0) return hipSuccess;
  RingAliasTiledArgs b = a;
  b.part = part;
  full_part_layout(b);
  hipError_t e = launch_alias_tiled_pair(b, batch, false, s);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(ring_dot_final_kernel, dim3(batch), dim3(256), 0, s, part,
                     a.nblocks * kAliasSlots, nullptr, sumsq, nullptr);
  return hipGetLastError();
}

hipError_t launch_ring_dot_tiled(const RingAliasTiledArgs& a, int batch, double* part,
                                 const double* num, double* pq, double* alpha, hipStream_t s) {
  if (batch == 0 || a.nblocks == 0) return hipSuccess;
  RingAliasTiledArgs b = a;
  b.part = part;
  b.alpha = nullptr;
  full_part_layout(b);
  hipError_t e = launch_alias_tiled_pair(b, batch, true, s);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(ring_dot_final_kernel, dim3(batch), dim3(256), 0, s, part,
                     a.nblocks * kAliasSlots, num, pq, alpha);
  return hipGetLastError();
}

hipError_t launch_ring_dot_tiled_polar(const RingAliasTiledArgs& a, int batch, double* part,
                                       int n_head, const double* num, double* pq, double* alpha,
                                       hipStream_t s) {
  if (batch == 0) return hipSuccess;
  RingAliasTiledArgs b = a;
  b.part = part;
  b.alpha = nullptr;
  b.n_belt = 0;
  b.part_map_stride = n_head + (int64_t)b.n_polar * kAliasSlots;
  b.polar_part_off = n_head;
  b.belt_part_off = 0;
  hipError_t e = launch_alias_tiled_pair(b, batch, true, s);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(ring_dot_final_kernel, dim3(batch), dim3(256), 0, s, part,
                     (int)b.part_map_stride, num, pq, alpha);
  return hipGetLastError();
}

hipError_t launch_ring_dot(const RingAliasArgs& a, const JobSet& js, int batch, double* part,
                           const double* num, double* pq, double* alpha, hipStream_t s) {
  const int njobs = ring_dot_jobs(js);
  if (batch == 0 || njobs == 0) return hipSuccess;
  RingAliasArgs b = a;
  b.jobs = js.jobs;
  b.part = part;
  b.alpha = nullptr;
  b.jobs_end = njobs;
  hipLaunchKernelGGL((ring_alias_kernel<kTpbAlias, true>), dim3(njobs, batch), dim3(kTpbAlias), 0,
                     s, b);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(ring_dot_final_kernel, dim3(batch), dim3(256), 0, s, part, njobs, num, pq,
                     alpha);
  return hipGetLastError();
}

hipError_t allow_large_lds_alias() {
  constexpr int T = kAliasPolarTpb, TD = kAliasDotTpb;
  constexpr int B = kAliasPolarLds, BD = kAliasDotLds;
  const void* alias[] = {(const void*)ring_alias_polar_kernel<true, T, B>,
                         (const void*)ring_alias_polar_kernel<false, T, B>,
                         (const void*)ring_alias_polar_kernel<true, TD, BD>};
  const int lds[] = {B, B, BD};
  for (int i = 0; i < 3; ++i) {
    const hipError_t e =
        hipFuncSetAttribute(alias[i], hipFuncAttributeMaxDynamicSharedMemorySize, lds[i]);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace s2h
