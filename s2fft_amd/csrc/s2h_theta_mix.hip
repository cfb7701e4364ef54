// MW / MWSS forward: the theta step between the ring FFTs and the projection
// as one matrix product per phi-column.
//
// The reference resamples the input rows to the MWSS grid at 2L
// (s2fft/utils/resampling.py: mw_to_mwss 248-355, upsample_by_two_mwss
// 64-160), weights those 2L + 1 rows and projects them.  Per column m every
// step is linear along theta, and with the parity sigma = (-1)^(m+spin) of
// the column it is one of two real operators U_sigma (input rows -> 2L + 1
// rows).  The projection of the weighted rows g against d (a trigonometric
// polynomial of parity sigma and degree below L) is a sum over the circle of
// 4L points, and only the harmonics |p| < L of w g enter it; the same sum over
// the circle of 2L points of w g reduced to those harmonics is
//   sum_{t<=2L} w_t g_t d(theta_t) = sum_{r<=L} (P_sigma g)_r d(pi r / L).
// So the forward's latitudinal rows are (P_sigma U_sigma) times the input
// column, on the L + 1 rows of the MWSS grid at L: half the rings to project.
//   P[r][t] = fold_r w_t (D(t - r) +- D(t + r)) / 4L,  fold = 1 at the poles, else 2,
//   U[t][j] = (K(t - j) +- K(t + j)) / n,
// D(x) = sin((2L-1)x/2) / sin(x/2) the Dirichlet kernel, K = D for MW (n = 2L - 1)
// and K = sin(Lx) cot(x/2) for MWSS (n = 2L, half the Nyquist term at +-L).
// Rows that are their own mirror image (theta = 0, pi) enter once.  Two cases
// go beyond the real operators:
//  * complex signals: the reference keeps the theta-Nyquist term at q = -L
//    alone, which adds -i sin(L theta_t) times the Nyquist coefficient N of
//    the column (N = n . column, zero for band-limited input): the rank-one
//    term i s n^T with s = P (-sin(L theta));
//  * the pole sample of an odd MW column: the reference mirrors the MWSS rows
//    after interpolating it, so its column of U is U_mwss times that row vector.
// The recursion evaluates d at the colatitudes whose cosines are FP64 numbers,
// theta_r + delta_r with |delta_r| up to eps / 2 over sin theta, which moves d
// by up to L delta.  The operators absorb it: sums against d(theta_r) become
// sums against d(theta_r + delta_r) by C -= (delta_r kappa'(r - r'))^T C, kappa
// the trigonometric cardinal function of the 2L points, kappa'(pi k / L) =
// (-1)^k cot(pi k / 2L) / 2.  (Half the rings average half as many rounding
// errors: without this the forward's error at L = 512 was 5.8e-14 instead of
// the 5.4e-14 of the 2L + 1 rings.)
// The adjoint uses the transposed matrices.
// The BF16 projections take the 2L + 1 rows w U instead (`wide`): their error is the
// rounding of rows and d, which twice the rows average out by sqrt 2.  From L + 1 rows
// the single BF16 projection had an error of 2.2e-3 instead of 1.5e-3, the split one
// 4.1e-6 instead of 2.9e-6 (L = 24 to 1024).  Split BF16 forward, MW L = 512, 8 maps:
// 677 us from 2L + 1 rows (493 from L + 1; the column FFT chain 7.9 ms).
//
// What bounds it: 8 L^2 flops per complex element of the column on
// V_MFMA_F64_16X16X4F64.  The operators are shared by every map, spin and column of one
// parity, so they are stored packed in the A-operand order (a wave's tile load is 512
// contiguous bytes, resident in L2).  Two kernels: theta_mix_kernel gathers the spectra
// (the B operand) straight into registers, 16 lanes reading 8 columns of one parity while
// the wave of the other parity beside it uses the rest of the lines, with loads D K-steps
// ahead of the products (MW L = 128, one map: 9.7 us; the column FFT chain 265 us);
// theta_mix_lds_kernel, for launches that fill the card, passes both through LDS (MW L =
// 512, spin 2, 64 maps: 1.55 ms, 44 TFLOP/s of products, 1.69 from registers; the chain
// 60.0 ms).  The projection of half the rings takes 1.03 ms there instead of 2.78.
#include <map>
#include <memory>
#include <mutex>
#include <tuple>
#include <vector>

#include "s2h_lat_common.h"
#include "s2h_plan.h"

namespace s2h {

namespace {

// sin(pi num / den) from the exactly reduced fraction (den > 0).
__device__ double sinpi_frac(int64_t num, int64_t den) {
  int64_t r = num % (2 * den);
  if (r < 0) r += 2 * den;
  double sg = 1.0;
  if (r >= den) {
    r -= den;
    sg = -1.0;
  }
  if (2 * r > den) r = den - r;
  return sg * sinpi((double)r / (double)den);
}
__device__ double cospi_frac(int64_t num, int64_t den) {
  return sinpi_frac(den - 2 * num, 2 * den);
}
// D(x) and sin(Lx) cot(x/2) at x / 2 = pi num / den.
__device__ double dirichlet(int L, int64_t num, int64_t den) {
  if (num % den == 0) return 2.0 * L - 1.0;
  return sinpi_frac((2 * L - 1) * num, den) / sinpi_frac(num, den);
}
__device__ double dirichlet_split(int L, int64_t num, int64_t den) {
  if (num % den == 0) return 2.0 * L;
  return sinpi_frac(2 * L * num, den) * cospi_frac(num, den) / sinpi_frac(num, den);
}

// U_mwss[t][j] of one parity (sg = +-1)
__device__ double u_mwss(int L, int t, int j, double sg) {
  const double a = dirichlet_split(L, t - 2 * j, 4 * L);
  if (j == 0 || j == L) return a / (2.0 * L);
  return (a + sg * dirichlet_split(L, t + 2 * j, 4 * L)) / (2.0 * L);
}

// U[par][t][j], t <= 2L, j < K (K = L for MW, L + 1 for MWSS)
__global__ void __launch_bounds__(kThreads) mix_up_kernel(int L, int K, int mw, double* u) {
  const int64_t n = (int64_t)(2 * L + 1) * K;
  const int par = blockIdx.y;
  const double sg = par ? -1.0 : 1.0;
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kThreads) {
    const int t = (int)(i / K), j = (int)(i % K);
    double v;
    if (!mw) {
      v = u_mwss(L, t, j, sg);
    } else {
      // theta_t -+ theta_j over 2: pi (t (2L-1) -+ 2L (2j+1)) / (4L (2L-1))
      const int64_t den = (int64_t)4 * L * (2 * L - 1), at = (int64_t)t * (2 * L - 1),
                    aj = (int64_t)2 * L * (2 * j + 1);
      if (j < L - 1) {
        v = (dirichlet(L, at - aj, den) + sg * dirichlet(L, at + aj, den)) / (2.0 * L - 1.0);
      } else if (!par) {
        v = dirichlet(L, at - aj, den) / (2.0 * L - 1.0);
      } else {
        continue;  // mix_pole_kernel
      }
    }
    u[par * n + i] = v;
  }
}

// the pole column j = L - 1 of odd MW columns: one workgroup per row t
__global__ void __launch_bounds__(kThreads) mix_pole_kernel(int L, double* u) {
  __shared__ double red[kThreads];
  const int t = blockIdx.x;
  const int64_t den = (int64_t)4 * L * (2 * L - 1), aj = (int64_t)2 * L * (2 * L - 1);
  double v = 0.0;
  for (int r = threadIdx.x; r <= L; r += kThreads)
    v = fma(u_mwss(L, t, r, -1.0),
            dirichlet(L, (int64_t)2 * r * (2 * L - 1) - aj, den) / (2.0 * L - 1.0), v);
  red[threadIdx.x] = v;
  __syncthreads();
  for (int o = kThreads / 2; o > 0; o >>= 1) {
    if (threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) u[((int64_t)(2 * L + 1) + t) * L + L - 1] = red[0];
}

// P[par][r][t] with the weights w_t (times phi)
__global__ void __launch_bounds__(kThreads) mix_down_kernel(int L, const double* w, double phi,
                                                            double* pm) {
  const int64_t n = (int64_t)(L + 1) * (2 * L + 1);
  const int par = blockIdx.y;
  const double sg = par ? -1.0 : 1.0;
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kThreads) {
    const int r = (int)(i / (2 * L + 1)), t = (int)(i % (2 * L + 1));
    const double fold = r == 0 || r == L ? 1.0 : 2.0;
    pm[par * n + i] = phi * fold / (4.0 * L) * w[t] *
                      (dirichlet(L, t - 2 * r, 4 * L) + sg * dirichlet(L, t + 2 * r, 4 * L));
  }
}

// M[par][r'][r] = -delta_r (kappa'(r - r') +- kappa'(r + r')), delta_0 = delta_L = 0
__device__ double cardinal_slope(int L, int k) {
  k %= 2 * L;
  if (k == 0) return 0.0;
  const double c = cospi_frac(k, 2 * L) / sinpi_frac(k, 2 * L);
  return (k & 1) ? -0.5 * c : 0.5 * c;
}
__global__ void __launch_bounds__(kThreads) mix_shift_kernel(int L, const double* delta,
                                                             double* sm) {
  const int64_t n = (int64_t)(L + 1) * (L + 1);
  const int par = blockIdx.y;
  const double sg = par ? -1.0 : 1.0;
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kThreads) {
    const int rp = (int)(i / (L + 1)), r = (int)(i % (L + 1));
    double v = cardinal_slope(L, r - rp);
    if (rp != 0 && rp != L) v += sg * cardinal_slope(L, r + rp);
    sm[par * n + i] = -delta[r] * v;
  }
}

__global__ void __launch_bounds__(kThreads) mix_add_kernel(int64_t n, const double* x, double* y) {
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kThreads)
    y[i] += x[i];
}

// U -> w U (times phi), and its rank-one vector w (-sin(L theta_t))
__global__ void __launch_bounds__(kThreads) mix_weight_kernel(int L, int K, const double* w,
                                                              double phi, double* u, double* su) {
  const int64_t T = 2 * L + 1, n = 2 * T * K;
  const int64_t i0 = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  for (int64_t i = i0; i < n; i += (int64_t)gridDim.x * kThreads) u[i] *= phi * w[i / K % T];
  for (int64_t i = i0; i < 2 * T; i += (int64_t)gridDim.x * kThreads) {
    const int t = (int)(i % T);
    su[i] = t & 1 ? ((t & 3) == 1 ? -phi : phi) * w[t] : 0.0;
  }
}

// n (K entries) and s (L + 1 entries) of the rank-one Nyquist term per parity
__global__ void __launch_bounds__(kThreads) mix_nyquist_kernel(int L, int K, int mw,
                                                               const double* pm, double* nv,
                                                               double* sv) {
  const int par = blockIdx.y;
  const int i = blockIdx.x * kThreads + threadIdx.x;
  if (i < K) {
    double v = 0.0;
    if (mw) {
      if (par && i == K - 1) v = ((L & 1) ? -1.0 : 1.0) * (2.0 * L - 2.0) / (2.0 * L - 1.0) / (2.0 * L);
    } else {
      v = ((i & 1) ? -1.0 : 1.0) / (2.0 * L);
      if (i != 0 && i != L) v = par ? 0.0 : 2.0 * v;
    }
    nv[par * K + i] = v;
  }
  if (i <= L) {
    const double* row = pm + ((int64_t)par * (L + 1) + i) * (2 * L + 1);
    double v = 0.0;
    for (int t = 1; t <= 2 * L; t += 2) v += (t & 3) == 1 ? -row[t] : row[t];
    sv[par * (L + 1) + i] = v;
  }
}

// C[par] = A[par] B[par]: (R x T) (T x K), row-major, once per plan
constexpr int kGT = 16;
__global__ void __launch_bounds__(kGT * kGT) mix_product_kernel(int R, int T, int K,
                                                                const double* a, const double* b,
                                                                double* c) {
  __shared__ double sa[kGT][kGT + 1], sb[kGT][kGT + 1];
  const int tx = threadIdx.x % kGT, ty = threadIdx.x / kGT;
  const int r = blockIdx.y * kGT + ty, k = blockIdx.x * kGT + tx;
  a += (int64_t)blockIdx.z * R * T;
  b += (int64_t)blockIdx.z * T * K;
  double acc = 0.0;
  for (int t0 = 0; t0 < T; t0 += kGT) {
    sa[ty][tx] = r < R && t0 + tx < T ? a[(int64_t)r * T + t0 + tx] : 0.0;
    sb[ty][tx] = k < K && t0 + ty < T ? b[(int64_t)(t0 + ty) * K + k] : 0.0;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kGT; ++q) acc = fma(sa[ty][q], sb[q][tx], acc);
    __syncthreads();
  }
  if (r < R && k < K) c[(int64_t)blockIdx.z * R * K + (int64_t)r * K + k] = acc;
}

// The interior rows come first, the pole rows last: position i -> MWSS row
// (0 .. L, wide: 0 .. 2L).  An output tile of pole rows alone is wanted for two columns only.
__host__ __device__ __forceinline__ int mix_row(int i, int L) {
  return i < L - 1 ? i + 1 : i == L - 1 ? L : 0;
}

// Packs one operator for the products: tile (rt, kt) holds rows 16 rt + lane % 16
// and k = 4 kt + lane / 16 at ((rt KT + kt) 64 + lane).  forward: rows are
// mix_row positions, k the input rows; adjoint: the transpose.
__global__ void __launch_bounds__(kThreads) mix_pack_kernel(int L, int K, const double* c, int RT,
                                                            int KT, int adjoint, double* out) {
  const int64_t n = (int64_t)RT * KT * 64;
  const int par = blockIdx.y;
  const double* cm = c + (int64_t)par * (L + 1) * K;
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * kThreads) {
    const int lane = (int)(i & 63);
    const int64_t tile = i >> 6;
    const int r = 16 * (int)(tile / KT) + (lane & 15), k = 4 * (int)(tile % KT) + (lane >> 4);
    const int row = adjoint ? k : r, col = adjoint ? r : k;  // row: position, col: input row
    out[par * n + i] = row <= L && col < K ? cm[(int64_t)mix_row(row, L) * K + col] : 0.0;
  }
}

constexpr int kRowTiles = 2;  // packed operators hold whole groups of 2 row tiles
constexpr int kStepPad = 8;   // and of 8 K-steps (zeros)
int pad_to(int n, int q) { return (n + q - 1) / q * q; }

}  // namespace

struct ThetaMix {
  int device = 0, L = 0, K = 0, mw = 0;
  double* fwd = nullptr;  // packed [parity][RT][KT][64]
  double* adj = nullptr;
  double* wide = nullptr; // w U on the 2L + 1 rows of MWSS at 2L
  double* nv = nullptr;   // [parity][K]
  double* sv = nullptr;   // [parity][L + 1], MWSS row order
  double* su = nullptr;   // [parity][2L + 1], for wide
  ~ThetaMix() {
    int cur = 0;
    (void)hipGetDevice(&cur);
    (void)hipSetDevice(device);
    for (double* q : {fwd, adj, wide, nv, sv, su})
      if (q) (void)hipFree(q);
    (void)hipSetDevice(cur);
  }
};

namespace {
int fwd_rt(int L) { return pad_to((L + 1 + 15) / 16, kRowTiles); }
int fwd_kt(int K) { return pad_to((K + 3) / 4, kStepPad); }
int wide_rt(int L) { return fwd_rt(2 * L); }
int adj_rt(int K) { return pad_to((K + 15) / 16, kRowTiles); }
int adj_kt(int L) { return pad_to((L + 1 + 3) / 4, kStepPad); }

std::mutex g_mix_mu;
std::map<std::tuple<int, int, int>, std::weak_ptr<ThetaMix>> g_mix;

int mix_build(ThetaMix* x, const std::vector<double>& weights, const std::vector<double>& delta,
              double phi) {
  const int L = x->L, K = x->K;
  const int64_t T = 2 * L + 1;
  struct Tmp {
    void* p[7] = {};
    ~Tmp() {
      for (void* q : p)
        if (q) (void)hipFree(q);
    }
    double* get(int i, int64_t n) {
      return hipMalloc(&p[i], sizeof(double) * n) == hipSuccess ? static_cast<double*>(p[i])
                                                                : nullptr;
    }
  } tmp;
  double* u = tmp.get(0, 2 * T * K);
  double* pm = tmp.get(1, 2 * T * (L + 1));
  double* c = tmp.get(2, (int64_t)2 * (L + 1) * K);
  double* w = tmp.get(3, T);
  double* dl = tmp.get(4, L + 1);
  double* sm = tmp.get(5, (int64_t)2 * (L + 1) * (L + 1));
  double* dc = tmp.get(6, 2 * T * (L + 1));
  const int64_t nf = (int64_t)2 * fwd_rt(L) * fwd_kt(K) * 64,
                nw = (int64_t)2 * wide_rt(L) * fwd_kt(K) * 64,
                na = (int64_t)2 * adj_rt(K) * adj_kt(L) * 64;
  if (!u || !pm || !c || !w || !dl || !sm || !dc ||
      hipMalloc(&x->fwd, sizeof(double) * nf) != hipSuccess ||
      hipMalloc(&x->adj, sizeof(double) * na) != hipSuccess ||
      hipMalloc(&x->wide, sizeof(double) * nw) != hipSuccess ||
      hipMalloc(&x->su, sizeof(double) * 2 * T) != hipSuccess ||
      hipMalloc(&x->nv, sizeof(double) * 2 * K) != hipSuccess ||
      hipMalloc(&x->sv, sizeof(double) * 2 * (L + 1)) != hipSuccess)
    return S2H_ERR_NOMEM;
  if (hipMemcpy(w, weights.data(), sizeof(double) * T, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemcpy(dl, delta.data(), sizeof(double) * (L + 1), hipMemcpyHostToDevice) != hipSuccess)
    return S2H_ERR_HIP;
  const auto blocks = [](int64_t n) {
    const int64_t b = (n + kThreads - 1) / kThreads;
    return dim3((unsigned)(b < 8192 ? b : 8192), 2);
  };
  hipLaunchKernelGGL(mix_up_kernel, blocks(T * K), dim3(kThreads), 0, 0, L, K, x->mw, u);
  if (x->mw) hipLaunchKernelGGL(mix_pole_kernel, dim3((unsigned)T), dim3(kThreads), 0, 0, L, u);
  hipLaunchKernelGGL(mix_down_kernel, blocks(T * (L + 1)), dim3(kThreads), 0, 0, L, w, phi, pm);
  // the shift acts on the rows of P, so that C and s take it alike
  hipLaunchKernelGGL(mix_shift_kernel, blocks((int64_t)(L + 1) * (L + 1)), dim3(kThreads), 0, 0, L,
                     dl, sm);
  hipLaunchKernelGGL(mix_product_kernel, dim3(((int)T + kGT - 1) / kGT, (L + kGT) / kGT, 2),
                     dim3(kGT * kGT), 0, 0, L + 1, L + 1, (int)T, sm, pm, dc);
  hipLaunchKernelGGL(mix_add_kernel, dim3(blocks(2 * T * (L + 1)).x), dim3(kThreads), 0, 0,
                     2 * T * (L + 1), dc, pm);
  hipLaunchKernelGGL(mix_nyquist_kernel, dim3((L + kThreads) / kThreads, 2), dim3(kThreads), 0, 0,
                     L, K, x->mw, pm, x->nv, x->sv);
  hipLaunchKernelGGL(mix_product_kernel, dim3((K + kGT - 1) / kGT, (L + kGT) / kGT, 2),
                     dim3(kGT * kGT), 0, 0, L + 1, (int)T, K, pm, u, c);
  hipLaunchKernelGGL(mix_pack_kernel, blocks(nf / 2), dim3(kThreads), 0, 0, L, K, c, fwd_rt(L),
                     fwd_kt(K), 0, x->fwd);
  hipLaunchKernelGGL(mix_pack_kernel, blocks(na / 2), dim3(kThreads), 0, 0, L, K, c, adj_rt(K),
                     adj_kt(L), 1, x->adj);
  hipLaunchKernelGGL(mix_weight_kernel, dim3(blocks(2 * T * K).x), dim3(kThreads), 0, 0, L, K, w,
                     phi, u, x->su);
  hipLaunchKernelGGL(mix_pack_kernel, blocks(nw / 2), dim3(kThreads), 0, 0, 2 * L, K, u,
                     wide_rt(L), fwd_kt(K), 0, x->wide);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(0);
  return e == hipSuccess ? S2H_OK : S2H_ERR_HIP;
}
}  // namespace

// The operators of (device, sampling, L), shared by every live plan that uses
// them (they do not depend on the spin) and freed with the last one.  They are built
// with the plan, since the calls neither allocate nor wait: 64 L^2 bytes (the
// projection's, its transpose for gradients, and twice that for BF16), 268 MB at L =
// 2048, and 128 L^2 bytes of temporaries meanwhile.
int theta_mix_get(int device, bool mw, int L, const std::vector<double>& weights,
                  const std::vector<double>& delta, std::shared_ptr<ThetaMix>* out) {
  std::lock_guard<std::mutex> lock(g_mix_mu);
  auto& slot = g_mix[std::make_tuple(device, mw ? 1 : 0, L)];
  *out = slot.lock();
  if (*out) return S2H_OK;
  auto x = std::make_shared<ThetaMix>();
  x->device = device;
  x->L = L;
  x->K = mw ? L : L + 1;
  x->mw = mw ? 1 : 0;
  // the phi zero-padding of MW -> MWSS scales by 2L / (2L - 1)
  const int st = mix_build(x.get(), weights, delta, mw ? (2.0 * L) / (2.0 * L - 1.0) : 1.0);
  if (st != S2H_OK) return st;
  slot = x;
  *out = x;
  return S2H_OK;
}

// ------------------------------------------------------------------ the product
namespace {

struct MixKernelArgs {
  const double* mat;        // packed [parity][RT][KT][64]
  const double* q;          // [parity][K]: v = q . column (full mode), by input row
  const double* p;          // [parity][rows]: out += i sgn p v, by output row; null: no term
  double sgn;
  int vmode[2];             // per parity: 0 none, 1 the first and last row of q, 2 all of q
  const cplx* in;
  int64_t in_map_stride;
  cplx* out;
  int64_t out_map_stride;
  int ncol, m_lo, spin, spin_step;
  int last;                 // of the MWSS rows on one side: rows 0 .. last
  int K, R;                 // input rows, output rows
  int KT, KTpad, RT;        // K-steps in use, K-steps / row tiles of the packed operator
  int in_poles, out_poles;  // rows in mix_row order
  int out_tiled;            // out in blocks of 8 rows (spec_row)
  int row_blocks, col_blocks;
};

__device__ __forceinline__ int mix_at(int i, int L, int poles) { return poles ? mix_row(i, L) : i; }

// One workgroup: MT 16-row tiles x 2 NT 16 columns; its four waves take the
// two column parities of the two column halves, so that the two waves of one
// half read the same lines and the two of one parity the same operator tiles.
// blockIdx.x -> (row block, column block): the row blocks of one column block
// follow each other on one XCD and read its spectra through that XCD's L2.
template <int MT, int NT, int D, bool VFULL>
__global__ void __launch_bounds__(256) theta_mix_kernel(MixKernelArgs a) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int j = lane & 15, kq = lane >> 4, comp = j & 1;
  const int seq = blockIdx.x >> 3;
  const int rb = seq % a.row_blocks;
  const int cb = (seq / a.row_blocks) * 8 + (blockIdx.x & 7);
  if (cb >= a.col_blocks) return;
  const int b = blockIdx.y;
  const int par = wave & 1;
  const int spin = a.spin + a.spin_step * b;
  const int c0 = (2 * cb + (wave >> 1)) * (16 * NT);
  if (c0 >= a.ncol) return;
  const int r0 = rb * 16 * MT;
  if (a.out_poles && r0 >= a.last - 1) {
    // pole rows only: the pole terms read the columns m = +-spin
    const int cs = spin - a.m_lo, cn = -spin - a.m_lo;
    if (!(cs >= c0 && cs < c0 + 16 * NT) && !(cn >= c0 && cn < c0 + 16 * NT)) return;
  }
  // columns c0 + 2 (8 nt + j / 2) + off have the parity (m + spin) % 2 = par
  const int off = (par + a.m_lo + spin) & 1;
  const double* bp[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    int col = c0 + 2 * (8 * nt + (j >> 1)) + off;
    if (col >= a.ncol) col = off < a.ncol ? off : 0;  // in bounds; not stored
    bp[nt] = reinterpret_cast<const double*>(a.in + (int64_t)b * a.in_map_stride + col) + comp;
  }
  const double* ap = a.mat + ((int64_t)par * a.RT + (int64_t)rb * MT) * a.KTpad * 64 + lane;
  const bool full = VFULL && a.vmode[par] == 2;
  const double* qv = a.q + par * a.K;

  lat::v4d acc[MT][NT], accv[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    accv[nt] = lat::v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt][nt] = lat::v4d{0.0, 0.0, 0.0, 0.0};
  }
  double av[D][MT], bv[D][NT], qa[D];
  // K-step kt: the packed operator is zero past K, and so is the operand here
  // (the rows past K repeat row K - 1's address)
  auto load = [&](int kt, double (&va)[MT], double (&vb)[NT], double& vq) {
    const int k = 4 * kt + kq;
    const int row = mix_at(k < a.K ? k : a.K - 1, a.last, a.in_poles);
    const int64_t ro = 2 * (int64_t)row * a.ncol;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) va[mt] = ap[((int64_t)mt * a.KTpad + kt) * 64];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const double v = bp[nt][ro];
      vb[nt] = k < a.K ? v : 0.0;
    }
    vq = full && k < a.K ? qv[row] : 0.0;
  };
#pragma unroll
  for (int u = 0; u < D; ++u) load(u, av[u], bv[u], qa[u]);
  for (int kt = 0; kt < a.KT; kt += D) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      double ca[MT], cb2[NT];
      const double cq = qa[u];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) ca[mt] = av[u][mt];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) cb2[nt] = bv[u][nt];
      // the last group re-reads its own steps (in bounds, unused)
      load(kt + D < a.KT ? kt + D + u : kt + u, av[u], bv[u], qa[u]);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          acc[mt][nt] = lat::Mma<double>::run(ca[mt], cb2[nt], acc[mt][nt]);
      if (full) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) accv[nt] = lat::Mma<double>::run(cq, cb2[nt], accv[nt]);
      }
    }
  }

  // rank-one term: every row of accv holds v; sparse q reads its two rows
  const bool term = a.p && a.vmode[par] != 0;
  double vv[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    vv[nt] = accv[nt][0];
    if (term && !full)
      vv[nt] = qv[0] * bp[nt][0] + qv[a.K - 1] * bp[nt][2 * (int64_t)(a.K - 1) * a.ncol];
    // i v: the real part takes -Im v, the imaginary part Re v
    vv[nt] = a.sgn * (comp ? 1.0 : -1.0) * __shfl_xor(vv[nt], 1);
  }
  double* ob = reinterpret_cast<double*>(a.out + (int64_t)b * a.out_map_stride) + comp;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = r0 + 16 * mt + lat::Mma<double>::row_of(r, kq);
      if (i >= a.R) continue;
      const int row = mix_at(i, a.last, a.out_poles);
      const double pr = term ? a.p[par * a.R + row] : 0.0;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        const int col = c0 + 2 * (8 * nt + (j >> 1)) + off;
        if (col < a.ncol) {
          double v = acc[mt][nt][r];
          if (term) v = fma(pr, vv[nt], v);
          ob[2 * (spec_row(row, a.ncol, a.out_tiled) + col * spec_cstride(a.out_tiled))] = v;
        }
      }
    }
  }
}

// The same product for launches that fill the card: operator and spectra pass
// through LDS, so that the four waves of a workgroup (two column parities, two
// column halves) share what they load and the matrix cores, not the L1's 64 bytes
// per cycle, set the pace.  One workgroup: 64 rows of both parities x 64 columns;
// a wave 4 row tiles x 2 column tiles; 16 input rows per LDS chunk, double-buffered
// through registers (72 KB: two workgroups per CU).  The spectra are staged by
// parity, (re, im) of 32 columns per input row, rows 640 bytes apart so that the two
// rows of a half wave use all banks.  At MW L = 512, 64 maps the matrix cores are busy
// for 68 % of its 1550 us (loads one chunk ahead instead of two: 2140 us).
constexpr int kMixRows = 64, kMixCols = 64, kMixK = 16;
constexpr int kMixPad = 80;  // doubles per staged row of one parity

template <bool VFULL>
__global__ void __launch_bounds__(256, 2) theta_mix_lds_kernel(MixKernelArgs a) {
  constexpr int MT = 4, NT = 2, KS = kMixK / 4;
  __shared__ __attribute__((aligned(16))) double as[2][2][MT][KS][64];  // [buffer][parity][tile][step]
  __shared__ __attribute__((aligned(16))) double bs[2][2][kMixK][kMixPad];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int j = lane & 15, kq = lane >> 4, comp = j & 1;
  const int seq = blockIdx.x >> 3;
  const int rb = seq % a.row_blocks;
  const int cb = (seq / a.row_blocks) * 8 + (blockIdx.x & 7);
  if (cb >= a.col_blocks) return;
  const int b = blockIdx.y;
  const int par = wave & 1, half = wave >> 1;
  const int spin = a.spin + a.spin_step * b;
  const int c0 = cb * kMixCols, r0 = rb * kMixRows;
  if (a.out_poles && r0 >= a.last - 1) {
    // pole rows only: the pole terms read the columns m = +-spin
    const int cs = spin - a.m_lo, cn = -spin - a.m_lo;
    if (!(cs >= c0 && cs < c0 + kMixCols) && !(cn >= c0 && cn < c0 + kMixCols)) return;
  }
  const int off = (a.m_lo + spin) & 1;  // parity of column c0 (c0 is even)
  const cplx* in = a.in + (int64_t)b * a.in_map_stride;

  // staging: 4 columns' values and 8 operator values per thread and chunk.  Column
  // c0 + c (c = tid % 64) goes to parity (c + off) % 2, place c / 2; the input rows
  // tid / 64 + 4 i.
  const int sc = tid & 63, sr = tid >> 6;
  const int scol = c0 + sc < a.ncol ? c0 + sc : a.ncol - 1;  // in bounds; not stored
  struct Staged {
    cplx b[4];
    double2 a[4];
  };
  // addresses: a uniform base per load plus the thread's own offset.  Input rows up to
  // `plain` follow their index (with poles: one further); the rest go through mix_at
  const int plain = a.in_poles ? a.last - 1 : a.K;
  const unsigned boff = 16u * (unsigned)(sr * a.ncol + scol);
  unsigned aoff[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    // tile of element tid + 256 i of a parity's [tile][step][64] pairs; tiles past the
    // operator's: the last again, not stored
    const int mt = 2 * i + (tid >> 7), rt = rb * MT + mt < a.RT ? rb * MT + mt : a.RT - 1;
    aoff[i] = 8u * (unsigned)(rt * a.KTpad * 64 + 2 * (tid & 127));
  }
  const auto load = [&](int kc, Staged& v) {
    if ((kc + 1) * kMixK <= plain) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const cplx* base = in + (int64_t)(kc * kMixK + 4 * i + (a.in_poles ? 1 : 0)) * a.ncol;
        v.b[i] = *reinterpret_cast<const cplx*>(reinterpret_cast<const char*>(base) + boff);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k = kc * kMixK + sr + 4 * i;
        v.b[i] = in[(int64_t)mix_at(k < a.K ? k : a.K - 1, a.last, a.in_poles) * a.ncol + scol];
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const double* base = a.mat + ((int64_t)(i >> 1) * a.RT * a.KTpad + kc * KS) * 64;
      v.a[i] = *reinterpret_cast<const double2*>(reinterpret_cast<const char*>(base) + aoff[i & 1]);
    }
  };
  double* bst = &bs[0][(sc + off) & 1][sr][2 * (sc >> 1)];
  double2* ast = reinterpret_cast<double2*>(&as[0][0][0][0][0]) + tid;
  const auto stage = [&](int kc, const Staged& v) {
    const int buf = kc & 1;
    const bool whole = (kc + 1) * kMixK <= a.K;  // else zero past K, as the operator is
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const bool in_k = whole || kc * kMixK + sr + 4 * i < a.K;
      *reinterpret_cast<cplx*>(bst + buf * (2 * kMixK * kMixPad) + 4 * i * kMixPad) =
          cplx{in_k ? v.b[i].x : 0.0, in_k ? v.b[i].y : 0.0};
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) ast[buf * (2 * MT * KS * 32) + 256 * i] = v.a[i];
  };

  lat::v4d acc[MT][NT], accv[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    accv[nt] = lat::v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt][nt] = lat::v4d{0.0, 0.0, 0.0, 0.0};
  }
  const bool full = VFULL && a.vmode[par] == 2;
  const double* qv = a.q + par * a.K;
  const int chunks = (a.K + kMixK - 1) / kMixK;
  const auto products = [&](int kc) {
    const int buf = kc & 1;
#pragma unroll
    for (int u = 0; u < KS; ++u) {
      double ca[MT], cbv[NT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) ca[mt] = as[buf][par][mt][u][lane];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) cbv[nt] = bs[buf][par][4 * u + kq][(half * NT + nt) * 16 + j];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          acc[mt][nt] = lat::Mma<double>::run(ca[mt], cbv[nt], acc[mt][nt]);
      if (full) {
        const int k = kc * kMixK + 4 * u + kq;
        const double cq = k < a.K ? qv[mix_at(k, a.last, a.in_poles)] : 0.0;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) accv[nt] = lat::Mma<double>::run(cq, cbv[nt], accv[nt]);
      }
    }
  };
  // loads run two chunks ahead of the products, LDS one (past the end: the last
  // chunk again, unused)
  Staged va, vb;
  load(0, va);
  load(min(1, chunks - 1), vb);
  stage(0, va);
  __syncthreads();
  for (int kc = 0; kc < chunks; kc += 2) {
    load(min(kc + 2, chunks - 1), va);
    products(kc);
    stage(kc + 1, vb);
    __syncthreads();
    if (kc + 1 >= chunks) break;
    load(min(kc + 3, chunks - 1), vb);
    products(kc + 1);
    stage(kc + 2, va);
    __syncthreads();
  }

  // rank-one term: every row of accv holds v; sparse q reads its two rows
  const bool term = a.p && a.vmode[par] != 0;
  int col[NT];
  double vv[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    // place 8 (2 half + nt) + j / 2 of the parity
    col[nt] = c0 + 2 * ((half * NT + nt) * 8 + (j >> 1)) + ((par + off) & 1);
    vv[nt] = accv[nt][0];
    if (term && !full) {
      const double* bp = reinterpret_cast<const double*>(in + (col[nt] < a.ncol ? col[nt] : 0)) + comp;
      vv[nt] = qv[0] * bp[0] + qv[a.K - 1] * bp[2 * (int64_t)(a.K - 1) * a.ncol];
    }
    // i v: the real part takes -Im v, the imaginary part Re v
    vv[nt] = a.sgn * (comp ? 1.0 : -1.0) * __shfl_xor(vv[nt], 1);
  }
  double* ob = reinterpret_cast<double*>(a.out + (int64_t)b * a.out_map_stride) + comp;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = r0 + 16 * mt + lat::Mma<double>::row_of(r, kq);
      if (i >= a.R) continue;
      const int row = mix_at(i, a.last, a.out_poles);
      const double pr = term ? a.p[par * a.R + row] : 0.0;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        if (col[nt] < a.ncol) {
          double v = acc[mt][nt][r];
          if (term) v = fma(pr, vv[nt], v);
          ob[2 * (spec_row(row, a.ncol, a.out_tiled) + col[nt] * spec_cstride(a.out_tiled))] = v;
        }
      }
    }
  }
}

hipError_t mix_launch_lds(MixKernelArgs k, int batch, hipStream_t s) {
  k.row_blocks = (k.R + kMixRows - 1) / kMixRows;
  k.col_blocks = (k.ncol + kMixCols - 1) / kMixCols;
  const unsigned gx = (unsigned)(8 * k.row_blocks * ((k.col_blocks + 7) / 8));
  if (k.p && (k.vmode[0] == 2 || k.vmode[1] == 2))
    hipLaunchKernelGGL(theta_mix_lds_kernel<true>, dim3(gx, batch), dim3(256), 0, s, k);
  else
    hipLaunchKernelGGL(theta_mix_lds_kernel<false>, dim3(gx, batch), dim3(256), 0, s, k);
  return hipGetLastError();
}

template <int MT, int NT, int D>
hipError_t mix_launch(MixKernelArgs k, int batch, hipStream_t s) {
  k.KT = pad_to(k.KT, D);
  k.row_blocks = (k.R + 16 * MT - 1) / (16 * MT);
  k.col_blocks = (k.ncol + 32 * NT - 1) / (32 * NT);
  const unsigned gx = (unsigned)(8 * k.row_blocks * ((k.col_blocks + 7) / 8));
  if (k.p && (k.vmode[0] == 2 || k.vmode[1] == 2))
    hipLaunchKernelGGL((theta_mix_kernel<MT, NT, D, true>), dim3(gx, batch), dim3(256), 0, s, k);
  else
    hipLaunchKernelGGL((theta_mix_kernel<MT, NT, D, false>), dim3(gx, batch), dim3(256), 0, s, k);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_theta_mix(const ThetaMix* x, const ThetaMixArgs& a, int batch, hipStream_t s) {
  if (batch == 0 || a.ncol == 0) return hipSuccess;
  MixKernelArgs k{};
  const int L = x->L;
  k.last = a.wide ? 2 * L : L;
  k.K = a.adjoint ? L + 1 : x->K;
  k.R = a.adjoint ? x->K : k.last + 1;
  k.mat = a.adjoint ? x->adj : a.wide ? x->wide : x->fwd;
  k.RT = a.adjoint ? adj_rt(x->K) : fwd_rt(k.last);
  k.KTpad = a.adjoint ? adj_kt(L) : fwd_kt(x->K);
  k.KT = (k.K + 3) / 4;
  k.in_poles = a.adjoint;
  k.out_poles = !a.adjoint;
  k.out_tiled = a.out_tiled;
  k.in = a.in;
  k.in_map_stride = a.in_map_stride;
  k.out = a.out;
  k.out_map_stride = a.out_map_stride;
  k.ncol = a.ncol;
  k.m_lo = a.m_lo;
  k.spin = a.spin;
  k.spin_step = a.spin_step;
  k.q = a.adjoint ? x->sv : x->nv;
  if (a.nyquist) {
    k.p = a.adjoint ? x->nv : a.wide ? x->su : x->sv;
    k.sgn = a.adjoint ? -1.0 : 1.0;
    // the term's n: none for even MW columns, one or two samples for odd ones
    k.vmode[0] = x->mw ? 0 : 2;
    k.vmode[1] = a.adjoint ? 2 : 1;
  }
  // Through LDS from 4096 waves of 4 x 2 tiles on (MW L = 512, 64 maps 1550 us against
  // 1690 with 2 x 2 tiles from registers, MWSS L = 512, spin 2, 16 maps 564 against 698,
  // MW 512 / 8, 4608 waves, 246 against 257; with fewer it starves: MW 512 / 3 124
  // against 112, MW 256 / 4 45 against 23); 2 x 2 tiles from 1536 waves on (2 parities
  // x 32 rows x 32 columns x maps), below that single tiles: at L = 193, 3 maps 23 us
  // with 1950 single-tile waves.
  const auto waves = [&](int mt, int nt) {
    return (int64_t)batch * 2 * ((k.R + 16 * mt - 1) / (16 * mt)) *
           ((k.ncol + 16 * nt - 1) / (16 * nt));
  };
  if (waves(4, 2) >= 4096) return mix_launch_lds(k, batch, s);
  if (waves(2, 2) >= 1536) return mix_launch<2, 2, 4>(k, batch, s);
  return mix_launch<1, 1, 8>(k, batch, s);
}

}  // namespace s2h
