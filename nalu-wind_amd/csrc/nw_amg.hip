// nw_amg.hip -- smoothed-aggregation AMG preconditioner on gfx950: the
// hierarchy built on the host (host/nw_amg_setup.cpp) is uploaded once and
// applied as a V-cycle with Chebyshev smoothing (degree 2, eigenvalue ratio
// 20 on D^-1 A, zero initial guess), restriction R = P^T and prolongation P
// as SpMVs, and a dense inverse on the coarsest level.  The V-cycle is a
// fixed linear operator, so it serves as a right preconditioner for GMRES.
// It runs in the solver's storage type: double for the FP64 method, float
// for the FP32-inner method (the FP32 copy is narrowed from the FP64 one on
// the device and shares its structure arrays).
//
// Every level works on its operator with the columns scaled to a unit
// diagonal, B = A D^-1, and on the iterate x^ = D x: then A x = B x^, the
// residual and the restriction are as they were, the smoother's D^-1 is gone
// (d^ = c1 d^ + c2 (b - B z^)), the prolongators become D P D_c^-1, and the
// V-cycle returns D M^-1 b, which A M^-1 b = B (D M^-1 b) and the solver's
// update x += D^-1 x^ take as it is.  Degree 2 from zero is then
//   x^ = alpha v - beta B v,  alpha = (1 + c1)/theta + c2, beta = c2/theta,
// one pass that reads the matrix and v and writes x^, where the starting
// term, d and z were vectors of their own (fine level, FP64: 5 vectors of
// traffic per smoothing beside the matrix instead of 10 before the coarse
// correction, 6 instead of 13 after it).
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <vector>

#include "nw_amg.h"
#include "nw_sparse.h"

namespace nw {

namespace {

// y = M x, the coarsest level's dense inverse: one wave per row, FP64 sums
// (a lane per row walked its row alone, each load 64 rows apart: 100 us for
// 265 rows).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_dense_mv(const T* __restrict__ M, int n,
                                                    const T* __restrict__ x, T* __restrict__ y)
{
  const int i = (int)((blockIdx.x * kBlock + threadIdx.x) / kWave);
  if (i >= n) return;
  const int lane = threadIdx.x & (kWave - 1);
  double s = 0.0;
#pragma unroll 4
  for (int j = lane; j < n; j += kWave) s += (double)M[(int64_t)i * n + j] * (double)x[j];
  for (int o = kWave / 2; o > 0; o >>= 1) s += __shfl_xor(s, o);
  if (lane == 0) y[i] = (T)s;
}

// Scales a stored matrix by rows and columns in place: v[p] *= row(r) / col(c)
// factors, rinv and cinv holding the inverses 1 / row and 1 / col of the
// diagonals (0: an empty row, scaled to 0); either may be null.  A lane per
// row in sliced ELL form (sp) or CSR (rp).
__global__ __launch_bounds__(kBlock) void k_scale_mat(
  const int64_t* __restrict__ sp, const int32_t* __restrict__ rp, const int32_t* __restrict__ ci,
  double* __restrict__ v, int n, const double* __restrict__ rinv,
  const double* __restrict__ cinv)
{
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  double f = 1.0;
  if (rinv) f = rinv[r] != 0.0 ? 1.0 / rinv[r] : 0.0;
  int64_t p, end, step;
  if (sp) {
    p = sp[r >> 6] + (r & 63);
    end = sp[(r >> 6) + 1];
    step = 64;
  } else {
    p = rp[r];
    end = rp[r + 1];
    step = 1;
  }
  for (; p < end; p += step) v[p] *= cinv ? f * cinv[ci[p]] : f;
}

}  // namespace

// A level operator, in sliced ELL form (sp != nullptr: the layout of Sell,
// G = 1 or 2 lanes per row) when its rows are short, else in CSR with G lanes per
// row (rp).  The fine-level A uses the graph's sliced ELL structure; the
// others own theirs.
template <typename T>
struct DevMat {
  int n = 0;  // rows
  int G = 1;  // lanes per row
  const int64_t* sp = nullptr;
  const int32_t* rp = nullptr;
  const int32_t* ci = nullptr;
  const int32_t* dia_w = nullptr;  // offset and delta forms of the fine
  const int32_t* dia_off = nullptr;  // level's slices
  const int32_t* base = nullptr;
  const uint16_t* cd = nullptr;
  bool stretch = false;
  const T* v = nullptr;
  int64_t nv = 0;  // stored values (padding included)
  SellView view() const { return {sp, ci, dia_w, dia_off, base, cd, stretch}; }
  T* own_v = nullptr;  // v, but for the fine level (the solver's copy)
  Sell own;            // sliced ELL structure
  int32_t* own_rp = nullptr;
  int32_t* own_ci = nullptr;
};

// Rows up to this many entries on average are applied in sliced ELL form
// (measured at 256^3: the 7-entry fine matrix and the prolongators gain
// 1.5-1.9x over CSR, and the 20-24-entry operators of levels 1-2 cut the
// whole solve by 5-10 %; the 36-200-entry coarser operators lose).
constexpr double kSellMaxAvgRow = 25.0;
// ... if there are this many rows: with fewer, a lane's walk over its row's
// entries, eight at a time, is what bounds it (restrictions to 43.5 and 10.9
// thousand rows of 15 and 13 entries, FP64: 21.3 and 18.1 us with two lanes;
// in CSR 14.8 and 13.4 with 4 lanes, 9.2 and 8.2 with 8, 10.7 and 5.2 with
// 16).  The line by whole iterations of graded boxes, FP64, level 1 (rows of
// 20 entries, its restriction and the level's own matrix) in sliced ELL / in
// CSR: 48 thousand rows 172 / 167 us, 59 182 / 179, 67 187.5 / 186, 77 191 /
// 194.5, 90 204 / 209, 114 231 / 240, 132 248 / 262, 161 279 / 295, 189 306 /
// 328; FP32 from equal at 77 to 215 / 232 at 161.
constexpr int64_t kSellMinRows = 70000;
// ... and, with fewer rows than hide it, no row of more than this many
// entries, the walk of two lanes over which the launch ends with (the
// restriction to 189 thousand rows of 15, the longest of 219, FP32: 23.4 us,
// in CSR 21.1; restrictions to level 1 have 39 to 54 at most)
constexpr int64_t kSellMaxRow = 128, kSellLongRows = 200000;

template <typename T>
static void mat_spmv(const DevMat<T>& M, const T* x, T* y, T alpha,
                     hipStream_t st)
{
  if (M.sp)
    NW_SELL_LAUNCH(k_sell_spmv, T, M.G, M.n, st, M.view(), M.v, x, y, M.n, alpha);
  else
    NW_ROW_LAUNCH(k_spmv, T, M.G, M.n, st, M.rp, M.ci, M.v, x, y, M.n, alpha);
}

template <typename T>
static void mat_spmv_add(const DevMat<T>& M, const T* x, T* y, hipStream_t st)
{
  if (M.sp)
    NW_SELL_LAUNCH(k_sell_spmv_add, T, M.G, M.n, st, M.view(), M.v, x, y, M.n);
  else
    NW_ROW_LAUNCH(k_spmv_add, T, M.G, M.n, st, M.rp, M.ci, M.v, x, y, M.n);
}

template <typename T>
static void mat_resid(const DevMat<T>& M, const T* x, const T* b, T* r,
                      hipStream_t st)
{
  if (M.sp)
    NW_SELL_LAUNCH(k_sell_resid, T, M.G, M.n, st, M.view(), M.v, x, b, r, M.n);
  else
    NW_ROW_LAUNCH(k_resid, T, M.G, M.n, st, M.rp, M.ci, M.v, x, b, r, M.n);
}

// out = alpha v - beta A v, with add added to out
template <typename T>
static void mat_smooth(const DevMat<T>& M, const T* v, T* out, T alpha, T beta, bool add,
                       hipStream_t st)
{
  if (M.sp && add)
    NW_SELL_LAUNCH_ADD(k_sell_smooth, T, M.G, M.n, st, M.view(), M.v, v, out, M.n, alpha, beta);
  else if (M.sp)
    NW_SELL_LAUNCH(k_sell_smooth, T, M.G, M.n, st, M.view(), M.v, v, out, M.n, alpha, beta);
  else if (add)
    NW_ROW_LAUNCH_ADD(k_smooth, T, M.G, M.n, st, M.rp, M.ci, M.v, v, out, M.n, alpha, beta);
  else
    NW_ROW_LAUNCH(k_smooth, T, M.G, M.n, st, M.rp, M.ci, M.v, v, out, M.n, alpha, beta);
}

template <typename T>
struct DevLevel {
  DevMat<T> A, P, R;
  double* dinv = nullptr;  // FP64 hierarchy only
  T *x = nullptr, *b = nullptr, *r = nullptr;
  double lmax = 0;
  int n = 0;
};

template <typename T>
struct DevHier {
  std::vector<DevLevel<T>> lv;
  T* cinv = nullptr;
  int nc = 0;
  bool ready = false;
};

struct AmgDevice {
  DevHier<double> d;
  DevHier<float> f;  // made from d on the device when first asked for
  std::vector<int64_t> rows, nnz;  // per level
  int nlev = 0;
  double setup_seconds = 0;
  double cheb_ratio = 20.0;
};

template <typename T>
static void free_mat(DevMat<T>& m)
{
  sell_free(m.own);
  (void)hipFree(m.own_rp);
  (void)hipFree(m.own_ci);
  (void)hipFree(m.own_v);
  m = DevMat<T>();
}

template <typename T>
static void free_hier(DevHier<T>& h)
{
  for (auto& L : h.lv) {
    free_mat(L.A);
    free_mat(L.P);
    free_mat(L.R);
    (void)hipFree(L.dinv);
    for (T* p : {L.x, L.b, L.r}) (void)hipFree(p);
  }
  h.lv.clear();
  (void)hipFree(h.cinv);
  h.cinv = nullptr;
  h.ready = false;
}

void amg_free(AmgDevice* a)
{
  if (!a) return;
  free_hier(a->f);  // shares structure arrays with d
  free_hier(a->d);
  delete a;
}

namespace {

// device buffers released when the scope ends
struct DevScratch {
  std::vector<void*> p;
  template <typename T>
  int alloc(T** q, int64_t n)
  {
    *q = nullptr;
    if (hipMalloc(q, sizeof(T) * std::max<int64_t>(n, 1)) != hipSuccess) return NW_E_ALLOC;
    p.push_back(*q);
    return NW_OK;
  }
  ~DevScratch()
  {
    for (void* q : p) (void)hipFree(q);
  }
};

template <typename T>
__global__ void k_narrow(const double* __restrict__ in, T* __restrict__ out, int64_t n)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = (T)in[i];
}

// The power iteration's start vector: x_i = 0.5 + u_i, u_i in [0, 1) a
// splitmix64 hash of i (independent of the launch)
__global__ void k_pow_start(double* __restrict__ x, int n)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint64_t z = (uint64_t)i + 0x9e3779b97f4a7c15ULL;
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
  z ^= z >> 31;
  x[i] = 0.5 + (double)(z >> 11) * (1.0 / 9007199254740992.0);
}

__global__ void k_pow_div(double* __restrict__ x, double d, int n)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] /= d;
}

// y = D^-1 y (y holding A x) and, per block in a fixed tree order, the
// partial sums of x.y and y.y; with dinv == nullptr only y.y of y as it is
__global__ __launch_bounds__(kBlock) void k_pow_scale(double* __restrict__ y,
                                                     const double* __restrict__ dinv,
                                                     const double* __restrict__ x, int n,
                                                     double* __restrict__ part)
{
  __shared__ double sxy[kBlock], syy[kBlock];
  const int t = threadIdx.x, i = blockIdx.x * kBlock + t;
  double a = 0.0, b = 0.0;
  if (i < n) {
    double v = y[i];
    if (dinv) {
      v *= dinv[i];
      y[i] = v;
      a = x[i] * v;
    }
    b = v * v;
  }
  sxy[t] = a;
  syy[t] = b;
  __syncthreads();
  for (int o = kBlock / 2; o > 0; o >>= 1) {
    if (t < o) {
      sxy[t] += sxy[t + o];
      syy[t] += syy[t + o];
    }
    __syncthreads();
  }
  if (t == 0) {
    part[2 * blockIdx.x] = sxy[0];
    part[2 * blockIdx.x + 1] = syy[0];
  }
}

// The fine level's filtered operator F of the smoothed-aggregation setup
// (host/nw_amg_setup.cpp, coarsen): entry (i, j != i) is kept when
// a_ij^2 > theta^2 |a_ii a_jj| and neither row is a Dirichlet row (no
// nonzero off-diagonal); the others are lumped into the diagonal.  Per
// row: a_ii and the Dirichlet flag.
__global__ void k_filter_diag(const int32_t* __restrict__ rp, const int32_t* __restrict__ ci,
                              const double* __restrict__ a, int n, double* __restrict__ d,
                              int8_t* __restrict__ dir)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double di = 0.0;
  int8_t only_diag = 1;
  for (int k = rp[i]; k < rp[i + 1]; ++k) {
    if (ci[k] == i)
      di = a[k];
    else if (a[k] != 0.0)
      only_diag = 0;
  }
  d[i] = di;
  dir[i] = only_diag;
}

__device__ inline bool filter_keep(int i, int j, double aij, const double* d,
                                   const int8_t* dir, double th2)
{
  return j == i || (!dir[i] && !dir[j] && aij * aij > th2 * fabs(d[i] * d[j]));
}

// F's diagonal a_ii + (sum of the row's dropped entries, in row order) and
// its inverse (0 for a zero diagonal)
__global__ void k_filter_lump(const int32_t* __restrict__ rp, const int32_t* __restrict__ ci,
                              const double* __restrict__ a, int n, const double* __restrict__ d,
                              const int8_t* __restrict__ dir, double th2,
                              double* __restrict__ fd, double* __restrict__ fdinv)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double lump = 0.0;
  for (int k = rp[i]; k < rp[i + 1]; ++k)
    if (!filter_keep(i, ci[k], a[k], d, dir, th2)) lump += a[k];
  const double f = d[i] + lump;
  fd[i] = f;
  fdinv[i] = f != 0.0 ? 1.0 / f : 0.0;
}

// y = F x over the kept entries in row order (the diagonal as F's)
__global__ void k_filter_spmv(const int32_t* __restrict__ rp, const int32_t* __restrict__ ci,
                              const double* __restrict__ a, int n, const double* __restrict__ d,
                              const int8_t* __restrict__ dir, double th2,
                              const double* __restrict__ fd, const double* __restrict__ x,
                              double* __restrict__ y)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double s = 0.0;
  for (int k = rp[i]; k < rp[i + 1]; ++k) {
    const int j = ci[k];
    if (j == i)
      s += fd[i] * x[j];
    else if (filter_keep(i, j, a[k], d, dir, th2))
      s += a[k] * x[j];
  }
  y[i] = s;
}

}  // namespace

// lambda_max(D^-1 A) by `iters` power-iteration steps from a fixed start
// vector (the hashed one, or the host array `start`; spmv(x, y) forms
// y = A x; dinv = 1 / diag): each step normalises
// x, forms y = D^-1 A x and the Rayleigh quotient x.y with the next norm
// y.y; block partial sums are added on the host in block order, so the
// estimate is reproducible.  x and y are n-vectors of work space.
template <typename M>
static int device_lmax(int n, double* x, double* y, const double* dinv, const M& spmv,
                       int iters, hipStream_t st, double* out,
                       const double* start = nullptr)
{
  const unsigned nb = grid_for(n, kBlock);
  DevScratch tmp;
  double* part = nullptr;
  NW_REQUIRE(tmp.alloc(&part, 2 * (int64_t)nb) == NW_OK, NW_E_ALLOC,
             "AMG eigenvalue estimate: device allocation failed");
  std::vector<double> hp(2 * (size_t)nb);
  auto sums = [&](double& xy, double& yy) -> int {
    NW_HIP(hipMemcpyAsync(hp.data(), part, sizeof(double) * hp.size(),
                          hipMemcpyDeviceToHost, st));
    NW_HIP(hipStreamSynchronize(st));
    xy = yy = 0.0;
    for (unsigned b = 0; b < nb; ++b) {
      xy += hp[2 * b];
      yy += hp[2 * b + 1];
    }
    return NW_OK;
  };
  if (start)
    NW_HIP(hipMemcpyAsync(x, start, sizeof(double) * n, hipMemcpyHostToDevice, st));
  else
    k_pow_start<<<nb, kBlock, 0, st>>>(x, n);
  k_pow_scale<<<nb, kBlock, 0, st>>>(x, nullptr, nullptr, n, part);
  NW_LAUNCH_CHECK();
  double lam = 1.0, nx2 = 0.0, unused = 0.0;
  int rc = sums(unused, nx2);
  if (rc) return rc;
  for (int it = 0; it < iters; ++it) {
    const double nx = std::sqrt(nx2);
    if (!(nx > 0)) break;
    k_pow_div<<<nb, kBlock, 0, st>>>(x, nx, n);
    spmv(x, y);
    k_pow_scale<<<nb, kBlock, 0, st>>>(y, dinv, x, n, part);
    NW_LAUNCH_CHECK();
    rc = sums(lam, nx2);
    if (rc) return rc;
    std::swap(x, y);
  }
  *out = lam;
  return NW_OK;
}

// Uploads a host CSR matrix.  Rows of more than kSellMaxAvgRow entries on
// average, fewer rows than kSellMinRows, or few with long ones among them
// stay in CSR: G lanes per row, that take its average length at once, or four
// times that if the rows are ragged (P and R: the longest has ten times the
// average; a level's own matrix is slower with more lanes, 8.0 -> 10.3 us at
// twice as many for 43.5 thousand rows of 28).  Others are packed into sliced ELL on the device from the
// uploaded CSR, with padding positions repeating the row's last column (value
// 0), so that they stay inside the columns of a rectangular P or R.
static int upload_mat(const amg::Csr& h, DevMat<double>& d, bool ragged, hipStream_t st)
{
  NW_REQUIRE(h.nrows >= 1 && h.nrows < INT32_MAX && h.ncols >= 1 && h.nnz() < INT32_MAX,
             NW_E_ARG, "AMG level too large or empty");
  const int64_t n = h.nrows, nnz = h.nnz();
  const double avg = (double)nnz / (double)n;
  const std::vector<int32_t> rp(h.rp.begin(), h.rp.end());
  d.n = (int)n;
  bool long_rows = false;
  if (n < kSellLongRows)
    for (int64_t i = 0; i < n; ++i) long_rows |= rp[i + 1] - rp[i] > kSellMaxRow;
  if (avg > kSellMaxAvgRow || n < kSellMinRows || long_rows) {
    d.G = lanes_per_row(ragged ? 4.0 * avg : avg);
    d.nv = nnz;
    NW_HIP(hipMalloc(&d.own_rp, sizeof(int32_t) * rp.size()));
    NW_HIP(hipMalloc(&d.own_ci, sizeof(int32_t) * std::max<int64_t>(nnz, 1)));
    NW_HIP(hipMalloc(&d.own_v, sizeof(double) * std::max<int64_t>(nnz, 1)));
    d.rp = d.own_rp;
    d.ci = d.own_ci;
    d.v = d.own_v;
    NW_HIP(hipMemcpyAsync(d.own_rp, rp.data(), sizeof(int32_t) * rp.size(),
                          hipMemcpyHostToDevice, st));
    NW_HIP(hipMemcpyAsync(d.own_ci, h.ci.data(), sizeof(int32_t) * nnz,
                          hipMemcpyHostToDevice, st));
    NW_HIP(hipMemcpyAsync(d.own_v, h.v.data(), sizeof(double) * nnz, hipMemcpyHostToDevice, st));
    NW_HIP(hipStreamSynchronize(st));
    return NW_OK;
  }
  DevScratch tmp;
  int32_t *drp = nullptr, *dci = nullptr;
  double* dv = nullptr;
  int rc = tmp.alloc(&drp, n + 1);
  if (!rc) rc = tmp.alloc(&dci, nnz);
  if (!rc) rc = tmp.alloc(&dv, nnz);
  NW_REQUIRE(rc == NW_OK, NW_E_ALLOC, "AMG level upload: device allocation failed");
  NW_HIP(hipMemcpyAsync(drp, rp.data(), sizeof(int32_t) * (n + 1), hipMemcpyHostToDevice, st));
  NW_HIP(hipMemcpyAsync(dci, h.ci.data(), sizeof(int32_t) * nnz, hipMemcpyHostToDevice, st));
  NW_HIP(hipMemcpyAsync(dv, h.v.data(), sizeof(double) * nnz, hipMemcpyHostToDevice, st));
  Sell& s = d.own;  // owned by d, also after a failure
  rc = sell_build(drp, dci, (int)n, s, st, true);
  if (rc) return rc;
  d.G = sell_lanes(n, avg);
  d.sp = s.sp;
  d.ci = s.ci;
  d.base = s.base;
  d.cd = s.cd;
  d.nv = s.len;
  NW_HIP(hipMalloc(&d.own_v, sizeof(double) * std::max<int64_t>(s.len, 1)));
  d.v = d.own_v;
  if (s.len > 0) {
    k_sell_values<double><<<grid_for(s.len, kBlock), kBlock, 0, st>>>(s.slot, s.ci, dv,
                                                                      nullptr, d.own_v, s.len);
    NW_LAUNCH_CHECK();
  }
  NW_HIP(hipStreamSynchronize(st));
  (void)hipFree(s.slot);  // the values are in place
  s.slot = nullptr;
  return NW_OK;
}

// The FP32 copy of an FP64 level matrix: the same structure arrays (not
// owned), values narrowed on the device.
static int narrow_mat(const DevMat<double>& s, DevMat<float>& d, hipStream_t st)
{
  d.n = s.n;
  d.G = s.G;
  d.sp = s.sp;
  d.rp = s.rp;
  d.ci = s.ci;
  d.base = s.base;
  d.cd = s.cd;
  d.nv = s.nv;
  NW_HIP(hipMalloc(&d.own_v, sizeof(float) * std::max<int64_t>(s.nv, 1)));
  d.v = d.own_v;
  if (s.nv > 0) {
    k_narrow<float><<<grid_for(s.nv, kBlock), kBlock, 0, st>>>(s.v, d.own_v, s.nv);
    NW_LAUNCH_CHECK();
  }
  return NW_OK;
}

template <typename T>
static int alloc_level_vectors(DevLevel<T>& L)
{
  for (T** p : {&L.x, &L.b, &L.r})
    NW_HIP(hipMalloc(p, sizeof(T) * std::max(L.n, 1)));
  return NW_OK;
}

// The FP64 hierarchy on the device from the host one.
static int upload_hier(Ctx* c, const amg::Hierarchy& h, DevHier<double>& H)
{
  hipStream_t st = c->stream;
  const int nl = (int)h.levels.size();
  H.lv.resize(nl);
  for (int l = 0; l < nl; ++l) {
    const amg::Level& hl = h.levels[l];
    DevLevel<double>& L = H.lv[l];
    L.n = (int)hl.A.nrows;
    L.lmax = hl.lmax;
    if (l == 0) {
      // the fine operator is the linear system's own matrix, in the
      // graph's sliced ELL order (the solver's copy, made at every solve)
      NW_REQUIRE(c->g.sell.ci && L.n == c->g.nnode, NW_E_STATE,
                 "sliced ELL form not built");
      L.A.n = L.n;
      L.A.sp = c->g.sell.sp;
      L.A.ci = c->g.sell.ci;
      L.A.stretch = sell_view(c->g.sell).stretch;
      L.A.dia_w = c->g.sell.dia_w;
      L.A.dia_off = c->g.sell.dia_off;
      L.A.base = c->g.sell.base;
      L.A.cd = c->g.sell.cd;
      L.A.nv = c->g.sell.len;
    } else {
      int rc = upload_mat(hl.A, L.A, false, st);
      if (rc) return rc;
    }
    NW_HIP(hipMalloc(&L.dinv, sizeof(double) * std::max(L.n, 1)));
    NW_HIP(hipMemcpyAsync(L.dinv, hl.dinv.data(), sizeof(double) * L.n,
                          hipMemcpyHostToDevice, st));
    int rc = alloc_level_vectors(L);
    if (!rc && l + 1 < nl) rc = upload_mat(hl.P, L.P, true, st);
    if (!rc && l + 1 < nl) rc = upload_mat(hl.R, L.R, true, st);
    if (rc) return rc;
  }
  H.nc = (int)h.levels.back().A.nrows;
  std::vector<double> cinv(h.coarse_inv.begin(), h.coarse_inv.end());
  if (nl == 1)  // solved directly: D A^-1, as the V-cycle returns
    for (int64_t i = 0; i < H.nc; ++i) {
      const double di = h.levels[0].dinv[i];
      for (int64_t j = 0; j < H.nc; ++j) cinv[i * H.nc + j] *= di != 0.0 ? 1.0 / di : 0.0;
    }
  NW_HIP(hipMalloc(&H.cinv, sizeof(double) * std::max<size_t>(cinv.size(), 1)));
  NW_HIP(hipMemcpyAsync(H.cinv, cinv.data(), sizeof(double) * cinv.size(),
                        hipMemcpyHostToDevice, st));
  NW_HIP(hipStreamSynchronize(st));
  H.ready = true;
  return NW_OK;
}

// The FP32 hierarchy from the FP64 one, on the device.
static int narrow_hier(Ctx* c, const DevHier<double>& D, DevHier<float>& H)
{
  hipStream_t st = c->stream;
  const int nl = (int)D.lv.size();
  H.lv.resize(nl);
  for (int l = 0; l < nl; ++l) {
    const DevLevel<double>& S = D.lv[l];
    DevLevel<float>& L = H.lv[l];
    L.n = S.n;
    L.lmax = S.lmax;
    if (l == 0) {
      L.A = DevMat<float>();
      L.A.n = S.A.n;
      L.A.sp = S.A.sp;
      L.A.ci = S.A.ci;
      L.A.stretch = S.A.stretch;
      L.A.dia_w = S.A.dia_w;
      L.A.dia_off = S.A.dia_off;
      L.A.base = S.A.base;
      L.A.cd = S.A.cd;
      L.A.nv = S.A.nv;
    } else {
      int rc = narrow_mat(S.A, L.A, st);
      if (rc) return rc;
    }
    int rc = alloc_level_vectors(L);
    if (!rc && l + 1 < nl) rc = narrow_mat(S.P, L.P, st);
    if (!rc && l + 1 < nl) rc = narrow_mat(S.R, L.R, st);
    if (rc) return rc;
  }
  H.nc = D.nc;
  const int64_t nci = (int64_t)D.nc * D.nc;
  NW_HIP(hipMalloc(&H.cinv, sizeof(float) * std::max<int64_t>(nci, 1)));
  if (nci > 0) {
    k_narrow<float><<<grid_for(nci, kBlock), kBlock, 0, st>>>(D.cinv, H.cinv, nci);
    NW_LAUNCH_CHECK();
  }
  NW_HIP(hipStreamSynchronize(st));
  H.ready = true;
  return NW_OK;
}

int amg_setup(Ctx* c, AmgDevice** out)
{
  const auto t0 = std::chrono::steady_clock::now();
  Graph& g = c->g;
  NW_REQUIRE(g.ndof == 1, NW_E_STATE, "AMG needs a 1-dof system");
  amg::Csr A = amg::csr_with_structure(g.nnode, g.h_row_ptr.data(), g.h_cols.data());
  NW_HIP(hipMemcpyAsync(A.v.data(), g.vals, sizeof(double) * g.nnzb,
                        hipMemcpyDeviceToHost, c->stream));
  NW_HIP(hipStreamSynchronize(c->stream));
  amg::Options o;
  o.smoother_lmax = false;  // estimated on the device after the upload
  {
    // the fine prolongator's damping estimate, lambda_max(D_F^-1 F), on
    // the device from the matrix there
    const int n = (int)g.nnode;
    const unsigned nb = grid_for(n, kBlock);
    DevScratch tmp;
    double *d = nullptr, *fd = nullptr, *fdinv = nullptr, *x = nullptr, *y = nullptr;
    int8_t* dir = nullptr;
    int arc = tmp.alloc(&d, n);
    if (!arc) arc = tmp.alloc(&fd, n);
    if (!arc) arc = tmp.alloc(&fdinv, n);
    if (!arc) arc = tmp.alloc(&x, n);
    if (!arc) arc = tmp.alloc(&y, n);
    if (!arc) arc = tmp.alloc(&dir, n);
    NW_REQUIRE(arc == NW_OK, NW_E_ALLOC, "AMG setup: device allocation failed");
    const double th2 = o.drop_tol * o.drop_tol;
    k_filter_diag<<<nb, kBlock, 0, c->stream>>>(g.row_ptr, g.cols, g.vals, n, d, dir);
    k_filter_lump<<<nb, kBlock, 0, c->stream>>>(g.row_ptr, g.cols, g.vals, n, d, dir, th2, fd,
                                                fdinv);
    NW_LAUNCH_CHECK();
    double lf = 0.0;
    // from the host setup's start vector, so that the estimate is the one
    // the host would make, up to the order of the dot-product sums
    const std::vector<double> x0 = amg::power_start(n);
    const int prc = device_lmax(n, x, y, fdinv, [&](const double* xv, double* yv) {
      k_filter_spmv<<<nb, kBlock, 0, c->stream>>>(g.row_ptr, g.cols, g.vals, n, d, dir, th2, fd,
                                                  xv, yv);
    }, o.power_iters, c->stream, &lf, x0.data());
    if (prc) return prc;
    o.filtered_lmax0 = lf;
  }
  amg::Hierarchy h;
  const int rc = amg::build(std::move(A), o, h);
  NW_REQUIRE(rc == 0, NW_E_ARG, "AMG setup failed (%d): coarse level too "
             "large or singular", rc);
  NW_REQUIRE(o.cheb_degree == 2, NW_E_ARG, "the V-cycle smooths with two Chebyshev terms");
  AmgDevice* a = new AmgDevice();
  a->cheb_ratio = o.cheb_ratio;
  a->nlev = (int)h.levels.size();
  for (const auto& L : h.levels) {
    a->rows.push_back(L.A.nrows);
    a->nnz.push_back(L.A.nnz());
  }
  int urc = upload_hier(c, h, a->d);
  // the smoothers' lambda_max(D^-1 A) on the device, every level but the
  // coarsest (solved directly), then the column scaling of the operators and
  // prolongators (the coarsest level's iterate is x itself)
  const int last = a->nlev - 1;
  for (int l = 0; !urc && l < last; ++l) {
    DevLevel<double>& L = a->d.lv[l];
    DevScratch tmp;
    double* y = nullptr;
    urc = tmp.alloc(&y, L.n);
    if (l == 0 && !urc) {
      const Sell& sl = g.sell;
      double* v = nullptr;
      urc = tmp.alloc(&v, sl.len);
      if (!urc) {
        k_sell_values<double><<<grid_for(sl.len, kBlock), kBlock, 0, c->stream>>>(
          sl.slot, sl.ci, g.vals, nullptr, v, sl.len);
        L.A.v = v;
      }
    }
    if (urc) {
      set_error("AMG setup: device allocation failed");
      break;
    }
    urc = device_lmax(L.n, L.x, y, L.dinv, [&](const double* x, double* yv) {
      mat_spmv<double>(L.A, x, yv, 1.0, c->stream);
    }, o.power_iters, c->stream, &L.lmax);
    if (l == 0) L.A.v = nullptr;
  }
  for (int l = 0; !urc && l < last; ++l) {
    DevLevel<double>& L = a->d.lv[l];
    if (l > 0)
      k_scale_mat<<<grid_for(L.n, kBlock), kBlock, 0, c->stream>>>(
        L.A.sp, L.A.rp, L.A.ci, L.A.own_v, L.n, nullptr, L.dinv);
    k_scale_mat<<<grid_for(L.n, kBlock), kBlock, 0, c->stream>>>(
      L.P.sp, L.P.rp, L.P.ci, L.P.own_v, L.n, L.dinv,
      l + 1 < last ? a->d.lv[l + 1].dinv : nullptr);
    if (hipGetLastError() != hipSuccess) {
      set_error("AMG setup: scaling kernel failed");
      urc = NW_E_HIP;
    }
  }
  if (!urc && hipStreamSynchronize(c->stream) != hipSuccess) {
    set_error("AMG setup: device error");
    urc = NW_E_HIP;
  }
  if (urc) {
    amg_free(a);
    return urc;
  }
  a->setup_seconds =
    std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  *out = a;
  return NW_OK;
}

int amg_levels(const AmgDevice* a) { return a ? a->nlev : 0; }
double amg_setup_seconds(const AmgDevice* a) { return a ? a->setup_seconds : 0; }
int amg_level_info(const AmgDevice* a, int l, int64_t* rows, int64_t* nnz)
{
  if (!a || l < 0 || l >= a->nlev) return NW_E_ARG;
  *rows = a->rows[l];
  *nnz = a->nnz[l];
  return NW_OK;
}

template <typename T>
static DevHier<T>& hier(AmgDevice* a);
template <>
DevHier<double>& hier<double>(AmgDevice* a)
{
  return a->d;
}
template <>
DevHier<float>& hier<float>(AmgDevice* a)
{
  return a->f;
}

const double* amg_fine_dinv(const AmgDevice* a) { return a->d.lv[0].dinv; }

template <typename T>
int amg_prepare(Ctx* c, AmgDevice* a, const T* fine, double* seconds)
{
  DevHier<T>& H = hier<T>(a);
  NW_REQUIRE(a->d.ready, NW_E_STATE, "AMG hierarchy not set up");
  if (seconds) *seconds = 0.0;
  if (!H.ready) {
    if constexpr (sizeof(T) == 4) {
      const auto t0 = std::chrono::steady_clock::now();
      int rc = narrow_hier(c, a->d, a->f);
      if (rc) return rc;
      if (seconds)
        *seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    }
  }
  const Sell& sl = c->g.sell;
  NW_REQUIRE(sl.ci && H.lv[0].A.ci == sl.ci, NW_E_STATE,
             "AMG fine level needs the graph's sliced ELL form");
  H.lv[0].A.v = fine;
  return NW_OK;
}

// Two Chebyshev terms on [1.1 lmax / ratio, 1.1 lmax] from zero (Saad, Alg.
// 12.1): z0 = v / theta, then d = c1 z0 + c2 (v - B z0) added to it.
struct Smoother {
  double alpha, beta;
};
static Smoother smoother(const AmgDevice* a, double lmax_est)
{
  const double lmax = 1.1 * lmax_est, lmin = lmax / a->cheb_ratio;
  const double theta = 0.5 * (lmax + lmin), delta = 0.5 * (lmax - lmin);
  const double sigma = theta / delta, rho = 1.0 / sigma;
  const double rho_new = 1.0 / (2.0 * sigma - rho);
  const double c1 = rho_new * rho, c2 = 2.0 * rho_new / delta;
  return {(1.0 + c1) / theta + c2, c2 / theta};
}

template <typename T>
static int vcycle(AmgDevice* a, DevHier<T>& H, int l, const T* b, T* x,
                  hipStream_t st)
{
  DevLevel<T>& L = H.lv[l];
  const int last = (int)H.lv.size() - 1;
  if (l == last) {
    k_dense_mv<T><<<grid_for((int64_t)H.nc * kWave, kBlock), kBlock, 0, st>>>(H.cinv, H.nc, b, x);
    NW_LAUNCH_CHECK();
    return NW_OK;
  }
  DevLevel<T>& C = H.lv[l + 1];
  const Smoother s = smoother(a, L.lmax);
  mat_smooth<T>(L.A, b, x, (T)s.alpha, (T)s.beta, false, st);  // pre-smooth from zero
  mat_resid<T>(L.A, x, b, L.r, st);
  mat_spmv<T>(L.R, L.r, C.b, (T)1, st);
  NW_LAUNCH_CHECK();
  const int rc = vcycle<T>(a, H, l + 1, C.b, C.x, st);
  if (rc) return rc;
  mat_spmv_add<T>(L.P, C.x, x, st);
  // post-smooth the correction of the new residual, added to x
  mat_resid<T>(L.A, x, b, L.r, st);
  mat_smooth<T>(L.A, L.r, x, (T)s.alpha, (T)s.beta, true, st);
  NW_LAUNCH_CHECK();
  return NW_OK;
}

template <typename T>
int amg_apply(AmgDevice* a, const T* b, T* x, hipStream_t st)
{
  return vcycle<T>(a, hier<T>(a), 0, b, x, st);
}

template int amg_prepare<double>(Ctx*, AmgDevice*, const double*, double*);
template int amg_prepare<float>(Ctx*, AmgDevice*, const float*, double*);
template int amg_apply<double>(AmgDevice*, const double*, double*, hipStream_t);
template int amg_apply<float>(AmgDevice*, const float*, float*, hipStream_t);

}  // namespace nw
