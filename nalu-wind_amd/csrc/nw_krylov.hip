// nw_krylov.hip -- pressure-Poisson Krylov solve on gfx950.
//
// Replaces TpetraLinearSystem::solve -> TpetraLinearSolver::solve (Belos
// GMRES with an Ifpack2 preconditioner, src/LinearSolver.C:209-254, settings
// src/LinearSolverConfig.C:37-140): restarted GMRES(m), right
// preconditioning, classical Gram-Schmidt with reorthogonalisation (the
// reference configures Belos' iterated CGS, "ICGS"), x0 = 0 by default,
// convergence on ||b - A x||_2 / ||b||_2 evaluated in FP64.
//
// Orthogonalisation is CGS2 with the second pass delayed by one step
// (Swirydowicz, Langou, Ananthan, Yang, Thomas, "Low synchronization
// Gram-Schmidt and GMRES algorithms", NLAA 2021): per Arnoldi step one
// fused dot pass over the basis ([Q, y]^T [y, z]) and one fused update pass
// that both finishes q_j = (y - Q s)/rho and forms the next candidate.  The
// Hessenberg column of step j-1 is corrected with the reorthogonalisation
// coefficients, so every column is final one step after it is first formed.
// The column, its Givens rotations and the update's coefficients are computed
// on the device (k_arnoldi_step); the host only learns, from a word in pinned
// memory, whether the cycle goes on.
//
// Every restart cycle begins from the FP64 residual r = b - A x and ends
// with x += M^-1 Q y in FP64, so a cycle is one iterative-refinement step.
// The cycle (SpMV, Gram-Schmidt, preconditioner) is templated on its
// storage type: double gives the plain FP64 method; float gives the
// FP32-inner / FP64-refined method over an FP32 copy of the matrix.  Dot
// products accumulate in FP64 and are reduced in a fixed order, so results
// are reproducible run to run.
//
// Preconditioners (right): Jacobi, applied by scaling the matrix columns
// once per solve (A D^-1, which the AMG V-cycle works on as well); Chebyshev of degree k on D^-1 A over
// [lmax/ratio, lmax] (Saad, Iterative Methods for Sparse Linear Systems,
// 2nd ed., Alg. 12.1), lmax from a seeded power iteration.
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <vector>

#include "nw_internal.h"
#include "nw_sparse.h"
#include "nw_amg.h"

namespace nw {

namespace {

constexpr int kMaxBasis = 64;  // kspace + 1 <= 64
constexpr int kTile = 8;       // basis vectors per dot tile
// row blocks of the fused dot kernels at most
constexpr int kRowBlocks = 2048;
constexpr int kDotVals = 2 * kTile + 3;  // per tile: Q.y, Q.z, y.y, y.z, z.z

// Row blocks of a dot over n rows (vec of them per lane and step) in ntiles
// tiles: one step per block until the blocks fill the chip (256 CUs), then
// up to kDotSteps steps, which pay for the reduction a block ends in.
inline int dot_row_blocks(int64_t n, int vec, int ntiles)
{
  constexpr int64_t kDotSteps = 4;
  const int64_t one = std::max<int64_t>(1, (n / vec + kBlock - 1) / kBlock);
  const int64_t fill = std::max(1, 1024 / ntiles);
  return (int)std::min({one, std::max(fill, one / kDotSteps), (int64_t)kRowBlocks});
}

__device__ inline double wave_sum(double v)
{
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// Sum NA per-thread accumulators over the block; thread k < NA writes
// out[k].
template <int NA>
__device__ inline void block_reduce_store(double (&acc)[NA],
                                          double* __restrict__ out)
{
  __shared__ double sh[kBlock / kWave][NA];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < NA; ++k) {
    const double s = wave_sum(acc[k]);
    if (lane == 0) sh[wv][k] = s;
  }
  __syncthreads();
  for (int k = threadIdx.x; k < NA; k += blockDim.x) {
    double s = 0.0;
    for (int w = 0; w < kBlock / kWave; ++w) s += sh[w][k];
    out[k] = s;
  }
}

// Sums of 16 values over the 64 lanes of a wave by halving: at each step a
// lane keeps the half of its values that its lane bit names and adds the
// partner's share of them, so 15 exchanges leave one value per group of four
// lanes and two more finish it (96 exchanges with a butterfly per value).
// Lane 4 k + {0..3} returns the sum of value k.
__device__ inline double wave_sum16(double (&a)[16])
{
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int h = 8; h >= 1; h >>= 1) {
    const int o = 4 * h;  // lane bit 5, 4, 3, 2
    const bool up = lane & o;
#pragma unroll
    for (int i = 0; i < h; ++i) {
      const double keep = up ? a[h + i] : a[i];
      const double send = up ? a[i] : a[h + i];
      a[i] = keep + __shfl_xor(send, o);
    }
  }
  double v = a[0];
  v += __shfl_xor(v, 2);
  v += __shfl_xor(v, 1);
  return v;
}

// out[v] = sum_b partial[v * nb + b], one workgroup per value, fixed-order
// tree (reproducible).
__global__ __launch_bounds__(kBlock) void k_reduce(
  const double* __restrict__ partial, int nb, double* __restrict__ out)
{
  const int v = blockIdx.x;
  const double* p = partial + (int64_t)v * nb;
  double s = 0.0;
  for (int b = threadIdx.x; b < nb; b += blockDim.x) s += p[b];
  double a[1] = {s};
  __shared__ double tot[1];
  block_reduce_store<1>(a, tot);
  if (threadIdx.x == 0) out[v] = tot[0];
}

// Device state of a cycle (doubles): the unrotated Hessenberg matrix H (the
// Arnoldi relation A M^-1 Q = Q H) and R, the same columns after the Givens
// rotations, both column by column; the rotations; the rotated right-hand
// side; the tentative column; the least-squares solution.
constexpr int kHsH = 0, kHsR = kHsH + kMaxBasis * kMaxBasis;
constexpr int kHsCs = kHsR + kMaxBasis * kMaxBasis, kHsSn = kHsCs + kMaxBasis;
constexpr int kHsG = kHsSn + kMaxBasis, kHsPrev = kHsG + kMaxBasis + 2;
constexpr int kHsY = kHsPrev + kMaxBasis, kHsRho = kHsY + kMaxBasis;
constexpr int kHsSize = kHsRho + 1;
// coef[0] tells the update whether to run; a, c, e, b[], d[] follow
constexpr int kCoefSize = 4 + 2 * kMaxBasis;

// Ends step j of a cycle (one workgroup): sums the nb partials of each dot
// (partial[b nv + v]), finishes Hessenberg column j - 1 and rotates it,
// decides whether the cycle goes on, and if it does forms the tentative
// column j and the coefficients of the update.  The decision goes to *status
// (pinned host memory) as token << 16 | stop << 8 | (columns done).
//
// A chain of latencies, so its loads are issued together and only the
// rotations and square roots follow each other: 3 to 9 us with the length of
// the cycle, 6.7 on average at 8,640 rows, where the same on the host (copy of
// the dots, synchronisation, copy of the coefficients) left the device idle
// for 12 us.
__global__ __launch_bounds__(kBlock) void k_arnoldi_step(
  const double* __restrict__ partial, int nb, int nv, int j, int grow, double beta,
  double stop_abs, double* __restrict__ hs, double* __restrict__ coef,
  unsigned long long* __restrict__ status, unsigned long long token)
{
  static_assert((kMaxBasis / kTile) * kDotVals <= kBlock, "a thread per dot");
  constexpr int kParts = kBlock / kWave;
  const int t = threadIdx.x, q = t & (kWave - 1), part = t / kWave;
  __shared__ double dots[kBlock], sv[kMaxBasis], tv[kMaxBasis], hc[kMaxBasis + 1],
    Hp[kParts][kMaxBasis], cs[kMaxBasis], sn[kMaxBasis], rc[kMaxBasis], sums[2];
  __shared__ bool conv;
  auto tell = [&](int stop, int kdim) {
    if (t != 0) return;
    coef[0] = stop ? 0.0 : 1.0;
    __hip_atomic_store(status, token << 16 | (unsigned long long)(stop << 8 | kdim),
                       __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  };
  const double prev = t < j ? hs[kHsPrev + t] : 0.0;
  const double rho_prev = j >= 1 ? hs[kHsRho] : 1.0;
  const double g_prev = j >= 2 ? hs[kHsG + j - 1] : beta;
  if (t < j) {
    cs[t] = hs[kHsCs + t];
    sn[t] = hs[kHsSn + t];
  }
  // the finished columns this thread multiplies by s: l = part mod kParts
  double hq[kMaxBasis / kParts];
#pragma unroll
  for (int u = 0; u < kMaxBasis / kParts; ++u) {
    const int l = part + u * kParts;
    hq[u] = l < j - 1 && q <= l + 1 ? hs[kHsH + l * kMaxBasis + q] : 0.0;
  }
  double d = 0.0;
  if (t < nv) {
#pragma unroll 8
    for (int b = 0; b < nb; ++b) d += partial[(int64_t)b * nv + t];
  }
  dots[t] = d;
  __syncthreads();
  const double yy = dots[2 * kTile], yz = dots[2 * kTile + 1];
  if (!(yy > 0) || !isfinite(yy)) {  // the column j - 1 stays unfinished
    tell(1, max(j - 1, 0));
    return;
  }
  const double sigma = 1.0 / sqrt(yy);
  if (t < kMaxBasis) {
    double a = 0.0, b = 0.0;
    if (t < j) {
      const int v = (t / kTile) * kDotVals + t % kTile;
      a = sigma * dots[v];          // s = Q^T u, u = sigma y
      b = sigma * dots[v + kTile];  // t = Q^T z
    }
    sv[t] = a;
    tv[t] = b;
    const double ss = wave_sum(a * a), st = wave_sum(a * b);
    if (t == 0) {
      sums[0] = ss;
      sums[1] = st;
    }
  }
  __syncthreads();
  const double ss = sums[0], st = sums[1];
  const double rho = ss < 1.0 ? sqrt(1.0 - ss) : 0.0;
  if (j >= 1) {
    // finish column j-1: A M^-1 q_{j-1} = Q (hprev + nu s) + nu rho q_j
    const double nu = (1.0 / sigma) / rho_prev;
    if (t <= j) {
      const double h = t < j ? prev + nu * sv[t] : nu * rho;
      hs[kHsH + (j - 1) * kMaxBasis + t] = h;
      hc[t] = h;
    }
  }
  __syncthreads();
  if (j >= 1 && t == 0) {
    const int col = j - 1;
    double a = hc[0];
#pragma unroll 8
    for (int k = 0; k < col; ++k) {
      const double b = hc[k + 1];
      rc[k] = cs[k] * a + sn[k] * b;
      a = -sn[k] * a + cs[k] * b;
    }
    const double b = hc[j];
    const double rr = sqrt(a * a + b * b);
    const double c = rr > 0 ? a / rr : 1.0, s = rr > 0 ? b / rr : 0.0;
    rc[col] = rr;
    hs[kHsCs + col] = c;
    hs[kHsSn + col] = s;
    hs[kHsG + j] = -s * g_prev;
    hs[kHsG + col] = c * g_prev;
    conv = fabs(s * g_prev) <= stop_abs;
  }
  // Hs = H[0..j][0..j-1] s, a quarter of the columns per wave
  {
    double a = 0.0;
#pragma unroll
    for (int u = 0; u < kMaxBasis / kParts; ++u) {
      const int l = part + u * kParts;
      if (l < j - 1) a += hq[u] * sv[l];
    }
    if (j >= 1 && part == (j - 1) % kParts && q <= j) a += hc[q] * sv[j - 1];
    Hp[part][q] = a;
  }
  __syncthreads();
  if (t < j) hs[kHsR + (j - 1) * kMaxBasis + t] = rc[t];
  // converged, end of the cycle or lucky breakdown
  if ((j >= 1 && conv) || !grow || !(rho > 1e-12)) {
    tell(1, j);
    return;
  }
  tell(0, j);
  // tentative column j from the dots of z = A M^-1 u, z = sigma z'
  //   V[j]   <- q_j = (sigma/rho) y - sum (s_q/rho) Q_q
  //   V[j+1] <- sigma z' - e sigma y - sum (c_q - e s_q) Q_q
  auto Hs = [&](int k) { return (Hp[0][k] + Hp[1][k]) + (Hp[2][k] + Hp[3][k]); };
  static_assert(kParts == 4, "four partial products");
  const double uz = sigma * sigma * yz, Hj = Hs(j);
  const double hjj = ((uz - st) / rho - Hj) / rho;
  const double e = (Hj + rho * hjj) / rho;
  if (t < j) {
    const double Ht = Hs(t), h = (tv[t] - Ht) / rho;
    hs[kHsPrev + t] = h;
    coef[4 + t] = sv[t] / rho;
    coef[4 + j + t] = (Ht + rho * h) - e * sv[t];
  }
  if (t == 0) {
    hs[kHsPrev + j] = hjj;
    hs[kHsRho] = rho;
    coef[1] = sigma / rho;
    coef[2] = sigma;
    coef[3] = e * sigma;
  }
}

// The least-squares solution R y = g of a cycle of kdim columns: R staged in
// LDS, then one wave, lane i holding g_i.
__global__ __launch_bounds__(kBlock) void k_arnoldi_solve(double* __restrict__ hs, int kdim)
{
  __shared__ double R[kMaxBasis * kMaxBasis];
  for (int i = threadIdx.x; i < kdim * kMaxBasis; i += kBlock)
    R[i] = (i & (kMaxBasis - 1)) <= i / kMaxBasis ? hs[kHsR + i] : 0.0;
  const int t = threadIdx.x;
  double g = t < kdim ? hs[kHsG + t] : 0.0;
  __syncthreads();
  if (t >= kWave) return;
  for (int i = kdim - 1; i >= 0; --i) {
    const double y = __shfl(g, i) / R[i * kMaxBasis + i];
    if (t < i) g -= R[i * kMaxBasis + t] * y;
    if (t == i) hs[kHsY + i] = y;
  }
}

// Fused Arnoldi dots.  Block b = rowblock * ntiles + tile (tiles of one row
// block are adjacent, so the y/z rows they share are re-read from L2).
// Tile t covers basis vectors Q_k, k in [8t, 8t+8) and k < nq; its value v
// of row block rb is value V = t kDotVals + v of partial[V sv + rb sb]: v =
// 0..7 Q_k.y, 8..15 Q_k.z, and in tile 0 16 = y.y, 17 = y.z, 18 = z.z.  z may
// be null (then its dots are zero).
//
// Bound by HBM (or the Infinity Cache) on large systems and by the block
// reduction on small ones: with 2048 row blocks at every size and a
// butterfly per value it took 23 us at least, 70 us on average at 8,640
// rows (jacobi, 31 vectors) and 64 us at 960 thousand (FP64, 16 vectors).
template <typename T>
__global__ __launch_bounds__(kBlock) void k_arnoldi_dots(
  const T* __restrict__ V, int64_t n, int nq, const T* __restrict__ y,
  const T* __restrict__ z, int ntiles, double* __restrict__ partial, int sv, int sb)
{
  static_assert(kTile == 8, "wave_sum16 reduces 2 kTile sums");
  constexpr int kVec = 16 / (int)sizeof(T);  // rows of one 16-byte load
  using Vec = T __attribute__((ext_vector_type(16 / sizeof(T)), aligned(sizeof(T))));
  const int tile = blockIdx.x % ntiles;
  const int rb = blockIdx.x / ntiles;
  const int nrb = gridDim.x / ntiles;
  const int k0 = tile * kTile;
  const int kc = min(kTile, nq - k0);
  double acc[16], ex[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int k = 0; k < 16; ++k) acc[k] = 0.0;
  const T* __restrict__ Q = V + (int64_t)k0 * n;
  auto add = [&](double yi, double zi, const double (&q)[kTile]) {
#pragma unroll
    for (int k = 0; k < kTile; ++k) {
      acc[k] += q[k] * yi;
      acc[kTile + k] += q[k] * zi;
    }
    if (tile == 0) {
      ex[0] += yi * yi;
      ex[1] += yi * zi;
      ex[2] += zi * zi;
    }
  };
  // all blocks of a tile sweep the rows together, 16 bytes of every vector
  // per lane and step (the vectors start at multiples of sizeof(T) only)
  for (int64_t i = (int64_t)rb * kBlock + threadIdx.x; i < n / kVec;
       i += (int64_t)nrb * kBlock) {
    Vec q[kTile], yv, zv;
#pragma unroll
    for (int k = 0; k < kTile; ++k)
      if (k < kc)
        q[k] = *reinterpret_cast<const Vec*>(Q + (int64_t)k * n + kVec * i);
      else
        q[k] = (T)0;
    yv = *reinterpret_cast<const Vec*>(y + kVec * i);
    if (z)
      zv = *reinterpret_cast<const Vec*>(z + kVec * i);
    else
      zv = (T)0;
#pragma unroll
    for (int u = 0; u < kVec; ++u) {
      double qu[kTile];
#pragma unroll
      for (int k = 0; k < kTile; ++k) qu[k] = (double)q[k][u];
      add((double)yv[u], (double)zv[u], qu);
    }
  }
  // the rows past the last whole vector
  const int64_t it = n / kVec * kVec + threadIdx.x;
  if (rb == 0 && it < n) {
    double qu[kTile];
#pragma unroll
    for (int k = 0; k < kTile; ++k) qu[k] = k < kc ? (double)Q[(int64_t)k * n + it] : 0.0;
    add((double)y[it], z ? (double)z[it] : 0.0, qu);
  }
  __shared__ double sh[kBlock / kWave][kDotVals];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  if (kc > 0) {
    const double s = wave_sum16(acc);
    // lane bits 5..2 chose value bits 3..0
    if ((lane & 3) == 0) sh[wv][lane >> 2] = s;
  } else if ((lane & 3) == 0) {
    sh[wv][lane >> 2] = 0.0;
  }
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const double s = tile == 0 ? wave_sum(ex[k]) : 0.0;
    if (lane == 0) sh[wv][16 + k] = s;
  }
  __syncthreads();
  for (int k = threadIdx.x; k < kDotVals; k += kBlock) {
    double s = 0.0;
    for (int w = 0; w < kBlock / kWave; ++w) s += sh[w][k];
    partial[(int64_t)(tile * kDotVals + k) * sv + (int64_t)rb * sb] = s;
  }
}

// Fused Arnoldi update: with Q_k = V[k] (k < nq), y = V[nq], z = V[nq+1]:
//   V[nq]   = a y - sum_k b_k Q_k          (the finished basis vector)
//   V[nq+1] = c z - e y - sum_k d_k Q_k    (the next candidate)
// coef = {go, a, c, e, b_0..b_{nq-1}, d_0..d_{nq-1}}; go == 0: the cycle has
// ended and nothing is done.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_arnoldi_update(
  T* __restrict__ V, int64_t n, int nq, const double* __restrict__ coef)
{
  if (coef[0] == 0.0) return;
  __shared__ double cb[kMaxBasis], cd[kMaxBasis];
  for (int k = threadIdx.x; k < nq; k += blockDim.x) {
    cb[k] = coef[4 + k];
    cd[k] = coef[4 + nq + k];
  }
  __syncthreads();
  const double a = coef[1], c = coef[2], e = coef[3];
  T* __restrict__ Y = V + (int64_t)nq * n;
  T* __restrict__ Z = Y + n;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const double yi = (double)Y[i];
    double q = a * yi;
    double w = c * (double)Z[i] - e * yi;
    int k = 0;
    for (; k + 4 <= nq; k += 4) {
      const double v0 = (double)V[(int64_t)(k + 0) * n + i];
      const double v1 = (double)V[(int64_t)(k + 1) * n + i];
      const double v2 = (double)V[(int64_t)(k + 2) * n + i];
      const double v3 = (double)V[(int64_t)(k + 3) * n + i];
      q -= cb[k] * v0 + cb[k + 1] * v1 + cb[k + 2] * v2 + cb[k + 3] * v3;
      w -= cd[k] * v0 + cd[k + 1] * v1 + cd[k + 2] * v2 + cd[k + 3] * v3;
    }
    for (; k < nq; ++k) {
      const double v0 = (double)V[(int64_t)k * n + i];
      q -= cb[k] * v0;
      w -= cd[k] * v0;
    }
    Y[i] = (T)q;
    Z[i] = (T)w;
  }
}

// u = sum_k coef[k] V[k] (k < nk), stored as T
template <typename T>
__global__ __launch_bounds__(kBlock) void k_combine(
  const T* __restrict__ V, int64_t n, int nk, const double* __restrict__ coef,
  T* __restrict__ u)
{
  __shared__ double cc[kMaxBasis];
  for (int k = threadIdx.x; k < nk; k += blockDim.x) cc[k] = coef[k];
  __syncthreads();
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    double s = 0.0;
    for (int k = 0; k < nk; ++k) s += cc[k] * (double)V[(int64_t)k * n + i];
    u[i] = (T)s;
  }
}

// x += (dinv ? dinv * u : u), FP64 accumulation of the correction
template <typename T>
__global__ void k_axpy_prec(double* __restrict__ x, const T* __restrict__ u,
                            const double* __restrict__ dinv, int64_t n)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double ui = (double)u[i];
  x[i] += dinv ? dinv[i] * ui : ui;
}

// r = b - A x (FP64) with per-block partial ||r||^2; G lanes per row
template <int G>
__global__ __launch_bounds__(kBlock) void k_residual(
  const int32_t* __restrict__ rp, const int32_t* __restrict__ ci,
  const double* __restrict__ va, const double* __restrict__ x,
  const double* __restrict__ b, double* __restrict__ r, int n,
  double* __restrict__ partial)
{
  double acc[1] = {0.0};
  for (int64_t t0 = (int64_t)blockIdx.x * blockDim.x; t0 < (int64_t)n * G;
       t0 += (int64_t)gridDim.x * blockDim.x) {
    const int64_t t = t0 + threadIdx.x;
    const int row = (int)(t / G);
    const int g = threadIdx.x & (G - 1);
    double s = row < n ? csr_dot<double, G>(rp, ci, va, x, row, g) : 0.0;
    for (int o = G / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, G);
    if (row < n && g == 0) {
      const double ri = b[row] - s;
      r[row] = ri;
      acc[0] += ri * ri;
    }
  }
  block_reduce_store<1>(acc, partial + blockIdx.x);
}

__global__ void k_diag_inv(const int32_t* __restrict__ diag,
                           const double* __restrict__ va,
                           double* __restrict__ dinv, int n,
                           int* __restrict__ bad)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double d = va[diag[i]];
  if (!(d != 0.0) || !isfinite(d)) atomicOr(bad, 1);
  dinv[i] = 1.0 / d;
}

template <typename T>
__global__ void k_convert(const double* __restrict__ a, T* __restrict__ b,
                          double scale, int64_t n)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) b[i] = (T)(a[i] * scale);
}

__global__ void k_seed_vec(double* __restrict__ x, int64_t n, uint64_t seed)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  uint64_t z = seed + 0x9e3779b97f4a7c15ULL * (uint64_t)(i + 1);
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
  z ^= z >> 31;
  x[i] = (double)(z >> 11) * (1.0 / 9007199254740992.0) + 0.5;
}

__global__ void k_vmul(double* __restrict__ y, const double* __restrict__ d,
                       int64_t n)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] *= d[i];
}

// *flag = 1 if a and b differ anywhere (flag cleared by the caller)
__global__ void k_differs(const double* __restrict__ a,
                          const double* __restrict__ b, int64_t n,
                          int* __restrict__ flag)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && a[i] != b[i]) *flag = 1;
}


unsigned stream_grid(int64_t n)
{
  return (unsigned)std::max<int64_t>(1, std::min<int64_t>(grid_for(n, kBlock), 4096));
}

// width[k] = longest row of slice k (a wave per slice)
__global__ __launch_bounds__(kBlock) void k_sell_width(
  const int32_t* __restrict__ rp, int n, int nslices, int32_t* __restrict__ width)
{
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  int len = t < n ? rp[t + 1] - rp[t] : 0;
  for (int o = kWave / 2; o > 0; o >>= 1) len = max(len, __shfl_xor(len, o, kWave));
  if ((threadIdx.x & (kWave - 1)) == 0 && (t >> 6) < nslices) width[t >> 6] = len;
}

// The offset form of each slice (a wave per slice): the sorted union of
// its rows' column offsets (column - row), taken one smallest offset at a
// time over the wave, when it has at most kDiaMax values and row + offset
// lies in [0, n) for every row of the slice; dia_w[k] = its size, or 0.
__global__ __launch_bounds__(kBlock) void k_dia_pattern(
  const int32_t* __restrict__ rp, const int32_t* __restrict__ ci, int n, int nslices,
  int32_t* __restrict__ dia_w, int32_t* __restrict__ dia_off)
{
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int k = t >> 6;
  if (k >= nslices) return;  // whole waves
  const int lane = t & 63;
  const bool valid = t < n;
  int pos = valid ? rp[t] : 0;
  const int end = valid ? rp[t + 1] : 0;
  int cnt = 0;
  bool ok = true;
  for (;;) {
    const int mine = pos < end ? ci[pos] - t : INT_MAX;
    int cand = mine;
    for (int o = kWave / 2; o > 0; o >>= 1) cand = min(cand, __shfl_xor(cand, o, kWave));
    if (cand == INT_MAX) break;  // the same on every lane
    if (cnt == kDiaMax) {
      ok = false;
      break;
    }
    const int64_t col = (int64_t)t + cand;
    if (__ballot(valid && (col < 0 || col >= n)) != 0) {
      ok = false;
      break;
    }
    if (lane == 0) dia_off[(int64_t)k * kDiaMax + cnt] = cand;
    ++cnt;
    if (mine == cand) ++pos;
  }
  if (lane == 0) dia_w[k] = ok ? cnt : 0;
}

// columns and CSR slots of every sliced-ELL position (a lane per row);
// padding positions take the row's own index as their column (square
// matrices) or, with pad_last, the row's last column (column 0 for an
// empty row), which stays inside any matrix's columns.  A slice in offset
// form puts each row's entry with offset dia_off[j] at position j.
__global__ __launch_bounds__(kBlock) void k_sell_struct(
  const int32_t* __restrict__ rp, const int32_t* __restrict__ ci, int n,
  const int64_t* __restrict__ sp, int nslices, int32_t* __restrict__ sci,
  int32_t* __restrict__ sslot, bool pad_last, const int32_t* __restrict__ dia_w,
  const int32_t* __restrict__ dia_off)
{
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int k = t >> 6;
  if (k >= nslices) return;
  const int64_t b = sp[k] + (t & 63);
  const int w = (int)((sp[k + 1] - sp[k]) >> 6);
  const int r0 = t < n ? rp[t] : 0;
  const int len = t < n ? rp[t + 1] - r0 : 0;
  if (dia_w && dia_w[k] > 0) {
    int q = r0;  // the row's entries, in column (= offset) order
    for (int j = 0; j < w; ++j) {
      const int64_t p = b + 64 * (int64_t)j;
      const int off = dia_off[(int64_t)k * kDiaMax + j];
      if (t < n) {
        sci[p] = t + off;
        if (q < r0 + len && ci[q] - t == off) {
          sslot[p] = q;
          ++q;
        } else {
          sslot[p] = -1;
        }
      } else {
        sci[p] = 0;
        sslot[p] = -1;
      }
    }
    return;
  }
  for (int j = 0; j < w; ++j) {
    const int64_t p = b + 64 * (int64_t)j;
    if (j < len) {
      sci[p] = ci[r0 + j];
      sslot[p] = r0 + j;
    } else {
      sci[p] = pad_last ? (len > 0 ? ci[r0 + len - 1] : 0) : (t < n ? t : 0);
      sslot[p] = -1;
    }
  }
}

// The delta form of each slice not in offset form (a wave per slice): when
// its columns span less than 65536, base[k] = the smallest and cd[p] = column
// - base; else base[k] = -1.
__global__ __launch_bounds__(kBlock) void k_sell_delta16(
  const int64_t* __restrict__ sp, const int32_t* __restrict__ sci, int nslices,
  const int32_t* __restrict__ dia_w, uint16_t* __restrict__ cd, int32_t* __restrict__ base)
{
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int k = t >> 6;
  if (k >= nslices) return;  // whole waves
  const int64_t b = sp[k] + (t & 63);
  const int w = (int)((sp[k + 1] - sp[k]) >> 6);
  int lo = INT_MAX, hi = 0;
  for (int j = 0; j < w; ++j) {
    const int c = sci[b + 64 * (int64_t)j];
    lo = min(lo, c);
    hi = max(hi, c);
  }
  for (int o = kWave / 2; o > 0; o >>= 1) {
    lo = min(lo, __shfl_xor(lo, o, kWave));
    hi = max(hi, __shfl_xor(hi, o, kWave));
  }
  const bool ok = w > 0 && (dia_w == nullptr || dia_w[k] == 0) && hi - lo < 65536;
  for (int j = 0; j < w; ++j) {
    const int64_t p = b + 64 * (int64_t)j;
    cd[p] = ok ? (uint16_t)(sci[p] - lo) : (uint16_t)0;
  }
  if ((t & 63) == 0) base[k] = ok ? lo : -1;
}

}  // namespace

void sell_free(Sell& s)
{
  for (void* p : {(void*)s.sp, (void*)s.ci, (void*)s.slot, (void*)s.dia_w, (void*)s.dia_off,
                  (void*)s.base, (void*)s.cd})
    (void)hipFree(p);
  s = Sell();
}

int sell_build(const int32_t* rp, const int32_t* ci, int n, Sell& s,
               hipStream_t st, bool pad_last, bool offsets)
{
  // the callers pass a new structure or one a failed build left part way
  sell_free(s);
  s.n = n;
  s.nslices = (n + kWave - 1) / kWave;
  const int ns = s.nslices;
  const unsigned grid = grid_for((int64_t)ns * kWave, kBlock);
  int32_t* dw = nullptr;
  NW_HIP(hipMalloc(&dw, sizeof(int32_t) * std::max(ns, 1)));
  k_sell_width<<<grid, kBlock, 0, st>>>(rp, n, ns, dw);
  std::vector<int32_t> w(ns), dia(offsets ? ns : 0);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess && offsets) {
    e = hipMalloc(&s.dia_w, sizeof(int32_t) * std::max(ns, 1));
    if (e == hipSuccess)
      e = hipMalloc(&s.dia_off, sizeof(int32_t) * (size_t)std::max(ns, 1) * kDiaMax);
    if (e == hipSuccess) {
      k_dia_pattern<<<grid, kBlock, 0, st>>>(rp, ci, n, ns, s.dia_w, s.dia_off);
      e = hipGetLastError();
    }
    if (e == hipSuccess)
      e = hipMemcpyAsync(dia.data(), s.dia_w, sizeof(int32_t) * ns, hipMemcpyDeviceToHost, st);
  }
  if (e == hipSuccess)
    e = hipMemcpyAsync(w.data(), dw, sizeof(int32_t) * ns, hipMemcpyDeviceToHost, st);
  if (e == hipSuccess) e = hipStreamSynchronize(st);
  (void)hipFree(dw);
  NW_HIP(e);
  std::vector<int64_t> sp(ns + 1, 0);
  s.dia_slices = 0;
  for (int k = 0; k < ns; ++k) {
    const int wk = offsets && dia[k] > 0 ? dia[k] : w[k];  // the union holds every row
    s.dia_slices += offsets && dia[k] > 0;
    sp[k + 1] = sp[k] + (int64_t)kWave * wk;
  }
  if (offsets && s.dia_slices == 0) {  // nothing to gain: the plain form
    (void)hipFree(s.dia_w);
    (void)hipFree(s.dia_off);
    s.dia_w = s.dia_off = nullptr;
  }
  s.len = sp[ns];
  NW_HIP(hipMalloc(&s.sp, sizeof(int64_t) * (ns + 1)));
  NW_HIP(hipMalloc(&s.ci, sizeof(int32_t) * std::max<int64_t>(s.len, 1)));
  NW_HIP(hipMalloc(&s.slot, sizeof(int32_t) * std::max<int64_t>(s.len, 1)));
  NW_HIP(hipMemcpyAsync(s.sp, sp.data(), sizeof(int64_t) * (ns + 1),
                        hipMemcpyHostToDevice, st));
  k_sell_struct<<<grid, kBlock, 0, st>>>(rp, ci, n, s.sp, ns, s.ci, s.slot, pad_last,
                                         s.dia_w, s.dia_off);
  NW_LAUNCH_CHECK();
  NW_HIP(hipMalloc(&s.base, sizeof(int32_t) * std::max(ns, 1)));
  NW_HIP(hipMalloc(&s.cd, sizeof(uint16_t) * std::max<int64_t>(s.len, 1)));
  k_sell_delta16<<<grid, kBlock, 0, st>>>(s.sp, s.ci, ns, s.dia_w, s.cd, s.base);
  NW_LAUNCH_CHECK();
  std::vector<int32_t> base(ns);
  NW_HIP(hipMemcpyAsync(base.data(), s.base, sizeof(int32_t) * ns, hipMemcpyDeviceToHost, st));
  NW_HIP(hipStreamSynchronize(st));
  s.delta_slices = 0;
  for (int k = 0; k < ns; ++k) s.delta_slices += base[k] >= 0;
  if (s.delta_slices == 0) {  // nothing to gain
    (void)hipFree(s.base);
    (void)hipFree(s.cd);
    s.base = nullptr;
    s.cd = nullptr;
  }
  NW_HIP(hipStreamSynchronize(st));
  return NW_OK;
}

// ---------------------------------------------------------------- workspace

template <typename T>
struct Space {
  T* V = nullptr;      // (m+1) x n basis
  T* mat = nullptr;    // matrix values in T (Jacobi: columns scaled)
  T* dinv = nullptr;   // Chebyshev only
  T *cz = nullptr, *cd = nullptr, *cz2 = nullptr, *u = nullptr;
};

struct Krylov {
  int64_t n = 0, nnz = 0;
  int m = 0;
  double* dinv = nullptr;  // FP64 1/diag
  double* r = nullptr;     // FP64 residual
  double* partial = nullptr;
  double* red = nullptr;   // reduced results (device)
  double* coef = nullptr;  // coefficients (device)
  double* hs = nullptr;    // a cycle's small dense state (device)
  // the steps' decisions in pinned memory, step by step in turn, and the
  // number of the last step enqueued
  volatile unsigned long long* status = nullptr;
  unsigned long long token = 0;
  double* pe = nullptr;    // power iteration work
  double* xg = nullptr;    // learned guess
  int* bad = nullptr;
  double* h_pinned = nullptr;  // host pinned scratch
  Space<double> d;
  Space<float> f;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
};

constexpr int kPartialCap = kRowBlocks * kTile * kDotVals;  // doubles
constexpr int kRedCap = kTile * kDotVals + 8;

template <typename T>
static void free_space(Space<T>& s)
{
  (void)hipFree(s.V);
  (void)hipFree(s.mat);
  (void)hipFree(s.dinv);
  (void)hipFree(s.cz);
  (void)hipFree(s.cd);
  (void)hipFree(s.cz2);
  (void)hipFree(s.u);
  s = Space<T>();
}

void free_krylov(Krylov* k)
{
  if (!k) return;
  (void)hipFree(k->dinv);
  (void)hipFree(k->r);
  (void)hipFree(k->partial);
  (void)hipFree(k->red);
  (void)hipFree(k->coef);
  (void)hipFree(k->hs);
  (void)hipHostFree((void*)k->status);
  (void)hipFree(k->pe);
  (void)hipFree(k->xg);
  (void)hipFree(k->bad);
  (void)hipHostFree(k->h_pinned);
  free_space(k->d);
  free_space(k->f);
  if (k->ev0) (void)hipEventDestroy(k->ev0);
  if (k->ev1) (void)hipEventDestroy(k->ev1);
  delete k;
}

template <typename T>
static int alloc_space(Space<T>& s, int64_t n, int64_t nnz, int m, bool cheb, bool amg)
{
  if (!s.V) NW_HIP(hipMalloc(&s.V, sizeof(T) * n * (m + 1)));
  if (!s.mat) NW_HIP(hipMalloc(&s.mat, sizeof(T) * nnz));  // sliced ELL order
  if (!s.u) NW_HIP(hipMalloc(&s.u, sizeof(T) * n));
  if ((cheb || amg) && !s.cz) NW_HIP(hipMalloc(&s.cz, sizeof(T) * n));
  if (cheb) {
    if (!s.dinv) NW_HIP(hipMalloc(&s.dinv, sizeof(T) * n));
    if (!s.cd) NW_HIP(hipMalloc(&s.cd, sizeof(T) * n));
    if (!s.cz2) NW_HIP(hipMalloc(&s.cz2, sizeof(T) * n));
  }
  return NW_OK;
}

// The solver state of one call.
struct Solve {
  Ctx* c;
  Krylov* k;
  const nw_solver_cfg* cfg;
  int G;  // lanes per row
  double lmax = 0, lmin = 0;
  int iters = 0;
  hipStream_t st = nullptr;

  // reduce nb x nv partials to nv values and copy them to the host
  int reduce(int nb, int nv, double* host)
  {
    k_reduce<<<nv, kBlock, 0, st>>>(k->partial, nb, k->red);
    NW_LAUNCH_CHECK();
    NW_HIP(hipMemcpyAsync(k->h_pinned, k->red, sizeof(double) * nv,
                          hipMemcpyDeviceToHost, st));
    NW_HIP(hipStreamSynchronize(st));
    std::memcpy(host, k->h_pinned, sizeof(double) * nv);
    return NW_OK;
  }

  // y = alpha A x with A in sliced ELL order (the space's matrix copy)
  template <typename T>
  int spmv(const T* va, const T* x, T* y, T alpha)
  {
    const int n = (int)k->n;
    k_sell_spmv<T, 1><<<grid_for(n, kBlock), kBlock, 0, st>>>(
      sell_view(c->g.sell), va, x, y, n, alpha);
    NW_LAUNCH_CHECK();
    return NW_OK;
  }

  // y = alpha A x with A the assembled CSR values
  int spmv_csr(const double* va, const double* x, double* y, double alpha)
  {
    const int n = (int)k->n;
    NW_ROW_LAUNCH(k_spmv, double, G, n, st, c->g.row_ptr, c->g.cols, va, x, y,
                  n, alpha);
    NW_LAUNCH_CHECK();
    return NW_OK;
  }

  template <typename T>
  int cheb_step(const T* va, const T* z, const T* v, const T* dinv, T* d, T* zo,
                T c1, T c2)
  {
    const int n = (int)k->n;
    k_sell_cheb_step<T><<<grid_for(n, kBlock), kBlock, 0, st>>>(
      sell_view(c->g.sell), va, z, v, dinv, d, zo, n, c1, c2);
    NW_LAUNCH_CHECK();
    return NW_OK;
  }

  // z = p(D^-1 A) D^-1 v, the Chebyshev polynomial (Jacobi is folded into
  // the matrix columns instead when it is the preconditioner)
  template <typename T>
  int cheb_apply(Space<T>& s, const T* v, T** zout)
  {
    const int n = (int)k->n;
    const double theta = 0.5 * (lmax + lmin), delta = 0.5 * (lmax - lmin);
    const double sigma = theta / delta;
    double rho = 1.0 / sigma;
    k_cheb_init<T><<<grid_for(n, kBlock), kBlock, 0, st>>>(v, s.dinv, s.cd, s.cz,
                                                          n, (T)(1.0 / theta));
    NW_LAUNCH_CHECK();
    T* z = s.cz;
    T* z2 = s.cz2;
    for (int it = 1; it < cfg->cheb_degree; ++it) {
      const double rho_new = 1.0 / (2.0 * sigma - rho);
      int rc = cheb_step<T>(s.mat, z, v, s.dinv, s.cd, z2, (T)(rho_new * rho),
                            (T)(2.0 * rho_new / delta));
      if (rc) return rc;
      std::swap(z, z2);
      rho = rho_new;
    }
    *zout = z;
    return NW_OK;
  }

  // W = A M^-1 v (under AMG as (A D^-1) (D M^-1 v): the V-cycle works on
  // column-scaled operators and returns D M^-1 v)
  template <typename T>
  int apply_op(Space<T>& s, const T* v, T* W)
  {
    if (cfg->precond == NW_PREC_AMG) {
      int rc = amg_apply<T>(c->amg, v, s.cz, st);
      if (rc) return rc;
      return spmv<T>(s.mat, s.cz, W, (T)1);
    }
    if (cfg->precond == NW_PREC_CHEBYSHEV) {
      T* z = nullptr;
      int rc = cheb_apply<T>(s, v, &z);
      if (rc) return rc;
      return spmv<T>(s.mat, z, W, (T)1);
    }
    return spmv<T>(s.mat, v, W, (T)1);
  }

  // Enqueues the dots of step j (Q = V[0..j), y = V[j], z = V[j+1] if grow)
  // and the work that ends the step; its decision arrives under *token.
  template <typename T>
  int arnoldi_step(const T* V, int j, bool grow, double beta, double stop_abs,
                   unsigned long long* token)
  {
    const int64_t n = k->n;
    const int ntiles = std::max(1, (j + kTile - 1) / kTile);
    const int nrb = dot_row_blocks(n, 16 / (int)sizeof(T), ntiles);
    const int nv = ntiles * kDotVals;
    // up to kDirect row blocks the step adds their partials itself (a thread
    // per value, rows of values); more go through a reduction of their own
    constexpr int kDirect = 48;
    const bool direct = nrb <= kDirect;
    k_arnoldi_dots<T><<<nrb * ntiles, kBlock, 0, st>>>(
      V, n, j, V + (int64_t)j * n, grow ? V + (int64_t)(j + 1) * n : nullptr,
      ntiles, k->partial, direct ? 1 : nrb, direct ? nv : 1);
    if (!direct) k_reduce<<<nv, kBlock, 0, st>>>(k->partial, nrb, k->red);
    NW_LAUNCH_CHECK();
    *token = ++k->token;
    k_arnoldi_step<<<1, kBlock, 0, st>>>(
      direct ? k->partial : k->red, direct ? nrb : 1, nv, j, grow ? 1 : 0, beta, stop_abs,
      k->hs, k->coef, const_cast<unsigned long long*>(k->status) + (*token & 1), *token);
    NW_LAUNCH_CHECK();
    return NW_OK;
  }

  // Waits for the decision of step `token`; the word is written by a kernel
  // already enqueued, so the wait ends with it or with the stream's error.
  int step_status(unsigned long long token, bool* stop, int* kdim)
  {
    const volatile unsigned long long* w = k->status + (token & 1);
    for (unsigned spin = 1;; ++spin) {
      const unsigned long long v = *w;
      if (v >> 16 == token) {
        *stop = (v >> 8 & 1) != 0;
        *kdim = (int)(v & 0xff);
        return NW_OK;
      }
      __builtin_ia32_pause();  // a whole AMG step goes by here: leave the core's
                               // other thread and the memory bus alone
      if (spin % 4096 == 0) {
        const hipError_t e = hipStreamQuery(st);
        if (e == hipErrorNotReady) {
          (void)hipGetLastError();  // not an error of a later launch
          continue;
        }
        NW_HIP(e);
        NW_REQUIRE(*w >> 16 == token, NW_E_HIP, "the solver step left no decision");
      }
    }
  }

  template <typename T>
  int arnoldi_update(T* V, int nq)
  {
    k_arnoldi_update<T><<<stream_grid(k->n), kBlock, 0, st>>>(V, k->n, nq, k->coef);
    NW_LAUNCH_CHECK();
    return NW_OK;
  }

  template <typename T>
  int combine(const T* V, int nk, const double* coef, T* u)
  {
    k_combine<T><<<stream_grid(k->n), kBlock, 0, st>>>(V, k->n, nk, coef, u);
    NW_LAUNCH_CHECK();
    return NW_OK;
  }

  // r = b - A x in FP64; returns ||r||
  int residual(const double* x, double* rnorm)
  {
    const int n = (int)k->n;
    // a grid of at most 4096 blocks strides over the rows: the partials of
    // one block per 256 lanes made the reduction after it, by one workgroup,
    // cost up to 38 us
    const int nb = (int)std::min<int64_t>(grid_for((int64_t)n * G, kBlock), 4096);
    switch (G) {
    case 1:
      k_residual<1><<<nb, kBlock, 0, st>>>(c->g.row_ptr, c->g.cols, c->g.vals, x, c->g.rhs, k->r, n, k->partial);
      break;
    case 2:
      k_residual<2><<<nb, kBlock, 0, st>>>(c->g.row_ptr, c->g.cols, c->g.vals, x, c->g.rhs, k->r, n, k->partial);
      break;
    case 4:
      k_residual<4><<<nb, kBlock, 0, st>>>(c->g.row_ptr, c->g.cols, c->g.vals, x, c->g.rhs, k->r, n, k->partial);
      break;
    case 8:
      k_residual<8><<<nb, kBlock, 0, st>>>(c->g.row_ptr, c->g.cols, c->g.vals, x, c->g.rhs, k->r, n, k->partial);
      break;
    case 16:
      k_residual<16><<<nb, kBlock, 0, st>>>(c->g.row_ptr, c->g.cols, c->g.vals, x, c->g.rhs, k->r, n, k->partial);
      break;
    default:
      k_residual<32><<<nb, kBlock, 0, st>>>(c->g.row_ptr, c->g.cols, c->g.vals, x, c->g.rhs, k->r, n, k->partial);
    }
    NW_LAUNCH_CHECK();
    double r2 = 0;
    int rc = reduce(nb, 1, &r2);
    *rnorm = std::sqrt(r2);
    return rc;
  }

  // ||v||^2 and v.w of FP64 vectors (w may equal v)
  int dot64(const double* v, const double* w, double* vw)
  {
    const int nrb = dot_row_blocks(k->n, 2, 1);
    k_arnoldi_dots<double><<<nrb, kBlock, 0, st>>>(
      v, k->n, 0, v, w, 1, k->partial, nrb, 1);
    NW_LAUNCH_CHECK();
    std::vector<double> r(kDotVals);
    int rc = reduce(nrb, kDotVals, r.data());
    *vw = r[2 * kTile + 1];
    return rc;
  }

  // One GMRES(m) cycle in type T on A d = r (r = k->r, FP64, ||r|| = beta),
  // then x += M^-1 Q y in FP64.  Stops early when the Arnoldi residual
  // estimate reaches stop_abs.
  template <typename T>
  int cycle(Space<T>& s, double* x, double beta, double stop_abs, int max_it)
  {
    const int64_t n = k->n;
    const int m = std::min(cfg->kspace, max_it);
    // With a cheap operator the steps run one ahead of their decisions: the
    // host enqueues step j + 1 before it knows whether step j ends the
    // cycle, so short kernels follow each other without a gap (a step past
    // the end changes nothing that is read: its column, rotation and basis
    // vectors lie behind the first kdim).  Under a polynomial or AMG a wasted
    // application would cost more than the gap, which the update hides.
    const bool ahead = cfg->precond == NW_PREC_NONE || cfg->precond == NW_PREC_JACOBI;
    T* V = s.V;
    k_convert<T><<<grid_for(n, kBlock), kBlock, 0, st>>>(k->r, V, 1.0 / beta, n);
    NW_LAUNCH_CHECK();
    int kdim = 0, rc = NW_OK;
    bool stop = false;
    unsigned long long token = 0;
    for (int j = 0; j <= m && !stop; ++j) {
      const bool grow = j < m;
      if (grow) {
        rc = apply_op<T>(s, V + (int64_t)j * n, V + (int64_t)(j + 1) * n);
        if (rc) return rc;
      }
      const unsigned long long before = token;
      rc = arnoldi_step<T>(V, j, grow, beta, stop_abs, &token);
      if (!rc && grow) rc = arnoldi_update<T>(V, j);
      if (!rc && (!ahead || j > 0)) rc = step_status(ahead ? before : token, &stop, &kdim);
      if (rc) return rc;
    }
    if (!stop) {
      rc = step_status(token, &stop, &kdim);
      if (rc) return rc;
    }
    iters += kdim;
    if (kdim == 0) return NW_OK;
    // least squares R y = g, u = Q y, x += M^-1 u
    k_arnoldi_solve<<<1, kBlock, 0, st>>>(k->hs, kdim);
    NW_LAUNCH_CHECK();
    rc = combine<T>(V, kdim, k->hs + kHsY, s.u);
    if (rc) return rc;
    const T* u = s.u;
    if (cfg->precond == NW_PREC_CHEBYSHEV) {
      T* z = nullptr;
      rc = cheb_apply<T>(s, s.u, &z);
      if (rc) return rc;
      u = z;
    } else if (cfg->precond == NW_PREC_AMG) {
      rc = amg_apply<T>(c->amg, s.u, s.cz, st);
      if (rc) return rc;
      u = s.cz;
    }
    // under Jacobi and AMG u is D M^-1 Q y, the iterate of A D^-1
    const double* dinv = cfg->precond == NW_PREC_JACOBI ? k->dinv
                         : cfg->precond == NW_PREC_AMG  ? amg_fine_dinv(c->amg)
                                                        : nullptr;
    k_axpy_prec<T><<<grid_for(n, kBlock), kBlock, 0, st>>>(x, u, dinv, n);
    NW_LAUNCH_CHECK();
    return NW_OK;
  }

  // lambda_max of D^-1 A by power iteration from a seeded vector (FP64)
  int power_lambda(double* lam)
  {
    const int64_t n = k->n;
    double* xa = k->pe;
    double* ya = k->pe + n;
    k_seed_vec<<<grid_for(n, kBlock), kBlock, 0, st>>>(xa, n, 12345);
    NW_LAUNCH_CHECK();
    double l = 0.0;
    for (int it = 0; it < 30; ++it) {
      double xx = 0;
      int rc = dot64(xa, xa, &xx);
      if (rc) return rc;
      const double inv = 1.0 / std::sqrt(xx);
      rc = spmv_csr(c->g.vals, xa, ya, inv);
      if (rc) return rc;
      k_vmul<<<grid_for(n, kBlock), kBlock, 0, st>>>(ya, k->dinv, n);
      NW_LAUNCH_CHECK();
      double xy = 0;
      rc = dot64(xa, ya, &xy);
      if (rc) return rc;
      l = xy * inv;
      std::swap(xa, ya);
    }
    *lam = l;
    return NW_OK;
  }
};

}  // namespace nw

using namespace nw;

extern "C" {

int nw_linsys_amg_level(nw_ctx* c, int level, int64_t* rows, int64_t* nnz)
{
  NW_REQUIRE(c && rows && nnz, NW_E_ARG, "null argument");
  NW_REQUIRE(c->amg, NW_E_ARG, "no AMG hierarchy (run an AMG solve first)");
  NW_REQUIRE(amg_level_info(c->amg, level, rows, nnz) == NW_OK, NW_E_ARG,
             "level %d out of range", level);
  return NW_OK;
}

int nw_linsys_spmv(nw_ctx* c, const double* d_x, double* d_y)
{
  NW_REQUIRE(c && c->g.ndof == 1 && d_x && d_y, NW_E_STATE,
             "spmv needs a built 1-dof system");
  const int n = (int)c->g.nnode;
  const int G = lanes_per_row((double)c->g.nnzb / std::max<int64_t>(n, 1));
  NW_ROW_LAUNCH(k_spmv, double, G, n, c->stream, c->g.row_ptr, c->g.cols,
                c->g.vals, d_x, d_y, n, 1.0);
  NW_LAUNCH_CHECK();
  return NW_OK;
}

int nw_linsys_solve(nw_ctx* c, const nw_solver_cfg* cfg, nw_solve_stats* out)
{
  NW_REQUIRE(c && cfg && out, NW_E_ARG, "null argument");
  NW_REQUIRE(c->g.ndof == 1, NW_E_STATE, "solve needs a built 1-dof system");
  NW_REQUIRE(cfg->kspace >= 1 && cfg->kspace < kMaxBasis, NW_E_ARG,
             "kspace must be in [1, %d)", kMaxBasis);
  NW_REQUIRE(cfg->tol > 0 && cfg->max_iters >= 0, NW_E_ARG, "bad tolerance");
  NW_REQUIRE(cfg->precond >= NW_PREC_NONE && cfg->precond <= NW_PREC_AMG,
             NW_E_ARG, "bad preconditioner");
  NW_REQUIRE(cfg->precond != NW_PREC_CHEBYSHEV ||
               (cfg->cheb_degree >= 1 && cfg->cheb_ratio > 1.0),
             NW_E_ARG, "bad Chebyshev parameters");
  NW_REQUIRE(cfg->mode == NW_SOLVE_FP64 || cfg->mode == NW_SOLVE_FP32_REFINE,
             NW_E_ARG, "bad solve mode");
  NW_REQUIRE(cfg->x0 == NW_X0_ZERO || cfg->x0 == NW_X0_SOLUTION ||
               cfg->x0 == NW_X0_LEARNED,
             NW_E_ARG, "bad x0 mode %d", cfg->x0);
  NW_REQUIRE(cfg->x0 != NW_X0_LEARNED || c->mpnn, NW_E_STATE,
             "x0 = learned needs a network (nw_linsys_set_learned_guess)");
  std::memset(out, 0, sizeof(*out));
  NW_HIP(hipSetDevice(c->device));
  const int64_t n = c->g.nnode, nnz = c->g.nnzb;
  const bool cheb = cfg->precond == NW_PREC_CHEBYSHEV;
  const bool amgp = cfg->precond == NW_PREC_AMG;
  const bool f32 = cfg->mode == NW_SOLVE_FP32_REFINE;
  if (c->kry && (c->kry->n != n || c->kry->m < cfg->kspace)) {
    free_krylov(c->kry);
    c->kry = nullptr;
  }
  if (!c->kry) {
    c->kry = new Krylov();
    c->kry->n = n;
    c->kry->nnz = nnz;
    c->kry->m = cfg->kspace;
  }
  Krylov* k = c->kry;
  if (!k->dinv) {
    NW_HIP(hipMalloc(&k->dinv, sizeof(double) * n));
    NW_HIP(hipMalloc(&k->r, sizeof(double) * n));
    NW_HIP(hipMalloc(&k->partial, sizeof(double) * kPartialCap));
    NW_HIP(hipMalloc(&k->red, sizeof(double) * kRedCap));
    NW_HIP(hipMalloc(&k->coef, sizeof(double) * kCoefSize));
    NW_HIP(hipMalloc(&k->hs, sizeof(double) * kHsSize));
    void* hst = nullptr;
    NW_HIP(hipHostMalloc(&hst, 2 * sizeof(unsigned long long), hipHostMallocCoherent));
    std::memset(hst, 0, 2 * sizeof(unsigned long long));
    k->status = static_cast<volatile unsigned long long*>(hst);
    NW_HIP(hipMalloc(&k->bad, sizeof(int)));
    NW_HIP(hipHostMalloc(&k->h_pinned, sizeof(double) * kRedCap));
    NW_HIP(hipEventCreate(&k->ev0));
    NW_HIP(hipEventCreate(&k->ev1));
  }
  if (!c->g.sell.ci) {
    int rc0 = sell_build(c->g.row_ptr, c->g.cols, (int)n, c->g.sell, c->stream,
                         false, true);
    if (rc0) return rc0;
  }
  const int64_t slen = c->g.sell.len;
  int rc = f32 ? alloc_space(k->f, n, slen, k->m, cheb, amgp)
               : alloc_space(k->d, n, slen, k->m, cheb, amgp);
  if (rc) return rc;
  if (cheb && !k->pe) NW_HIP(hipMalloc(&k->pe, sizeof(double) * 2 * n));

  hipStream_t st = c->stream;
  // k->dinv = 1 / diag; refuses a zero or non-finite diagonal
  auto diag_inv = [&]() -> int {
    NW_HIP(hipMemsetAsync(k->bad, 0, sizeof(int), st));
    k_diag_inv<<<grid_for(n, kBlock), kBlock, 0, st>>>(c->g.diag, c->g.vals,
                                                      k->dinv, (int)n, k->bad);
    NW_LAUNCH_CHECK();
    int bad = 0;
    NW_HIP(hipMemcpyAsync(&bad, k->bad, sizeof(int), hipMemcpyDeviceToHost, st));
    NW_HIP(hipStreamSynchronize(st));
    NW_REQUIRE(!bad, NW_E_NONFINITE, "zero or non-finite diagonal in the matrix");
    return NW_OK;
  };
  if (amgp && (!c->amg || !cfg->reuse_preconditioner)) {
    // before the setup: a hierarchy outlives this call, and its 1 / diag (0
    // for a zero diagonal) scales the operator of every solve that reuses it
    rc = diag_inv();
    if (rc) return rc;
    amg_free(c->amg);
    c->amg = nullptr;
    rc = amg_setup(c, &c->amg);
    if (rc) return rc;
    out->setup_ms = 1e3 * amg_setup_seconds(c->amg);
  }
  if (amgp) {
    // the cycle's matrix copy is the V-cycle's fine level
    double narrow_s = 0.0;  // the FP32 hierarchy, made on first use
    rc = f32 ? amg_prepare<float>(c, c->amg, k->f.mat, &narrow_s)
             : amg_prepare<double>(c, c->amg, k->d.mat);
    if (rc) return rc;
    out->setup_ms += 1e3 * narrow_s;
    out->precond_levels = amg_levels(c->amg);
  }
  NW_HIP(hipEventRecord(k->ev0, st));
  Solve S{c, k, cfg, lanes_per_row((double)nnz / std::max<int64_t>(n, 1))};
  S.st = st;
  // preconditioner setup: 1/diag, the matrix in the cycle type
  rc = diag_inv();
  if (rc) return rc;
  const double* colscale = cfg->precond == NW_PREC_JACOBI ? k->dinv
                           : amgp                         ? amg_fine_dinv(c->amg)
                                                          : nullptr;
  const Sell& sl = c->g.sell;
  if (f32) {
    k_sell_values<float><<<grid_for(sl.len, kBlock), kBlock, 0, st>>>(
      sl.slot, sl.ci, c->g.vals, colscale, k->f.mat, sl.len);
    if (cheb)
      k_convert<float><<<grid_for(n, kBlock), kBlock, 0, st>>>(k->dinv, k->f.dinv, 1.0, n);
  } else {
    k_sell_values<double><<<grid_for(sl.len, kBlock), kBlock, 0, st>>>(
      sl.slot, sl.ci, c->g.vals, colscale, k->d.mat, sl.len);
    if (cheb)
      k_convert<double><<<grid_for(n, kBlock), kBlock, 0, st>>>(k->dinv, k->d.dinv, 1.0, n);
  }
  NW_LAUNCH_CHECK();
  if (cheb) {
    double lam = 0;
    rc = S.power_lambda(&lam);
    if (rc) return rc;
    S.lmax = 1.1 * lam;
    S.lmin = S.lmax / cfg->cheb_ratio;
  }
  double* x = c->g.sln;
  if (cfg->x0 == NW_X0_ZERO) NW_HIP(hipMemsetAsync(x, 0, sizeof(double) * n, st));
  // History of starting guesses (the learned guess's inputs and recorded
  // training pairs): xh[0..nh-1] are the guesses of the latest (up to
  // kHist) solves that started from the solution vector with distinct
  // guesses, newest first.  A solve from x0 = 0, or from the same guess as
  // the last one (another method on the same step), leaves the history as
  // it is.  The buffers rotate; only the new guess is copied.
  if (cfg->x0 != NW_X0_ZERO) {
    bool shift = true;
    if (c->nh > 0) {
      NW_HIP(hipMemsetAsync(k->bad, 0, sizeof(int), st));
      k_differs<<<grid_for(n, kBlock), kBlock, 0, st>>>(x, c->xh[0], n, k->bad);
      NW_LAUNCH_CHECK();
      int differs = 0;
      NW_HIP(hipMemcpyAsync(&differs, k->bad, sizeof(int),
                            hipMemcpyDeviceToHost, st));
      NW_HIP(hipStreamSynchronize(st));
      shift = differs != 0;
    }
    if (shift) {
      double* last = c->xh[kHist - 1];
      for (int j = kHist - 1; j > 0; --j) c->xh[j] = c->xh[j - 1];
      if (!last) NW_HIP(hipMalloc(&last, sizeof(double) * n));
      c->xh[0] = last;
      NW_HIP(hipMemcpyAsync(c->xh[0], x, sizeof(double) * n,
                            hipMemcpyDeviceToDevice, st));
      c->nh = std::min(c->nh + 1, kHist);
    }
  }
  double bb = 0;
  rc = S.dot64(c->g.rhs, c->g.rhs, &bb);
  if (rc) return rc;
  out->bnorm = std::sqrt(bb);
  const double bnorm = out->bnorm > 0 ? out->bnorm : 1.0;
  double rnorm = 0;
  rc = S.residual(x, &rnorm);
  if (rc) return rc;
  out->guess = cfg->x0;
  if (cfg->x0 == NW_X0_LEARNED) {
    // the network's prediction from (A, b, x0); kept only if it lowers the
    // residual, otherwise GMRES starts from x0 (the previous-step guess)
    if (!k->xg) NW_HIP(hipMalloc(&k->xg, sizeof(double) * n));
    rc = mpnn_predict_device(c->mpnn, c->xh, c->nh, k->xg);
    out->guess_ms = mpnn_last_ms(c->mpnn);
    double rl = 0;
    if (rc == NW_OK) rc = S.residual(k->xg, &rl);
    if (rc != NW_OK && rc != NW_E_NONFINITE) return rc;
    if (rc == NW_OK && std::isfinite(rl) && rl < rnorm) {
      NW_HIP(hipMemcpyAsync(x, k->xg, sizeof(double) * n,
                            hipMemcpyDeviceToDevice, st));
      rnorm = rl;
    } else {
      out->guess = NW_X0_SOLUTION;
      rc = S.residual(x, &rnorm);  // the cycle starts from the residual in k->r
      if (rc) return rc;
    }
    rc = NW_OK;
  }
  out->x0_rel = rnorm / bnorm;
  while (rnorm > cfg->tol * bnorm && S.iters < cfg->max_iters &&
         std::isfinite(rnorm)) {
    const double stop_abs = cfg->tol * bnorm;
    const int budget = cfg->max_iters - S.iters;
    const int before = S.iters;
    if (f32) {
      const double inner = std::max(cfg->inner_tol, 0.0) * rnorm;
      rc = S.cycle<float>(k->f, x, rnorm, std::max(stop_abs, inner), budget);
    } else {
      rc = S.cycle<double>(k->d, x, rnorm, stop_abs, budget);
    }
    if (rc) return rc;
    ++out->refinements;
    rc = S.residual(x, &rnorm);
    if (rc) return rc;
    if (S.iters == before) break;  // no progress possible (breakdown)
  }
  NW_HIP(hipEventRecord(k->ev1, st));
  NW_HIP(hipEventSynchronize(k->ev1));
  float ms = 0;
  NW_HIP(hipEventElapsedTime(&ms, k->ev0, k->ev1));
  out->ms = ms;
  out->iters = S.iters;
  out->reorthogonalizations = S.iters;
  out->final_abs = rnorm;
  out->final_rel = rnorm / bnorm;
  out->converged = rnorm <= cfg->tol * bnorm;
  if (!std::isfinite(rnorm)) {
    set_error("solve diverged (non-finite residual)");
    return NW_E_NONFINITE;
  }
  if (!out->converged) {
    set_error("GMRES stopped at %d iterations, relative residual %.3e",
              out->iters, out->final_rel);
    return NW_E_NOCONV;
  }
  return NW_OK;
}

}  // extern "C"
