// nw_sparse.h -- sparse kernels shared by the Krylov solver and the AMG
// preconditioner: SpMV, residual and the fused Chebyshev step in two
// layouts.  Sliced ELL (one or two lanes per row, independent loads) serves
// many short rows: the fine matrix and the larger AMG levels' operators,
// prolongators and restrictions.  CSR with G lanes per row serves long rows
// and small levels, and the assembled matrix as it is (power iteration,
// nw_linsys_spmv).
#pragma once

#include "nw_internal.h"
#include "nw_sell.h"

namespace nw {

// rows from which one lane per row is as fast as two: 64 waves per CU over
// the launch, twice what a CU holds at once (measured at 0.21 and 0.93 M rows,
// sell_lanes)
constexpr int64_t kSellFillRows = 256 * 64 * 64;

// Lanes per row for CSR rows of `avg` entries: each lane takes kCsrUnroll
// entries per step as independent loads, so a row of average length is
// covered by about one step (measured on the 20-entry AMG coarse operator
// at 256^3: 8 lanes x 4 loads beat 16 lanes x 1 load by ~1.6x).  A whole wave
// takes twice as many per step (4424 rows of 363 entries, FP32: 5.7 us, 9.1
// with 32 lanes, four loads a step).
constexpr int kCsrUnroll = 4;
inline int lanes_per_row(double avg)
{
  int g = 1;
  while (g < kWave && g * kCsrUnroll < avg) g *= 2;
  return g;
}

// Partial sum of row `row` over the entries g, g+G, ... (lane g of G),
// U = kCsrUnroll (G = 64: twice that) entries per step loaded before any is used; padding entries
// repeat the row's last column with value 0.  Rows are contiguous, so the
// G lanes of a row read consecutive entries.
template <typename T, int G>
__device__ inline T csr_dot(const int32_t* __restrict__ rp,
                            const int32_t* __restrict__ ci,
                            const T* __restrict__ va, const T* __restrict__ x,
                            int row, int g)
{
  constexpr int U = G == kWave ? 2 * kCsrUnroll : kCsrUnroll;
  const int k0 = rp[row], k1 = rp[row + 1];
  T s = 0;
  for (int k = k0 + g; k < k1; k += G * U) {
    int c[U];
    T v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kk = k + u * G;
      const bool ok = kk < k1;
      c[u] = ci[ok ? kk : k1 - 1];
      v[u] = ok ? va[kk] : (T)0;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) s += v[u] * x[c[u]];
  }
  return s;
}

// y = alpha * (A x); G lanes per row.
template <typename T, int G>
__global__ __launch_bounds__(kBlock) void k_spmv(
  const int32_t* __restrict__ rp, const int32_t* __restrict__ ci,
  const T* __restrict__ va, const T* __restrict__ x, T* __restrict__ y, int n,
  T alpha)
{
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int row = (int)(t / G);
  const int g = threadIdx.x & (G - 1);
  T s = row < n ? csr_dot<T, G>(rp, ci, va, x, row, g) : (T)0;
  for (int o = G / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, G);
  if (row < n && g == 0) y[row] = alpha * s;
}

// d = dinv * v * inv_theta; z = d
template <typename T>
__global__ void k_cheb_init(const T* __restrict__ v, const T* __restrict__ dinv,
                            T* __restrict__ d, T* __restrict__ z, int n,
                            T inv_theta)
{
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const T di = dinv[i] * v[i] * inv_theta;
  d[i] = di;
  z[i] = di;
}

// Two Chebyshev terms on v from zero, with A's columns scaled to a unit
// diagonal: out = alpha v - beta A v (with ADD added to out); see
// AmgDevice in nw_amg.hip.
template <typename T, int G, bool ADD = false>
__global__ __launch_bounds__(kBlock) void k_smooth(
  const int32_t* __restrict__ rp, const int32_t* __restrict__ ci,
  const T* __restrict__ va, const T* __restrict__ v, T* __restrict__ out, int n,
  T alpha, T beta)
{
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int row = (int)(t / G);
  const int g = threadIdx.x & (G - 1);
  T s = row < n ? csr_dot<T, G>(rp, ci, va, v, row, g) : (T)0;
  for (int o = G / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, G);
  if (row < n && g == 0) {
    const T e = alpha * v[row] - beta * s;
    out[row] = ADD ? out[row] + e : e;
  }
}

// y += A x (prolongation-correction); G lanes per row.
template <typename T, int G>
__global__ __launch_bounds__(kBlock) void k_spmv_add(
  const int32_t* __restrict__ rp, const int32_t* __restrict__ ci,
  const T* __restrict__ va, const T* __restrict__ x, T* __restrict__ y, int n)
{
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int row = (int)(t / G);
  const int g = threadIdx.x & (G - 1);
  T s = row < n ? csr_dot<T, G>(rp, ci, va, x, row, g) : (T)0;
  for (int o = G / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, G);
  if (row < n && g == 0) y[row] += s;
}

// r = b - A x; G lanes per row.
template <typename T, int G>
__global__ __launch_bounds__(kBlock) void k_resid(
  const int32_t* __restrict__ rp, const int32_t* __restrict__ ci,
  const T* __restrict__ va, const T* __restrict__ x, const T* __restrict__ b,
  T* __restrict__ r, int n)
{
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int row = (int)(t / G);
  const int g = threadIdx.x & (G - 1);
  T s = row < n ? csr_dot<T, G>(rp, ci, va, x, row, g) : (T)0;
  for (int o = G / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, G);
  if (row < n && g == 0) r[row] = b[row] - s;
}

// ------------------------------------------------------------ sliced ELL
// G lanes per row (sell_lanes): a wave takes 64 / G consecutive rows of a
// slice, lane l the entries j = l / (64 / G) mod G of row l % (64 / G), so
// that for every j the lanes read consecutive values and columns; all loads
// of a lane are independent (issued eight at a time), and a wave keeps its
// rows' gathers in flight instead of walking a dependent chain.  Padding
// reads x at a valid column with value 0.  With one lane the row sum runs
// over j in order; G lanes' sums are added by a fixed butterfly.  A slice in
// offset form (A.dia_w[k] > 0) takes its columns as row + the slice's
// offsets (dia_column), which are the same for the whole wave (scalar loads
// with one lane), and reads no column array; a slice in delta form (A.base[k] >= 0)
// reads 16-bit columns relative to its base instead of the 32-bit columns.
// The hardware deals workgroups to the 8 XCDs in turn.  With A.stretch
// (matrices mostly in offset form: a box's, whose rows are alike) each XCD
// takes stretches of kStretch blocks (131 thousand rows) instead, so that the
// x of a row's neighbours is fetched into one L2 and not into several:
// 32.7 -> 25.7 us for the 4.2 M 7-entry rows of a 160^3 box (FP32), 14.4 ->
// 12.5 for 0.96 M (FP64), 251 -> 238 for 17 M (FP64).  One eighth of the rows
// to each is slower on large boxes (17 M rows, FP64: 256), 2048 blocks too
// (245).  Coarse AMG levels' rows are longer in one part of a stretched mesh
// than in another: the XCDs' shares differ (27 -> 39 us on the 933 thousand
// rows of a 160^3 box's level 1), and stretches of 1 to 16 thousand rows gain
// nothing.
constexpr unsigned kStretch = 512;
struct SellLane {
  int row, g;
};
template <int G>
__device__ inline SellLane sell_lane(bool stretch)
{
  constexpr int R = kWave / G;
  unsigned b = blockIdx.x;
  if (stretch) {
    const unsigned first = b / (8 * kStretch) * (8 * kStretch);  // of its round
    const unsigned size = min(8 * kStretch, gridDim.x - first);
    const unsigned q = size / 8, r = size % 8, xcd = b % 8;
    b = first + xcd * q + min(xcd, r) + (b - first) / 8;
  }
  const int t = b * kBlock + threadIdx.x;
  const int lane = t & (kWave - 1);
  return {(t / kWave) * R + lane % R, lane / R};
}

// Lanes that leave before the row sum: those without a row, or with several
// lanes per row only whole waves of them (the others take part in its
// butterfly).
template <int G>
__device__ inline bool sell_idle(SellLane l, int n)
{
  return (G == 1 ? l.row : l.row - l.row % (kWave / G)) >= n;
}

template <typename T, int G>
__device__ inline T sell_dot(const SellView& A, const T* __restrict__ va,
                             const T* __restrict__ x, SellLane l, int n)
{
  // rows of one wave are in one slice: the slice index is wave-uniform
  const int row = l.row;
  const int k = __builtin_amdgcn_readfirstlane(row >> 6);
  const int64_t b = A.sp[k] + (row & 63);
  const int w = (int)((A.sp[k + 1] - A.sp[k]) >> 6);
  T s = 0;
  auto sum = [&](auto column) {
    for (int j0 = l.g; j0 < w; j0 += 8 * G) {
      int c[8];
      T v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int j = min(j0 + u * G, w - 1);
        c[u] = column(j);
        v[u] = j0 + u * G < w ? va[b + 64 * (int64_t)j] : (T)0;
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) s += v[u] * x[c[u]];
    }
  };
  const int base = A.base ? A.base[k] : -1;
  if (A.dia_w && A.dia_w[k] > 0) {
    const int32_t* off = A.dia_off + (int64_t)k * kDiaMax;
    // (the check of the row, 1 % of the product, only where lanes stay)
    sum([&](int j) { return G == 1 ? row + off[j] : dia_column(row, off[j], n); });
  } else if (base >= 0) {
    sum([&](int j) { return base + A.cd[b + 64 * (int64_t)j]; });
  } else {
    sum([&](int j) { return A.ci[b + 64 * (int64_t)j]; });
  }
  for (int o = kWave / G; o < kWave; o *= 2) s += __shfl_xor(s, o);
  return s;
}

// Lanes per row of a sliced ELL matrix of n rows, `avg` entries on average:
// one where its waves fill the chip by themselves or its rows are too short
// to share, else two (level 1 of the 0.96 M-row box, 207 thousand rows of 20
// entries, FP64: 12.5 us with two lanes, 13.9 with one, 13.0 with four; of the
// 4.2 M-row one, 933 thousand rows, FP32: 27 against 28 us).
inline int sell_lanes(int64_t n, double avg)
{
  return n < kSellFillRows && avg >= 8.0 ? 2 : 1;
}

// y = alpha * (A x)
template <typename T, int G>
__global__ __launch_bounds__(kBlock) void k_sell_spmv(
  SellView A, const T* __restrict__ va, const T* __restrict__ x, T* __restrict__ y, int n,
  T alpha)
{
  const SellLane l = sell_lane<G>(A.stretch);
  if (sell_idle<G>(l, n)) return;
  const T s = sell_dot<T, G>(A, va, x, l, n);
  if (l.row < n && l.g == 0) y[l.row] = alpha * s;
}

// y += A x
template <typename T, int G>
__global__ __launch_bounds__(kBlock) void k_sell_spmv_add(
  SellView A, const T* __restrict__ va, const T* __restrict__ x, T* __restrict__ y, int n)
{
  const SellLane l = sell_lane<G>(A.stretch);
  if (sell_idle<G>(l, n)) return;
  const T s = sell_dot<T, G>(A, va, x, l, n);
  if (l.row < n && l.g == 0) y[l.row] += s;
}

// Chebyshev step: r = v - A z; d = c1 d + c2 dinv r; zo = z + d.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_sell_cheb_step(
  SellView A, const T* __restrict__ va, const T* __restrict__ z, const T* __restrict__ v,
  const T* __restrict__ dinv, T* __restrict__ d, T* __restrict__ zo, int n,
  T c1, T c2)
{
  const SellLane l = sell_lane<1>(A.stretch);
  const int row = l.row;
  if (row >= n) return;
  const T s = sell_dot<T, 1>(A, va, z, l, n);
  const T dn = c1 * d[row] + c2 * dinv[row] * (v[row] - s);
  d[row] = dn;
  zo[row] = z[row] + dn;
}

// out = alpha v - beta A v, with ADD added to out (k_smooth)
template <typename T, int G, bool ADD = false>
__global__ __launch_bounds__(kBlock) void k_sell_smooth(
  SellView A, const T* __restrict__ va, const T* __restrict__ v, T* __restrict__ out, int n,
  T alpha, T beta)
{
  const SellLane l = sell_lane<G>(A.stretch);
  const int row = l.row;
  if (sell_idle<G>(l, n)) return;
  const T s = sell_dot<T, G>(A, va, v, l, n);
  if (row < n && l.g == 0) {
    const T e = alpha * v[row] - beta * s;
    out[row] = ADD ? out[row] + e : e;
  }
}

// r = b - A x
template <typename T, int G>
__global__ __launch_bounds__(kBlock) void k_sell_resid(
  SellView A, const T* __restrict__ va, const T* __restrict__ x, const T* __restrict__ b,
  T* __restrict__ r, int n)
{
  const SellLane l = sell_lane<G>(A.stretch);
  if (sell_idle<G>(l, n)) return;
  const T s = sell_dot<T, G>(A, va, x, l, n);
  if (l.row < n && l.g == 0) r[l.row] = b[l.row] - s;
}

// out[p] = T(a[slot[p]] * (colscale ? colscale[ci[p]] : 1)), 0 for padding
template <typename T>
__global__ void k_sell_values(const int32_t* __restrict__ slot,
                              const int32_t* __restrict__ ci,
                              const double* __restrict__ a,
                              const double* __restrict__ colscale,
                              T* __restrict__ out, int64_t len)
{
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= len) return;
  const int32_t k = slot[p];
  out[p] = k < 0 ? (T)0 : (T)(colscale ? a[k] * colscale[ci[p]] : a[k]);
}

// Builds the sliced ELL structure of the CSR graph (rp, ci; device arrays)
// with n rows into s, which must be new or left by a failed build (its
// arrays are released first).  Padding positions read the row's own index as column
// (square matrices), or with pad_last the row's last column, which keeps
// them inside the columns of a rectangular matrix.  With offsets (square
// matrices only) the slices that qualify are stored in offset form; the
// others whose columns span less than 65536 get 16-bit ones.
int sell_build(const int32_t* rp, const int32_t* ci, int n, Sell& s,
               hipStream_t st, bool pad_last = false, bool offsets = false);
void sell_free(Sell& s);

inline SellView sell_view(const Sell& s)
{
  return {s.sp, s.ci, s.dia_w, s.dia_off, s.base, s.cd, 2 * s.dia_slices > s.nslices};
}

// launch helper: dispatch a G-templated row kernel by lanes-per-row
// (kernel<T, G>; NW_ROW_LAUNCH_ADD: kernel<T, G, true>)
#define NW_ROW_LAUNCH_ADD(kernel, T, G, n, stream, ...)                      \
  do {                                                                       \
    const unsigned nw_blocks_ = grid_for((int64_t)(n) * (G), kBlock);        \
    switch (G) {                                                             \
    case 1:                                                                  \
      kernel<T, 1, true><<<nw_blocks_, kBlock, 0, stream>>>(__VA_ARGS__);    \
      break;                                                                 \
    case 2:                                                                  \
      kernel<T, 2, true><<<nw_blocks_, kBlock, 0, stream>>>(__VA_ARGS__);    \
      break;                                                                 \
    case 4:                                                                  \
      kernel<T, 4, true><<<nw_blocks_, kBlock, 0, stream>>>(__VA_ARGS__);    \
      break;                                                                 \
    case 8:                                                                  \
      kernel<T, 8, true><<<nw_blocks_, kBlock, 0, stream>>>(__VA_ARGS__);    \
      break;                                                                 \
    case 16:                                                                 \
      kernel<T, 16, true><<<nw_blocks_, kBlock, 0, stream>>>(__VA_ARGS__);   \
      break;                                                                 \
    case 32:                                                                 \
      kernel<T, 32, true><<<nw_blocks_, kBlock, 0, stream>>>(__VA_ARGS__);   \
      break;                                                                 \
    default:                                                                 \
      kernel<T, 64, true><<<nw_blocks_, kBlock, 0, stream>>>(__VA_ARGS__);   \
    }                                                                        \
  } while (0)

// kernel<T, G> or kernel<T, G, true> of the sliced ELL kernels
#define NW_SELL_LAUNCH(kernel, T, G, n, stream, ...)                         \
  do {                                                                       \
    const unsigned nw_blocks_ = grid_for((int64_t)(n) * (G), kBlock);        \
    if ((G) == 1)                                                            \
      kernel<T, 1><<<nw_blocks_, kBlock, 0, stream>>>(__VA_ARGS__);          \
    else                                                                     \
      kernel<T, 2><<<nw_blocks_, kBlock, 0, stream>>>(__VA_ARGS__);          \
  } while (0)
#define NW_SELL_LAUNCH_ADD(kernel, T, G, n, stream, ...)                     \
  do {                                                                       \
    const unsigned nw_blocks_ = grid_for((int64_t)(n) * (G), kBlock);        \
    if ((G) == 1)                                                            \
      kernel<T, 1, true><<<nw_blocks_, kBlock, 0, stream>>>(__VA_ARGS__);    \
    else                                                                     \
      kernel<T, 2, true><<<nw_blocks_, kBlock, 0, stream>>>(__VA_ARGS__);    \
  } while (0)

#define NW_ROW_LAUNCH(kernel, T, G, n, stream, ...)                          \
  do {                                                                       \
    const unsigned nw_blocks_ = grid_for((int64_t)(n) * (G), kBlock);        \
    switch (G) {                                                             \
    case 1:                                                                  \
      kernel<T, 1><<<nw_blocks_, kBlock, 0, stream>>>(__VA_ARGS__);          \
      break;                                                                 \
    case 2:                                                                  \
      kernel<T, 2><<<nw_blocks_, kBlock, 0, stream>>>(__VA_ARGS__);          \
      break;                                                                 \
    case 4:                                                                  \
      kernel<T, 4><<<nw_blocks_, kBlock, 0, stream>>>(__VA_ARGS__);          \
      break;                                                                 \
    case 8:                                                                  \
      kernel<T, 8><<<nw_blocks_, kBlock, 0, stream>>>(__VA_ARGS__);          \
      break;                                                                 \
    case 16:                                                                 \
      kernel<T, 16><<<nw_blocks_, kBlock, 0, stream>>>(__VA_ARGS__);         \
      break;                                                                 \
    case 32:                                                                 \
      kernel<T, 32><<<nw_blocks_, kBlock, 0, stream>>>(__VA_ARGS__);         \
      break;                                                                 \
    default:                                                                 \
      kernel<T, 64><<<nw_blocks_, kBlock, 0, stream>>>(__VA_ARGS__);         \
    }                                                                        \
  } while (0)

}  // namespace nw
