// nw_geometry.hip -- GeometryInteriorAlg (src/ngp_algorithms/
// GeometryInteriorAlg.C:70-225) on gfx950: the edge area vectors and dual
// nodal volumes of a Hex8 / Tet4 / Wed6 / Pyr5 mesh from its node
// coordinates.
//
//   k_elements     one lane per element: its sub-control-surface (SCS) area
//                  vectors and sub-control volumes (SCV) into two scratch
//                  buffers; the elements are grouped by type (the mesh's
//                  order within a type), so that a block has one topology;
//   k_edge_area    one lane per edge: sums +-SCS over the edge's surfaces in
//                  element order, + when the surface's L node is the edge's
//                  node[0] (GeometryInteriorAlg.C:209-219);
//   k_dual_volume  one lane per node: sums its SCVs in element order.
// The reference adds element contributions into the edge and node fields
// with atomics; here the incidence lists built once per mesh fix the order
// of every sum, so the result is reproducible: the area vectors are the
// same sums, in the same order, as the host producers in host/nw_mesh.cpp
// and nw_mixed.cpp, and the volumes agree with them to rounding (they are
// taken in element-centred coordinates here).
//
// Each SCS is a quad of four points of the subdivided element and its area
// vector is half the cross product of its diagonals (a Pyr5 surface next to
// the apex is a triangle: a quad with a repeated point);
// each SCV is a hexahedron of eight such points whose volume is Grandy's
// (hex_volume_grandy, include/master_element/Hex8GeometryFunctions.h:85:
// each face as four triangles about its centroid),
// except in Pyr5: bent hexahedra at the base nodes (bhex_volume_grandy,
// :163) and an octahedron at the apex (src/master_element/Pyr5CVFEM.C:
// 395-433).  A point is the average of a set of element vertices.
#include <algorithm>
#include <vector>

#include "nw_geom.h"
#include "nw_internal.h"

namespace nw {

namespace {

// Points of the subdivided element as {count, vertices...}: corners first.
// Hex8 (include/master_element/Hex8GeometryFunctions.h:258-330): edge
// midpoints, face centroids face by face, centroid.
struct HexTopo {
  static constexpr int kNodes = 8, kScs = 12;
  static constexpr int8_t pts[27][9] = {
    {1, 0},          {1, 1},          {1, 2},          {1, 3},
    {1, 4},          {1, 5},          {1, 6},          {1, 7},
    {2, 0, 1},       {2, 1, 2},       {2, 2, 3},       {2, 3, 0},
    {4, 0, 1, 2, 3}, {2, 4, 5},       {2, 5, 6},       {2, 6, 7},
    {2, 7, 4},       {4, 4, 5, 6, 7}, {2, 1, 5},       {2, 0, 4},
    {4, 0, 1, 4, 5}, {2, 3, 7},       {2, 2, 6},       {4, 2, 3, 6, 7},
    {4, 1, 2, 5, 6}, {4, 0, 3, 4, 7}, {8, 0, 1, 2, 3, 4, 5, 6, 7}};
  // HexSCS::determinant_scs (src/master_element/Hex8CVFEM.C:567-591)
  static constexpr int8_t quad[12][4] = {
    {20, 8, 12, 26},  {24, 9, 12, 26},  {10, 12, 26, 23}, {11, 25, 26, 12},
    {13, 20, 26, 17}, {17, 14, 24, 26}, {17, 15, 23, 26}, {16, 17, 26, 25},
    {19, 20, 26, 25}, {20, 18, 24, 26}, {22, 23, 26, 24}, {21, 25, 26, 23}};
  // The sub-hexahedron about each corner (HexSCV::determinant_scv,
  // src/master_element/Hex8CVFEM.C:365-389), seen from it: its three edges'
  // midpoints m0, m1, m2 (right-handed) and the centroids of the element's
  // faces between them, F01, F12, F20; the seventh and eighth points are the
  // corner and the element's centroid.
  static constexpr int8_t octant[8][6] = {
    {8, 11, 19, 12, 25, 20}, {9, 8, 18, 12, 20, 24}, {10, 9, 22, 12, 24, 23},
    {11, 10, 21, 12, 23, 25}, {16, 13, 19, 17, 20, 25}, {13, 14, 18, 17, 24, 20},
    {14, 15, 22, 17, 23, 24}, {15, 16, 21, 17, 25, 23}};
};

// Tet4 (src/master_element/Tet4CVFEM.C:243-343, 522-618)
struct TetTopo {
  static constexpr int kNodes = 4, kScs = 6;
  static constexpr int8_t pts[15][9] = {
    {1, 0},       {1, 1},       {1, 2},          {1, 3},       {2, 0, 1},
    {2, 1, 2},    {2, 2, 0},    {3, 0, 1, 2},    {2, 2, 3},    {2, 3, 1},
    {3, 1, 2, 3}, {2, 0, 3},    {3, 0, 2, 3},    {3, 0, 1, 3}, {4, 0, 1, 2, 3}};
  static constexpr int8_t quad[6][4] = {{4, 7, 14, 13}, {7, 14, 10, 5},
                                        {6, 12, 14, 7}, {11, 13, 14, 12},
                                        {13, 9, 10, 14}, {10, 8, 12, 14}};
};

// Wed6 (src/master_element/Wed6CVFEM.C:267-369, 541-646)
struct WedTopo {
  static constexpr int kNodes = 6, kScs = 9;
  static constexpr int8_t pts[21][9] = {
    {1, 0},          {1, 1},          {1, 2},       {1, 3},
    {1, 4},          {1, 5},          {2, 0, 1},    {2, 1, 2},
    {2, 2, 0},       {3, 0, 1, 2},    {2, 3, 4},    {2, 4, 5},
    {2, 5, 3},       {3, 3, 4, 5},    {2, 1, 4},    {2, 0, 3},
    {4, 0, 1, 4, 3}, {2, 2, 5},       {4, 1, 4, 5, 2},
    {4, 5, 3, 0, 2}, {6, 0, 1, 2, 3, 4, 5}};
  static constexpr int8_t quad[9][4] = {
    {6, 9, 20, 16},   {7, 9, 20, 18},   {9, 8, 19, 20},
    {10, 16, 20, 13}, {13, 11, 18, 20}, {12, 13, 20, 19},
    {15, 16, 20, 19}, {16, 14, 18, 20}, {19, 20, 18, 17}};
  static constexpr int8_t scv[6][8] = {
    {0, 15, 16, 6, 8, 19, 20, 9},    {9, 6, 1, 7, 20, 16, 14, 18},
    {8, 9, 7, 2, 19, 20, 18, 17},    {19, 15, 16, 20, 12, 3, 10, 13},
    {20, 16, 14, 18, 13, 10, 4, 11}, {19, 20, 18, 17, 12, 13, 11, 5}};
};

// Pyr5 (src/master_element/Pyr5CVFEM.C:437-571, 771-900): base edge
// midpoints, base centroid, apex edge midpoints and triangle centroids,
// element centroid.
struct PyrTopo {
  static constexpr int kNodes = 5, kScs = 12;
  static constexpr int8_t pts[19][9] = {
    {1, 0},       {1, 1},       {1, 2},          {1, 3},       {1, 4},
    {2, 0, 1},    {2, 1, 2},    {2, 2, 3},       {2, 3, 0},    {4, 0, 1, 2, 3},
    {2, 1, 4},    {2, 4, 0},    {3, 0, 1, 4},    {2, 2, 4},    {3, 1, 2, 4},
    {2, 3, 4},    {3, 3, 4, 2}, {3, 0, 4, 3},    {5, 0, 1, 2, 3, 4}};
  static constexpr int8_t quad[12][4] = {
    {5, 9, 18, 12},   {6, 9, 18, 14},   {7, 9, 18, 16},   {8, 17, 18, 9},
    {12, 12, 18, 17}, {11, 12, 12, 17}, {14, 14, 18, 12}, {10, 14, 14, 12},
    {16, 16, 18, 14}, {13, 16, 16, 14}, {17, 17, 18, 16}, {15, 17, 17, 16}};
  // base sub-volumes (bent hexahedra, top face split along 5-7), then the
  // apex octahedron's ten vertices
  static constexpr int8_t scv[4][8] = {{0, 5, 9, 8, 11, 12, 18, 17},
                                       {1, 6, 9, 5, 10, 14, 18, 12},
                                       {2, 7, 9, 6, 13, 16, 18, 14},
                                       {3, 8, 9, 7, 15, 17, 18, 16}};
  static constexpr int8_t apex[10] = {4, 18, 15, 17, 11, 12, 10, 14, 13, 16};
};

// Area vector of the quad (q0, q1, q2, q3): half the cross product of its
// diagonals, the sum over its four triangles about any point.
__device__ inline void quad_area(const double (&q)[4][3], double* a)
{
  double u[3], v[3];
  for (int d = 0; d < 3; ++d) {
    u[d] = q[2][d] - q[0][d];
    v[d] = 0.5 * (q[3][d] - q[1][d]);
  }
  a[0] = u[1] * v[2] - v[1] * u[2];
  a[1] = u[2] * v[0] - v[2] * u[0];
  a[2] = u[0] * v[1] - v[0] * u[1];
}

__device__ inline double det3(const double* a, const double* b, const double* c)
{
  return (a[1] * b[2] - b[1] * a[2]) * c[0] + (a[2] * b[0] - b[2] * a[0]) * c[1] +
         (a[0] * b[1] - b[0] * a[1]) * c[2];
}

// 12 times the flux of x/3 through the quad (a, b, c, d) taken as four
// triangles about its centroid m.  The flux of the four triangles (a, b, m)
// ... (d, a, m) is linear in m, and with m at a or c (b or d) they are the
// two triangles of a split along ac (bd): at the centroid the flux is the
// mean of the two splits',
//   [(a x b).(c + d) + (c x d).(a + b)] / 12,
// a quarter of the operations of the four triangles.
__device__ inline double quad_flux12(const double* a, const double* b, const double* c,
                                     const double* d)
{
  const double cd[3] = {c[0] + d[0], c[1] + d[1], c[2] + d[2]};
  const double ab[3] = {a[0] + b[0], a[1] + b[1], a[2] + b[2]};
  return det3(a, b, cd) + det3(c, d, ab);
}

// Faces of a hexahedron (exodus order), outward.
__device__ constexpr int8_t kHexFace[6][4] = {{0, 3, 2, 1}, {4, 5, 6, 7}, {0, 1, 5, 4},
                                              {7, 6, 2, 3}, {1, 2, 6, 5}, {0, 4, 7, 3}};

// Volume of the hexahedron h by the divergence theorem over its faces'
// centroid triangles (Grandy 1997); BENT: the top face is the two triangles
// on either side of its 5-7 diagonal, the Pyr5 base sub-volumes.
template <bool BENT>
__device__ inline double grandy_volume(const double (&h)[8][3])
{
  double v = 0.0;
#pragma unroll
  for (int f = 0; f < 6; ++f) {
    const double *a = h[kHexFace[f][0]], *b = h[kHexFace[f][1]], *c = h[kHexFace[f][2]],
                 *d = h[kHexFace[f][3]];
    if (BENT && f == 1)
      v += 2.0 * (det3(a, b, d) + det3(b, c, d));
    else
      v += quad_flux12(a, b, c, d);
  }
  return v * (1.0 / 12.0);
}

// Volume of the Pyr5 apex sub-volume from its ten vertices o (apex,
// element centroid, then around the apex: edge midpoint, triangle centroid,
// ...): its four bent faces are split at the midpoints of o3-o9, o3-o5,
// o5-o7, o7-o9 (points 10-13) into the 24 triangles below.
__device__ inline double octahedron_volume(const double (&o)[10][3])
{
  constexpr int8_t tri[24][3] = {
    {1, 3, 10}, {2, 10, 3}, {2, 9, 10}, {10, 9, 1}, {4, 3, 11}, {3, 1, 11},
    {11, 1, 5}, {4, 11, 5}, {1, 12, 5}, {1, 7, 12}, {12, 7, 6}, {5, 12, 6},
    {9, 8, 13}, {13, 8, 7}, {13, 7, 1}, {9, 13, 1}, {4, 5, 0},  {5, 6, 0},
    {6, 7, 0},  {7, 8, 0},  {0, 8, 9},  {0, 9, 2},  {0, 2, 3},  {0, 3, 4}};
  constexpr int8_t mid[4][2] = {{3, 9}, {3, 5}, {5, 7}, {7, 9}};
  double p[14][3];
#pragma unroll
  for (int n = 0; n < 10; ++n)
    for (int d = 0; d < 3; ++d) p[n][d] = o[n][d];
#pragma unroll
  for (int k = 0; k < 4; ++k)
    for (int d = 0; d < 3; ++d) p[10 + k][d] = 0.5 * (o[mid[k][0]][d] + o[mid[k][1]][d]);
  double v = 0.0;
#pragma unroll
  for (int t = 0; t < 24; ++t) v += det3(p[tri[t][0]], p[tri[t][1]], p[tri[t][2]]);
  return v * (1.0 / 6.0);
}

// Point k of the subdivided element of topology T from its corners c; with
// CENTRED the corners' mean is the origin, which the last point then is.
template <class T, bool CENTRED>
__device__ inline void sub_point(const double (&c)[T::kNodes][3], int k,
                                 double (&p)[3])
{
  const int cnt = T::pts[k][0];
  for (int d = 0; d < 3; ++d) {
    double s = 0.0;
#pragma unroll
    for (int i = 1; i <= 8; ++i)
      if (i <= cnt) s += c[T::pts[k][i]][d];
    p[d] = CENTRED && cnt == T::kNodes ? 0.0 : s * (1.0 / cnt);
  }
}

// Makes the compiler forget what it knows of the corners, so that it forms
// the points of the next surfaces or volumes anew from the corners (a few
// adds) instead of keeping all of them in registers (256 and spills, against 162
// and none: three waves per SIMD).
template <int N>
__device__ inline void forget(double (&c)[N][3])
{
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int a = 0; a < N; ++a)
    for (int d = 0; d < 3; ++d) asm volatile("" : "+v"(c[a][d]));
  __builtin_amdgcn_sched_barrier(0);
}

// Writes a wave's area vectors v[s][3] of NS surfaces to NS planes of 24-byte
// records, `rows` records each, through LDS: every plane one contiguous
// range.
template <int NS>
__device__ inline void put_areas(const double (&v)[NS][3], int lane, int rows,
                                 double* __restrict__ sh, double* __restrict__ dst,
                                 int64_t plane)
{
  wave_lds_sync();  // the records before these have been read
#pragma unroll
  for (int s = 0; s < NS; ++s)
    for (int d = 0; d < 3; ++d) sh[(s * kWave + lane) * 3 + d] = v[s][d];
  wave_lds_sync();
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const int i = lane + k * kWave;
      if (i < 3 * rows) dst[s * plane + i] = sh[s * kWave * 3 + i];
    }
}

constexpr int kScsStaged = 3;  // surfaces staged in LDS together

// SCS area vectors and SCV volumes of one wave's elements of topology T.
template <class T, int TOPO>
__device__ inline void elements(const geom::ElemGroup& g, int64_t row0, int lane,
                                const int32_t* __restrict__ conn,
                                const double* __restrict__ coords,
                                double* __restrict__ scs, double* __restrict__ scv,
                                double* __restrict__ sh)
{
  const int rows = (int)min((int64_t)kWave, g.n - row0);
  const int64_t row = row0 + min(lane, rows - 1);  // lanes past the end repeat the last
  double c[T::kNodes][3];
  const int4* cn = reinterpret_cast<const int4*>(conn + 8 * (g.first + row));
  const int4 n0 = cn[0], n1 = T::kNodes > 4 ? cn[1] : make_int4(0, 0, 0, 0);
  const int nd[8] = {n0.x, n0.y, n0.z, n0.w, n1.x, n1.y, n1.z, n1.w};
#pragma unroll
  for (int a = 0; a < T::kNodes; ++a)
    for (int d = 0; d < 3; ++d) c[a][d] = coords[3 * (int64_t)nd[a] + d];
#pragma unroll
  for (int s0 = 0; s0 < T::kScs; s0 += kScsStaged) {
    forget(c);
    double v[kScsStaged][3];
#pragma unroll
    for (int s = 0; s < kScsStaged; ++s) {
      double q[4][3];
#pragma unroll
      for (int i = 0; i < 4; ++i) sub_point<T, false>(c, T::quad[s0 + s][i], q[i]);
      quad_area(q, v[s]);
    }
    put_areas<kScsStaged>(v, lane, rows, sh, scs + 3 * (g.scs + s0 * g.n + row0), 3 * g.n);
  }
  // the volumes do not depend on the origin: taking it at the element's
  // centroid keeps the face fluxes near the size of the volumes (absolute
  // coordinates make them larger by the distance to the origin over the
  // element's size, and the volumes lose that many digits to cancellation)
  for (int d = 0; d < 3; ++d) {
    double o = 0.0;
#pragma unroll
    for (int a = 0; a < T::kNodes; ++a) o += c[a][d];
    o *= 1.0 / T::kNodes;
#pragma unroll
    for (int a = 0; a < T::kNodes; ++a) c[a][d] -= o;
  }
  // every volume is stored where it is formed (lanes past the end store the
  // last element's again)
  constexpr int NV = geom::scv_stored(TOPO);
  double* vol = scv + g.scv + row;
  if constexpr (TOPO == 0) {
    // twelve times the flux out of the three quarter faces at the corner and
    // the three faces that meet at the element's centroid, the origin (a quad
    // with a corner there has the flux of one triangle)
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      forget(c);
      double m[3][3], F[3][3];
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        sub_point<T, true>(c, T::octant[v][i], m[i]);
        sub_point<T, true>(c, T::octant[v][3 + i], F[i]);
      }
      double phi = 0.0;
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const int j = (i + 1) % 3, k = (i + 2) % 3;
        phi += quad_flux12(c[v], m[j], F[i], m[i]) + det3(m[i], F[i], F[k]);
      }
      vol[v * g.n] = phi * (1.0 / 12.0);
    }
  } else if constexpr (TOPO == 1) {
    // the median planes cut a tetrahedron into four equal parts
    double e[3][3];
    for (int a = 0; a < 3; ++a)
      for (int d = 0; d < 3; ++d) e[a][d] = c[a + 1][d] - c[0][d];
    vol[0] = det3(e[0], e[1], e[2]) * (1.0 / 24.0);
  } else {
    constexpr bool kPyr = TOPO == 3;
#pragma unroll
    for (int v = 0; v < (kPyr ? 4 : NV); ++v) {
      forget(c);
      double h[8][3];
#pragma unroll
      for (int i = 0; i < 8; ++i) sub_point<T, true>(c, T::scv[v][i], h[i]);
      vol[v * g.n] = grandy_volume<kPyr>(h);
    }
    if constexpr (kPyr) {
      forget(c);
      double o[10][3];
#pragma unroll
      for (int i = 0; i < 10; ++i) sub_point<T, true>(c, T::apex[i], o[i]);
      vol[4 * g.n] = octahedron_volume(o);
    }
  }
}

// One lane per element, blocks of one topology.
//
// Bound by the scratch it writes (352 bytes per Hex8).  The kernels it
// replaces, one for the surfaces and one for the volumes, with every value
// in a plane of its own and four triangles per sub-face, took 535 us for
// 2.1 M Hex8 (volumes 394 us, bound by FP64 arithmetic) and 574 us for the
// 0.74 M mixed elements of a 64^3 box, whose waves ran every topology of
// their lanes in turn.
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(3))) void k_elements(
  ElemGroups G, const int32_t* __restrict__ conn, const double* __restrict__ coords,
  double* __restrict__ scs, double* __restrict__ scv)
{
  __shared__ double sh[kBlock / kWave][kWave * 3 * kScsStaged];
  const int lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave;
  const int b = blockIdx.x;
  const int t = b >= G.first_block[3] ? 3 : b >= G.first_block[2] ? 2 : b >= G.first_block[1] ? 1 : 0;
  const geom::ElemGroup& g = G.g[t];
  const int64_t row0 = (int64_t)(b - G.first_block[t]) * kBlock + wv * kWave;
  if (row0 >= g.n) return;
  if (t == 0)
    elements<HexTopo, 0>(g, row0, lane, conn, coords, scs, scv, sh[wv]);
  else if (t == 1)
    elements<TetTopo, 1>(g, row0, lane, conn, coords, scs, scv, sh[wv]);
  else if (t == 2)
    elements<WedTopo, 2>(g, row0, lane, conn, coords, scs, scv, sh[wv]);
  else
    elements<PyrTopo, 3>(g, row0, lane, conn, coords, scs, scv, sh[wv]);
}

// areav[3 e + d] = sum over the edge's surfaces (element order) of
// +-scs[3 i + d], i the surface's record: e_inc = 2 i + flip.  Four
// surfaces' loads are in flight at a time; blocks in XCD-aware order, so that
// the records of neighbouring edges' elements are shared in one L2.
__global__ __launch_bounds__(kBlock) void k_edge_area(
  int64_t E, const int32_t* __restrict__ e_ptr, const int32_t* __restrict__ e_inc,
  const double* __restrict__ scs, double* __restrict__ areav)
{
  constexpr int U = 4;
  const int64_t e = (int64_t)xcd_block((int)gridDim.x) * kBlock + threadIdx.x;
  if (e >= E) return;
  double a[3] = {0.0, 0.0, 0.0};
  const int k1 = e_ptr[e + 1];
  for (int k = e_ptr[e]; k < k1; k += U) {
    int32_t c[U];
    double v[U][3];
#pragma unroll
    for (int u = 0; u < U; ++u) c[u] = k + u < k1 ? e_inc[k + u] : -1;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (c[u] >= 0)
        for (int d = 0; d < 3; ++d) v[u][d] = scs[3 * (int64_t)(c[u] >> 1) + d];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (c[u] >= 0) {
        const double sgn = (c[u] & 1) ? -1.0 : 1.0;
        for (int d = 0; d < 3; ++d) a[d] += v[u][d] * sgn;
      }
  }
  for (int d = 0; d < 3; ++d) areav[3 * e + d] = a[d];
}

// dualvol[n] = sum over the node's elements (element order) of its SCV,
// scv[n_inc]
__global__ __launch_bounds__(kBlock) void k_dual_volume(
  int64_t N, const int32_t* __restrict__ n_ptr, const int32_t* __restrict__ n_inc,
  const double* __restrict__ scv, double* __restrict__ dualvol)
{
  constexpr int U = 8;
  const int64_t n = (int64_t)xcd_block((int)gridDim.x) * kBlock + threadIdx.x;
  if (n >= N) return;
  double s = 0.0;
  const int k1 = n_ptr[n + 1];
  for (int k = n_ptr[n]; k < k1; k += U) {
    int32_t c[U];
    double v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) c[u] = k + u < k1 ? n_inc[k + u] : -1;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (c[u] >= 0) v[u] = scv[c[u]];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (c[u] >= 0) s += v[u];
  }
  dualvol[n] = s;
}

}  // namespace

void geom_free(Geom* g)
{
  if (!g) return;
  (void)hipFree(g->conn);
  (void)hipFree(g->e_ptr);
  (void)hipFree(g->e_inc);
  (void)hipFree(g->n_ptr);
  (void)hipFree(g->n_inc);
  (void)hipFree(g->scs);
  (void)hipFree(g->scv);
  delete g;
}

}  // namespace nw

using namespace nw;

namespace {

template <class T>
int upload(T** dst, const T* src, int64_t n, hipStream_t s)
{
  NW_HIP(hipMalloc(dst, sizeof(T) * std::max<int64_t>(n, 1)));
  NW_HIP(hipMemcpyAsync(*dst, src, sizeof(T) * n, hipMemcpyHostToDevice, s));
  return NW_OK;
}

}  // namespace

extern "C" {

int nw_mesh_elements(nw_ctx* c, int64_t nelem, const int32_t* type,
                     const int32_t* conn)
{
  NW_REQUIRE(c && nelem >= 0 && (conn || nelem == 0), NW_E_ARG, "bad element arguments");
  NW_REQUIRE(c->nnode > 0 && c->nedge >= 0, NW_E_STATE, "mesh not set");
  std::vector<int32_t> e_ptr, e_inc, n_ptr, n_inc;
  const int rc = geom::build_incidence(nelem, type, conn, c->nnode, c->nedge,
                                       c->h_edges.data(), e_ptr, e_inc, n_ptr,
                                       n_inc);
  NW_REQUIRE(rc == NW_OK, NW_E_ARG,
             "bad elements (type or node out of range, an element edge not in "
             "the edge list, or more than 2^26 elements)");
  NW_HIP(hipSetDevice(c->device));
  NW_HIP(hipStreamSynchronize(c->stream));
  geom_free(c->geom);
  c->geom = new Geom;
  Geom* g = c->geom;
  g->nelem = nelem;
  // the elements grouped by type, in mesh order within a type
  geom::ElemGroup(&grp)[4] = g->groups.g;
  int64_t nscs = 0, nscv = 0;
  geom::layout_elements(nelem, type, grp, &nscs, &nscv);
  for (int t = 0; t < 4; ++t)
    g->groups.first_block[t + 1] =
      g->groups.first_block[t] + (int)((grp[t].n + kBlock - 1) / kBlock);
  std::vector<int32_t> gconn;
  geom::group_elements(nelem, type, conn, grp, gconn, e_inc, n_inc);
  int r = 0;
  if ((r = upload(&g->conn, gconn.data(), 8 * nelem, c->stream)) ||
      (r = upload(&g->e_ptr, e_ptr.data(), (int64_t)e_ptr.size(), c->stream)) ||
      (r = upload(&g->e_inc, e_inc.data(), (int64_t)e_inc.size(), c->stream)) ||
      (r = upload(&g->n_ptr, n_ptr.data(), (int64_t)n_ptr.size(), c->stream)) ||
      (r = upload(&g->n_inc, n_inc.data(), (int64_t)n_inc.size(), c->stream)))
    return r;
  NW_HIP(hipMalloc(&g->scs, sizeof(double) * 3 * std::max<int64_t>(nscs, 1)));
  NW_HIP(hipMalloc(&g->scv, sizeof(double) * std::max<int64_t>(nscv, 1)));
  NW_HIP(hipStreamSynchronize(c->stream));
  return NW_OK;
}

int nw_compute_geometry(nw_ctx* c)
{
  NW_REQUIRE(c, NW_E_ARG, "null context");
  NW_REQUIRE(c->geom, NW_E_STATE, "no elements (nw_mesh_elements)");
  const Geom* g = c->geom;
  const double* coords = nullptr;
  double *areav = nullptr, *dualvol = nullptr;
  int rc = 0;
  if ((rc = require_field(c, NW_F_COORDINATES, &coords)) ||
      (rc = ensure_field(c, NW_E_AREA_VECTOR, &areav)) ||
      (rc = ensure_field(c, NW_F_DUAL_VOLUME, &dualvol)))
    return rc;
  const auto padded = [](int64_t n) { return (grid_for(n, kBlock) + 7) / 8 * 8; };
  if (g->nelem > 0)
    k_elements<<<g->groups.first_block[4], kBlock, 0, c->stream>>>(g->groups, g->conn, coords,
                                                                  g->scs, g->scv);
  if (c->nedge > 0)
    k_edge_area<<<padded(c->nedge), kBlock, 0, c->stream>>>(c->nedge, g->e_ptr, g->e_inc,
                                                            g->scs, areav);
  k_dual_volume<<<padded(c->nnode), kBlock, 0, c->stream>>>(c->nnode, g->n_ptr, g->n_inc,
                                                            g->scv, dualvol);
  NW_LAUNCH_CHECK();
  return NW_OK;
}

}  // extern "C"
