// nw_geom.h -- element geometry shared by the host mesh producers and the
// host setup of the device geometry.
#pragma once

#include <cstdint>
#include <vector>

namespace nw {
namespace geom {

// Area vectors of the 12 Hex8 sub-control surfaces, SCS order of
// HexSCS::determinant_scs (src/master_element/Hex8CVFEM.C:567-591).
void hex_scs(const double c[8][3], double a[12][3]);

// Nodes and sub-control surfaces of topology t (0 Hex8, 1 Tet4, 2 Wed6,
// 3 Pyr5).
int topo_nodes(int t);
int topo_scs(int t);

// Incidence lists of a mesh of nelem elements (type [nelem], NULL = all
// Hex8; conn [nelem][8], unused slots -1) over its nedge edges
// (edges [nedge][2]): for edge e, e_inc[e_ptr[e] .. e_ptr[e+1]) holds
// 2 (12 el + s) + flip for every sub-control surface s of element el on
// that edge, in element order, flip = 1 when the surface's L node is the
// edge's node[1]; for node n, n_inc[n_ptr[n] .. n_ptr[n+1]) holds 8 el + a
// for every element el whose local node a it is, in element order.
// Returns NW_E_ARG for bad input, an element edge missing from the edge
// list or more than 2^26 elements.
int build_incidence(int64_t nelem, const int32_t* type, const int32_t* conn,
                    int64_t nnode, int64_t nedge, const int32_t* edges,
                    std::vector<int32_t>& e_ptr, std::vector<int32_t>& e_inc,
                    std::vector<int32_t>& n_ptr, std::vector<int32_t>& n_inc);

// The elements of one topology: `n` of them from position `first` of the
// grouped order.  Their SCS scratch is a plane of n area vectors per surface
// (surface s of the i-th: record scs + s n + i of 24 bytes), their SCV
// scratch a plane of n values per sub-volume (value scv + a n + i), or the
// one plane that all four sub-volumes of a tetrahedron share.
struct ElemGroup {
  int64_t first = 0, n = 0, scs = 0, scv = 0;
};
// planes of the SCV scratch
constexpr int scv_stored(int topo)
{
  return topo == 0 ? 8 : topo == 1 ? 1 : topo == 2 ? 6 : 5;
}

// Counts the elements by topology and lays out their scratch; *nscs and
// *nscv: records and values in all.
void layout_elements(int64_t nelem, const int32_t* type, ElemGroup (&grp)[4],
                     int64_t* nscs, int64_t* nscv);
// The connectivity grouped by topology, gconn [nelem][8], and the lists of
// build_incidence turned into scratch indices: e_inc into 2 (SCS record) +
// flip, n_inc into SCV values; the lists keep their order.
void group_elements(int64_t nelem, const int32_t* type, const int32_t* conn,
                    const ElemGroup (&grp)[4], std::vector<int32_t>& gconn,
                    std::vector<int32_t>& e_inc, std::vector<int32_t>& n_inc);

}  // namespace geom
}  // namespace nw
