// ipf_split.h -- launchers of the element / node launches (ipf_split.hip).
#pragma once

#include <cstdint>

#include "ipf_kernels.h"

namespace ipf {

constexpr int kSplitColors = 8;  // colors (and so groups of one shape) at most

// One element launch: the tiles of one shape, every color.  Segment c is the
// shape's group of one color: launch tiles [end[c - 1], end[c]), and where its
// tile 0 would start if the group began at launch tile 0 -- so that a tile's
// addresses follow from its number without a load.
struct SplitDev {
    int nseg;
    int end[kSplitColors];
    int tile0[kSplitColors];   // context tile (tmeta)
    int pt0[kSplitColors];     // new point
    int slot0[kSplitColors];   // element slot (corners)
    int ent0[kSplitColors];    // node entry (node, ef)
    const int* tmeta;
    int64_t ntiles;
    const double* geo;     // 8 corner values per element slot
    const double* tab;     // shape table of the shape
    const int* node;       // x DoF per element slot and node
    const MatConst* mats;
};

// ef[entry] (two doubles) = the element's force on its node, fmt FMT_G64 / FMT_G32
void launch_elem_residual(int fmt, int shape, bool fast, const SplitDev& g, const double* u, const PointState& st,
                          double* ef, hipStream_t stream);
// The residual's element forces and every point's w Dep (FMT_G64).
void launch_elem_dep(int shape, const SplitDev& g, const double* u, const PointState& st, double* dep, int64_t npad,
                     double* ef, hipStream_t stream);
// With rz_old (a CG iteration, see ipf_kernels.h): v is z, and the vector
// multiplied is z + beta p, formed as it is gathered.
struct CgBeta {
    const double* p;
    const double* rz_old;  // null: no CG, the product with v itself
    const double* rz_partial;
    int nrz;
};
void launch_elem_tangent(int fmt, int shape, const SplitDev& g, const double* v, const CgBeta& cg, double* dep,
                         const float* dep32, int64_t npad, double* ef, hipStream_t stream);

// map: stride (4 or 8) ints per node, one per color; filled with -1, then one
// call per group (n0: the group's first node entry)
void launch_fill_int(int64_t n, int* p, int v, hipStream_t stream);
void launch_node_map(int shape, const GroupDev& g, int64_t n0, int color, int stride, int* map, hipStream_t stream);
// out[n] = start - sum of the node's element forces in color order (start null: 0)
void launch_nodes(int64_t n, int stride, const int* map, const double* ef, const double* start, double* out,
                  hipStream_t stream);
// p = z + beta p_old, q = K p from the element forces of that p, 0 where mask
// is set, partial[nb] of p.q, *rz_new = r.z
void launch_nodes_cg(int64_t n, int stride, const int* map, const double* ef, const signed char* mask, const double* z,
                     const CgBeta& cg, double* rz_new, double* p, double* q, double* partial, int nb,
                     hipStream_t stream);

}  // namespace ipf
