// ipf_split.h -- launchers of the element / node launches (ipf_split.hip).
#pragma once

#include <cstdint>

#include "ipf_kernels.h"
#include "ipf_learned.h"

namespace ipf {

constexpr int kSplitColors = 8;  // colors (and so groups of one shape) at most

// One element launch: the tiles of one shape, every color.  Segment c is the
// shape's group of one color, `count` tiles; launch tile t is tile t / nseg of
// segment t mod nseg while every segment has one (t < even nseg), then what is
// left segment by segment.  Neighbouring elements of different colors so run
// side by side on one XCD, whose L2 holds the lines they share -- u, and rows
// of per-point values in the reference order -- and a tile's addresses follow
// from its number without a load.
struct SplitDev {
    int nseg;
    int even;                     // the smallest segment's tiles
    unsigned magic;               // ceil(2^32 / nseg): t / nseg = mulhi(t, magic) for t < 2^29
    int count[kSplitColors];
    int tile0[kSplitColors];      // context tile (tmeta)
    int pt0[kSplitColors];        // new point
    int slot0[kSplitColors];      // element slot (corners)
    int ent0[kSplitColors];       // node entry (node, ef)
    int64_t val0[kSplitColors];   // value of the compact FP64 B
    const int* tmeta;
    int64_t ntiles;
    const void* B;         // FMT_G64 / FMT_G32: 8 corner values per element slot; FMT_C64: the values
    const double* tab;     // shape table of the shape
    const int* node;       // x DoF per element slot and node
    const MatConst* mats;
};

// What an element launch does (ipf_split.hip, k_elem).
enum ElemOp {
    EL_RESIDUAL = 0,   // u -> ef
    EL_CERTIFIED = 1,  // the same, certified elastic points by their trial stress
    EL_TANGENT = 2,    // u, dep -> ef of K u
    EL_CG = 3,         // z, p, dep -> ef of K (z + beta p)
    EL_DEP = 4,        // u -> ef, dep
    EL_STRAIN = 5,     // u -> point (strains)
    EL_FORCE = 6,      // point (w sigma) -> ef
    EL_FEATURES = 7    // u -> feat, label, target
};

// z + beta p as a CG iteration gathers it (ipf_kernels.h).
struct CgBeta {
    const double* p;
    const double* rz_old;
    const double* rz_partial;
    int nrz;
};

struct ElemArgs {
    const double* u;
    PointState st;
    double* dep;          // w Dep, SoA, npad apart
    const float* dep32;   // its FP32 copy (FMT_G32)
    int64_t npad;
    CgBeta cg;
    double* ef;           // two doubles per node entry: the element's force on its node
    double* point;        // 3 per point, reference order
    const int64_t* orig;  // reference point of each new point
    float* feat;
    int* label;
    float* target;
};

// fmt: FMT_G64 or FMT_C64; FMT_G32 for the residuals and the products.
void launch_elem(int op, int fmt, int shape, const SplitDev& g, const ElemArgs& a, hipStream_t stream);

// The return map of one shape's points: strains to w sigma and (wdep set)
// w Dep, reference order.  Needs tile0, pt0, tmeta and mats of g only.
void launch_stress(int shape, const SplitDev& g, const double* strain, double* wsigma, double* wdep,
                   const int64_t* orig, const PointState& st, bool commit, hipStream_t stream);

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
