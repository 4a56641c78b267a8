// ipf_split.hip -- the residual and the tangent product in two kinds of
// launch: one element launch per shape over the tiles of every color, which
// writes each element's nodal forces to its own place (ef), and one node
// launch that sums each node's elements in color order -- the order, and so
// the bits, of the colored launches (ipf_kernels_fmt.hip).  Two launches
// instead of one per color (and shape); the price is ef, written once and read
// once (16 bytes per element and node), against r read and written once per
// color.  Bound by the launches and each wavefront's chain of round trips on
// small meshes, where it is used (kSplitPoints, ipf_device.hip, with the times
// of both).
#include "ipf_fmt.h"
#include "ipf_split.h"

namespace ipf {

namespace {

// Segment and tile inside it of launch tile t (SplitDev).
struct SplitTile {
    int seg, t;
};

__device__ __forceinline__ SplitTile split_tile(const SplitDev& g, int t) {
    const int q = (int)__umulhi((unsigned)t, g.magic);
    if (q < g.even) return SplitTile{t - q * g.nseg, q};
    int rest = t - g.even * g.nseg, seg = 0;
#pragma unroll
    for (int c = 0; c < kSplitColors - 1; c++)
        if (c == seg && rest >= g.count[c] - g.even) {
            rest -= g.count[c] - g.even;
            seg = c + 1;
        }
    return SplitTile{seg, g.even + rest};
}

// Values of the tile's points, N each, between LDS (point order) and the
// reference order: an element's points are consecutive there, so the
// wavefront reads and writes whole rows of it (lane by lane it would touch
// every row N times).  oel: each element's first reference point.
template <int N, int NIP>
__device__ __forceinline__ void store_points(const double* sh, const int64_t* oel, int nv, double* __restrict__ dst) {
    for (int t = threadIdx.x; t < nv * NIP * N; t += kWave) {
        const int el = t / (NIP * N);
        dst[N * oel[el] + (t - el * NIP * N)] = sh[t];
    }
}

template <int N, int NIP>
__device__ __forceinline__ void load_points(double* sh, const int64_t* oel, int nv, const double* __restrict__ src) {
    for (int t = threadIdx.x; t < nv * NIP * N; t += kWave) {
        const int el = t / (NIP * N);
        sh[t] = src[N * oel[el] + (t - el * NIP * N)];
    }
}

// One wavefront per tile: gather, strain, stress (or w Dep times the strain),
// B^T products and the sums over each element's points, as k_residual_fmt /
// k_tangent_fmt with PAIR; the two sums of node rj of element re leave in one
// 16-byte store, the tile's stores in a row.  Every address follows from the
// tile's number (SplitDev), so the indexes, the state or w Dep, the corners
// and the partials of beta are requested at once and the gather is the second
// and last round trip (a product with w Dep requested after the gather and
// the addresses read from a table: 20x20 Q2 7.8 us, so 6.3).
template <int SHAPE, int FMT, int OP>
__global__ void __launch_bounds__(kWave, (OP == EL_DEP ? (FC<SHAPE, FMT>::CE <= 20 ? 3 : 2) : FC<SHAPE, FMT>::MIN_WAVES))
k_elem(SplitDev g, const double* __restrict__ u, ElemArgs a) {
    using C = FC<SHAPE, FMT>;
    using T = typename C::T;
    constexpr bool CG = OP == EL_CG, TAN = OP == EL_TANGENT || CG, FEAT = OP == EL_FEATURES;
    constexpr bool STRESS = OP == EL_RESIDUAL || OP == EL_CERTIFIED || OP == EL_DEP;
    constexpr bool GATHER = OP != EL_FORCE, FORCES = OP != EL_STRAIN && !FEAT;
    constexpr bool POINTS = OP == EL_STRAIN || OP == EL_FORCE;  // per-point values in the reference order
    const PointState& st = a.st;
    constexpr bool F32 = TAN && FMT == FMT_G32;
    constexpr int NSH = C::CE / 2;
    constexpr int H = 2 * ((NSH + 1) / 2), H2 = C::CE - H;
    constexpr int RS = row_stride(H, sizeof(T)), RS2 = row_stride(H2, sizeof(T));
    constexpr int NE = C::ET * NSH;
    static_assert(NE <= kWave, "one node per lane");
    constexpr bool PARK = OP == EL_DEP && park_B(C::CE);
    constexpr int PS = PARK ? row_stride(C::NV, sizeof(T)) : 0;
    __shared__ T lds[FORCES ? C::TP * (PARK ? PS : RS > RS2 ? RS : RS2) : 1];
    __shared__ double us[GATHER ? 2 * NE : 1];
    __shared__ double pts[POINTS ? 3 * C::TP : 1];
    __shared__ int64_t oel[POINTS ? C::ET : 1];
    const int lane = threadIdx.x;
    const SplitTile at = split_tile(g, (int)xcd_tile(blockIdx.x, gridDim.x));
    const int t = at.t;
    int tile0 = g.tile0[0], pt0 = g.pt0[0], slot0 = g.slot0[0], ent0 = g.ent0[0];
    int64_t val0 = g.val0[0];
#pragma unroll
    for (int c = 1; c < kSplitColors; c++)
        if (c == at.seg) {
            tile0 = g.tile0[c];
            pt0 = g.pt0[c];
            slot0 = g.slot0[c];
            ent0 = g.ent0[c];
            val0 = g.val0[c];
        }
    const int tm = g.tmeta[tile0 + t];
    const int64_t E0 = slot0 + t * C::ET, N0 = ent0 + t * NE;
    const int nv = tm & 255;
    const int el = lane / C::NIP;
    const bool slot = lane < C::TP;
    const bool valid = slot && el < nv;
    // indexes, then the point's state, then the values the indexes address,
    // all outside branches (padding slots hold node DoF 0 and points of their own)
    int d = 0;
    if constexpr (GATHER) d = ld_stream(&g.node[N0 + min(lane, NE - 1)]) & kDofMask;
    const WaveSum rz_sum(CG ? a.cg.nrz : 1, CG ? a.cg.rz_partial : u);
    const double rz_old = CG ? *a.cg.rz_old : 0.0;
    const int64_t P = pt0 + t * C::TP + (slot ? lane : 0);
    double ep[4];
    if constexpr (STRESS || FEAT) {
        ep[0] = ld_stream(&st.ep0[P]);
        ep[1] = ld_stream(&st.ep1[P]);
        ep[2] = ld_stream(&st.ep2[P]);
        ep[3] = ld_stream(&st.ep3[P]);
    }
    double alpha = 0.0;
    if constexpr (FEAT) alpha = ld_stream(&st.alpha[P]);
    int64_t o = -1;
    if constexpr (POINTS || FEAT) o = ld_stream(&a.orig[P]);
    double dp[9];
    float dpf[9];
    if constexpr (TAN) {
#pragma unroll
        for (int k = 0; k < 9; k++) {
            if constexpr (F32)
                dpf[k] = ld_stream(&a.dep32[k * a.npad + P]);
            else
                dp[k] = ld_stream(&a.dep[k * a.npad + P]);
        }
    }
    double ux = 0.0, uy = 0.0;
    if constexpr (GATHER) {
        ux = u[d];
        uy = u[d + 1];
    }
    if constexpr (CG) {
        const double px = a.cg.p[d], py = a.cg.p[d + 1];
        const double beta = cg_beta(rz_sum.get(a.cg.nrz, a.cg.rz_partial), rz_old);
        ux = ux + beta * px;
        uy = uy + beta * py;
    }
    T b[C::NV];
    double w = 0.0;
    if constexpr (FmtTraits<FMT>::GEOM) {
        if (valid) {
            w = geom_values<SHAPE>(static_cast<const double*>(g.B) + 8 * E0, g.tab, 0, lane, b);
        } else {
#pragma unroll
            for (int k = 0; k < C::NV; k++) b[k] = T(0);
        }
    } else {
        if constexpr (STRESS) w = ld_stream(&st.w[P]);
        if (slot) {
            load_values<SHAPE, FMT>(static_cast<const T*>(g.B) + val0 + t * (int64_t)(C::NV * C::TP), 0, lane, b);
        } else {
#pragma unroll
            for (int k = 0; k < C::NV; k++) b[k] = T(0);
        }
    }
    if (GATHER && lane < NE) {
        us[2 * lane] = ux;
        us[2 * lane + 1] = uy;
    }
    if (POINTS && slot && lane == el * C::NIP) oel[el] = o;
    // returned strains and forces keep what the blocks' zeros make of an
    // infinite or NaN value (a return map makes NaN of such a point anyway)
    const bool odd_u =
        OP == EL_STRAIN && __ballot(!(__builtin_isfinite(ux) && __builtin_isfinite(uy))) != 0;
    __syncthreads();
    if constexpr (OP == EL_FORCE) {
        load_points<3, C::NIP>(pts, oel, nv, a.point);
        __syncthreads();
    }
    double x[3] = {0.0, 0.0, 0.0};
    if (valid) {
        double e3[3];
        if constexpr (GATHER) strain_fmt<SHAPE, FMT>(b, us + el * C::CE, e3);
        if (PARK) park<C::NV>(lds + lane * PS, b);
        if constexpr (OP == EL_STRAIN) {
#pragma unroll
            for (int k = 0; k < 3; k++) pts[3 * lane + k] = e3[k];
            if (odd_u) {
                for (int a = 0; a < NSH; a++) {
                    pts[3 * lane] += 0.0 * us[el * C::CE + 2 * a + 1];
                    pts[3 * lane + 2] += 0.0 * us[el * C::CE + 2 * a];
                }
            }
        } else if constexpr (OP == EL_FORCE) {
#pragma unroll
            for (int k = 0; k < 3; k++) x[k] = pts[3 * lane + k];
            const double xx = x[0];
            x[0] += 0.0 * x[2];
            x[2] += 0.0 * xx;
        } else if constexpr (FEAT) {
            point_features(e3, ep, alpha, g.mats[tm >> 8], a.feat + o * mlp::FEAT_STRIDE, a.label[o], a.target[o]);
        } else if constexpr (TAN) {
#pragma unroll
            for (int k = 0; k < 3; k++) {
                if constexpr (F32) {
                    float a = dpf[3 * k] * float(e3[0]);
                    a = a + dpf[3 * k + 1] * float(e3[1]);
                    a = a + dpf[3 * k + 2] * float(e3[2]);
                    x[k] = -double(a);
                } else {
                    double a = dp[3 * k] * e3[0];
                    a = a + dp[3 * k + 1] * e3[1];
                    a = a + dp[3 * k + 2] * e3[2];
                    x[k] = -a;  // the node sums subtract
                }
            }
        } else {
            const MatConst& mc = g.mats[tm >> 8];
            if constexpr (OP == EL_DEP) {
                double d9[9];
                int mt, br;
                point_sigma<true>(e3, ep, alpha, mt, br, mc, w, x, d9);
#pragma unroll
                for (int k = 0; k < 9; k++) a.dep[k * a.npad + P] = d9[k];
                if (PARK) unpark<C::NV>(lds + lane * PS, b);
            } else if (!(OP == EL_CERTIFIED && certified_elastic(e3, ep, mc, w, x))) {
                int mt, br;
                point_sigma<false>(e3, ep, alpha, mt, br, mc, w, x, nullptr);
            }
        }
    }
    if constexpr (OP == EL_STRAIN) {
        __syncthreads();
        store_points<3, C::NIP>(pts, oel, nv, a.point);
    }
    if constexpr (!FORCES) return;
    if (PARK) __syncthreads();  // every row read back before the rows are staged
    // node rj of element re: its x and y columns, in the half that holds the node
    const int re = lane / NSH, rj = lane - re * NSH;
    const bool task = lane < NE && re < nv;
    const bool first = rj < H / 2;
    dv2 f = {0.0, 0.0};
    if (slot) bt_cols<SHAPE, FMT, 0, H>(b, x, lds + lane * RS);
    __syncthreads();
    if (task && first) {
        const T* L = lds + re * C::NIP * RS + 2 * rj;
        T fx = L[0], fy = L[1];
#pragma unroll
        for (int ip = 1; ip < C::NIP; ip++) {
            fx = fx + L[ip * RS];
            fy = fy + L[ip * RS + 1];
        }
        f = dv2{double(fx), double(fy)};
    }
    __syncthreads();
    if (slot) bt_cols<SHAPE, FMT, H, C::CE>(b, x, lds + lane * RS2);
    __syncthreads();
    if (task && !first) {
        const T* L = lds + re * C::NIP * RS2 + 2 * rj - H;
        T fx = L[0], fy = L[1];
#pragma unroll
        for (int ip = 1; ip < C::NIP; ip++) {
            fx = fx + L[ip * RS2];
            fy = fy + L[ip * RS2 + 1];
        }
        f = dv2{double(fx), double(fy)};
    }
    if (task) reinterpret_cast<dv2*>(a.ef)[N0 + lane] = f;
}

// The separate steps and the features, per 716 k Q2 points (dense B, a launch
// per color, every point's three values stored lane by lane -> now): strain
// 4 x 16.9 -> 17.9 us, force 4 x 19.0 + clear 4.8 -> 18.5 + nodes 7.4, stress
// 4 x 10.9 -> 31.4 (bound by the return map's instructions); features of 1.44 M
// points 4 x (33.0 + 16.7) -> 49.9.

// The return map of a shape's points, strains and stresses (DEP: w Dep too) in
// the reference order through LDS rows (store_points).
template <int SHAPE, bool DEP>
__global__ void __launch_bounds__(kWave, DEP ? 3 : 4)
k_stress(SplitDev g, const double* __restrict__ strain, double* __restrict__ wsigma, double* __restrict__ wdep,
         const int64_t* __restrict__ orig, PointState st, int commit) {
    constexpr int NIP = shape_nip(SHAPE), ET = shape_et(SHAPE), TP = shape_tp(SHAPE), N = DEP ? 9 : 3;
    __shared__ double sh[N * TP];
    __shared__ int64_t oel[ET];
    const int lane = threadIdx.x;
    const SplitTile at = split_tile(g, (int)xcd_tile(blockIdx.x, gridDim.x));
    const int t = at.t;
    int tile0 = g.tile0[0], pt0 = g.pt0[0];
#pragma unroll
    for (int c = 1; c < kSplitColors; c++)
        if (c == at.seg) {
            tile0 = g.tile0[c];
            pt0 = g.pt0[c];
        }
    const int tm = g.tmeta[tile0 + t];
    const int nv = tm & 255, el = lane / NIP;
    const bool slot = lane < TP, valid = slot && el < nv;
    const int64_t P = pt0 + t * TP + (slot ? lane : 0);
    const int64_t o = ld_stream(&orig[P]);
    double ep[4] = {ld_stream(&st.ep0[P]), ld_stream(&st.ep1[P]), ld_stream(&st.ep2[P]), ld_stream(&st.ep3[P])};
    double alpha = commit ? st.alpha[P] : 0.0;
    const double w = ld_stream(&st.w[P]);
    if (slot && lane == el * NIP) oel[el] = o;
    __syncthreads();
    load_points<3, NIP>(sh, oel, nv, strain);
    __syncthreads();
    double ws[3] = {0.0, 0.0, 0.0}, d9[9];
    if (valid) {
        const double e3[3] = {sh[3 * lane], sh[3 * lane + 1], sh[3 * lane + 2]};
        int mt, br;
        point_sigma<DEP>(e3, ep, alpha, mt, br, g.mats[tm >> 8], w, ws, d9);
        if (commit) {
            st.ep0[P] = ep[0];
            st.ep1[P] = ep[1];
            st.ep2[P] = ep[2];
            st.ep3[P] = ep[3];
            st.alpha[P] = alpha;
            st.mtype[P] = (signed char)mt;
            st.branch[P] = (signed char)br;
        }
    }
    __syncthreads();
    if (valid) {
#pragma unroll
        for (int k = 0; k < 3; k++) sh[3 * lane + k] = ws[k];
    }
    __syncthreads();
    store_points<3, NIP>(sh, oel, nv, wsigma);
    if constexpr (DEP) {
        __syncthreads();
        if (valid) {
#pragma unroll
            for (int k = 0; k < 9; k++) sh[9 * lane + k] = d9[k];
        }
        __syncthreads();
        store_points<9, NIP>(sh, oel, nv, wdep);
    }
}

// map[node * 4 NQ + color] = the entry of ef that the color's element adds to
// the node, -1 where the color has none.
__global__ void k_fill_int(int64_t n, int* __restrict__ p, int v) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ void k_node_map(GroupDev g, int et, int nsh, int64_t n0, int color, int stride, int* __restrict__ map) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int per = et * nsh;
    if (i >= g.ntiles * per) return;
    const int64_t t = i / per;
    if ((int)(i - t * per) / nsh >= tile_nvalid(g, t)) return;
    const int64_t node = (g.node[i] & kDofMask) >> 1;
    map[node * stride + color] = (int)(n0 + i);
}

// the node's entries of ef, one per color
template <int NQ>
__device__ __forceinline__ void node_entries(const int* __restrict__ map, int64_t k, int* m) {
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        const int4 v = reinterpret_cast<const int4*>(map)[k * NQ + q];
        m[4 * q] = v.x;
        m[4 * q + 1] = v.y;
        m[4 * q + 2] = v.z;
        m[4 * q + 3] = v.w;
    }
}

// x, y -= the node's element forces in color order.  Every load is issued
// before the first use: a color without an element reads entry 0, unused.
template <int NQ>
__device__ __forceinline__ void node_sum(const int* m, const dv2* __restrict__ ef, double& x, double& y) {
    dv2 f[4 * NQ];
#pragma unroll
    for (int c = 0; c < 4 * NQ; c++) f[c] = ef[max(m[c], 0)];
#pragma unroll
    for (int c = 0; c < 4 * NQ; c++) {
        x = m[c] >= 0 ? x + (-f[c].x) : x;
        y = m[c] >= 0 ? y + (-f[c].y) : y;
    }
}

// out = start - sum (start null: 0), one thread per node of two DoFs (the
// last DoF of an odd count has none to share it with)
template <int NQ>
__global__ void __launch_bounds__(256)
k_nodes(int64_t n, const int* __restrict__ map, const dv2* __restrict__ ef, const double* __restrict__ start,
        double* __restrict__ out) {
    const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (2 * k >= n) return;
    const bool two = 2 * k + 1 < n;
    double x = start ? start[2 * k] : 0.0, y = start && two ? start[2 * k + 1] : 0.0;
    int m[4 * NQ];
    node_entries<NQ>(map, k, m);
    node_sum<NQ>(m, ef, x, y);
    out[2 * k] = x;
    if (two) out[2 * k + 1] = y;
}

// The node sums of a CG matvec: p = z + beta p_old, q = 0 - sum on the free
// DoFs, 0 on the fixed ones, and the block partials of p.q.
template <int NQ>
__global__ void __launch_bounds__(256)
k_nodes_cg(int64_t n, const int* __restrict__ map, const dv2* __restrict__ ef, const signed char* __restrict__ mask,
           const double* __restrict__ z, CgBeta cg, double* __restrict__ rz_new, double* __restrict__ p,
           double* __restrict__ q, double* __restrict__ partial) {
    __shared__ double sh[4];
    double s = 0.0, beta = 0.0;
    // the first node's requests leave with those of beta
    const WaveSum ws(cg.nrz, cg.rz_partial);
    const double rz_old = *cg.rz_old;
    const int64_t last = (n - 1) / 2;  // the last node
    const int64_t S = (int64_t)gridDim.x * 256;
    bool first = true;
    for (int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x; first || k <= last; k += S) {
        const int64_t i0 = 2 * min(k, last), i1 = min(i0 + 1, n - 1);
        int m[4 * NQ];
        node_entries<NQ>(map, i0 / 2, m);
        const double z0 = z[i0], z1 = z[i1], q0 = cg.p[i0], q1 = cg.p[i1];
        const bool m0 = mask[i0] != 0, m1 = mask[i1] != 0;
        double x = 0.0, y = 0.0;
        node_sum<NQ>(m, ef, x, y);
        if (first) {  // every lane of the wavefront
            const double rz = ws.get(cg.nrz, cg.rz_partial);
            beta = cg_beta(rz, rz_old);
            if (blockIdx.x == 0 && threadIdx.x == 0) *rz_new = rz;
            first = false;
        }
        if (k <= last) {
            if (m0) x = 0.0;
            if (m1) y = 0.0;
            const double p0 = z0 + beta * q0;
            q[i0] = x;
            p[i0] = p0;
            s = s + p0 * x;
            if (i1 > i0) {
                const double p1 = z1 + beta * q1;
                q[i1] = y;
                p[i1] = p1;
                s = s + p1 * y;
            }
        }
    }
    const double sum = block_sum_waves<4>(s, sh);
    if (threadIdx.x == 0) partial[blockIdx.x] = sum;
}

template <int FMT, int OP>
void elem(int shape, const SplitDev& g, const ElemArgs& a, hipStream_t s) {
    dispatch_shape(shape, [&](auto sc) {
        constexpr int S = decltype(sc)::value;
        hipLaunchKernelGGL((k_elem<S, FMT, OP>), dim3((unsigned)g.ntiles), dim3(kWave), 0, s, g, a.u, a);
    });
}

template <int FMT>
void elem_op(int op, int shape, const SplitDev& g, const ElemArgs& a, hipStream_t s) {
    switch (op) {
        case EL_RESIDUAL: elem<FMT, EL_RESIDUAL>(shape, g, a, s); break;
        case EL_CERTIFIED: elem<FMT, EL_CERTIFIED>(shape, g, a, s); break;
        case EL_TANGENT: elem<FMT, EL_TANGENT>(shape, g, a, s); break;
        case EL_CG: elem<FMT, EL_CG>(shape, g, a, s); break;
        default: break;
    }
    if constexpr (FMT != FMT_G32) {
        switch (op) {
            case EL_DEP: elem<FMT, EL_DEP>(shape, g, a, s); break;
            case EL_STRAIN: elem<FMT, EL_STRAIN>(shape, g, a, s); break;
            case EL_FORCE: elem<FMT, EL_FORCE>(shape, g, a, s); break;
            case EL_FEATURES: elem<FMT, EL_FEATURES>(shape, g, a, s); break;
            default: break;
        }
    }
}

}  // namespace

void launch_elem(int op, int fmt, int shape, const SplitDev& g, const ElemArgs& a, hipStream_t s) {
    if (g.ntiles == 0) return;
    if (fmt == FMT_G64)
        elem_op<FMT_G64>(op, shape, g, a, s);
    else if (fmt == FMT_C64)
        elem_op<FMT_C64>(op, shape, g, a, s);
    else if (fmt == FMT_G32)
        elem_op<FMT_G32>(op, shape, g, a, s);
}

void launch_stress(int shape, const SplitDev& g, const double* strain, double* wsigma, double* wdep,
                   const int64_t* orig, const PointState& st, bool commit, hipStream_t s) {
    if (g.ntiles == 0) return;
    const dim3 grid((unsigned)g.ntiles), block(kWave);
    dispatch_shape(shape, [&](auto sc) {
        constexpr int S = decltype(sc)::value;
        if (wdep)
            hipLaunchKernelGGL((k_stress<S, true>), grid, block, 0, s, g, strain, wsigma, wdep, orig, st, commit ? 1 : 0);
        else
            hipLaunchKernelGGL((k_stress<S, false>), grid, block, 0, s, g, strain, wsigma, wdep, orig, st,
                               commit ? 1 : 0);
    });
}

void launch_fill_int(int64_t n, int* p, int v, hipStream_t s) {
    if (n) hipLaunchKernelGGL(k_fill_int, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, p, v);
}

void launch_node_map(int shape, const GroupDev& g, int64_t n0, int color, int stride, int* map, hipStream_t s) {
    const int et = shape_et(shape), nsh = shape_ce(shape) / 2;
    const int64_t n = g.ntiles * et * nsh;
    if (n)
        hipLaunchKernelGGL(k_node_map, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, g, et, nsh, n0, color,
                           stride, map);
}

void launch_nodes(int64_t n, int stride, const int* map, const double* ef, const double* start, double* out,
                  hipStream_t s) {
    if (n == 0) return;
    const dim3 grid((unsigned)(((n + 1) / 2 + 255) / 256)), block(256);
    const dv2* e = reinterpret_cast<const dv2*>(ef);
    if (stride == 4)
        hipLaunchKernelGGL(k_nodes<1>, grid, block, 0, s, n, map, e, start, out);
    else
        hipLaunchKernelGGL(k_nodes<2>, grid, block, 0, s, n, map, e, start, out);
}

void launch_nodes_cg(int64_t n, int stride, const int* map, const double* ef, const signed char* mask, const double* z,
                     const CgBeta& cg, double* rz_new, double* p, double* q, double* partial, int nb, hipStream_t s) {
    const dv2* e = reinterpret_cast<const dv2*>(ef);
    if (stride == 4)
        hipLaunchKernelGGL(k_nodes_cg<1>, dim3(nb), dim3(256), 0, s, n, map, e, mask, z, cg, rz_new, p, q, partial);
    else
        hipLaunchKernelGGL(k_nodes_cg<2>, dim3(nb), dim3(256), 0, s, n, map, e, mask, z, cg, rz_new, p, q, partial);
}

}  // namespace ipf
