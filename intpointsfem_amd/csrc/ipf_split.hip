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

enum ElemOp { EL_RESIDUAL = 0, EL_CERTIFIED = 1, EL_TANGENT = 2, EL_CG = 3, EL_DEP = 4 };

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
k_elem(SplitDev g, const double* __restrict__ u, PointState st, double* __restrict__ dep,
       const float* __restrict__ dep32, int64_t npad, CgBeta cg, dv2* __restrict__ ef) {
    using C = FC<SHAPE, FMT>;
    using T = typename C::T;
    constexpr bool CG = OP == EL_CG, TAN = OP == EL_TANGENT || CG;
    constexpr bool F32 = TAN && FMT == FMT_G32;
    constexpr int NSH = C::CE / 2;
    constexpr int H = 2 * ((NSH + 1) / 2), H2 = C::CE - H;
    constexpr int NE = C::ET * NSH;
    static_assert(NE <= kWave, "one node per lane");
    __shared__ T lds[C::TP * H];
    __shared__ double us[2 * NE];
    const int lane = threadIdx.x;
    const int t = (int)xcd_tile(blockIdx.x, gridDim.x);
    int tile0 = g.tile0[0], pt0 = g.pt0[0], slot0 = g.slot0[0], ent0 = g.ent0[0];
#pragma unroll
    for (int c = 1; c < kSplitColors; c++)
        if (c < g.nseg && t >= g.end[c - 1]) {
            tile0 = g.tile0[c];
            pt0 = g.pt0[c];
            slot0 = g.slot0[c];
            ent0 = g.ent0[c];
        }
    const int tm = g.tmeta[tile0 + t];
    const int64_t E0 = slot0 + t * C::ET, N0 = ent0 + t * NE;
    const int nv = tm & 255;
    const int el = lane / C::NIP;
    const bool slot = lane < C::TP;
    const bool valid = slot && el < nv;
    // indexes, then the point's state, then the values the indexes address,
    // all outside branches (padding slots hold node DoF 0 and points of their own)
    const int d = ld_stream(&g.node[N0 + min(lane, NE - 1)]) & kDofMask;
    const WaveSum rz_sum(CG ? cg.nrz : 1, CG ? cg.rz_partial : u);
    const double rz_old = CG ? *cg.rz_old : 0.0;
    const int64_t P = pt0 + t * C::TP + (slot ? lane : 0);
    double ep[4];
    if constexpr (!TAN) {
        ep[0] = ld_stream(&st.ep0[P]);
        ep[1] = ld_stream(&st.ep1[P]);
        ep[2] = ld_stream(&st.ep2[P]);
        ep[3] = ld_stream(&st.ep3[P]);
    }
    double dp[9];
    float dpf[9];
    if constexpr (TAN) {
#pragma unroll
        for (int k = 0; k < 9; k++) {
            if constexpr (F32)
                dpf[k] = ld_stream(&dep32[k * npad + P]);
            else
                dp[k] = ld_stream(&dep[k * npad + P]);
        }
    }
    double ux = u[d], uy = u[d + 1];
    if constexpr (CG) {
        const double px = cg.p[d], py = cg.p[d + 1];
        const double beta = cg_beta(rz_sum.get(cg.nrz, cg.rz_partial), rz_old);
        ux = ux + beta * px;
        uy = uy + beta * py;
    }
    T b[C::NV];
    double w = 0.0;
    if (valid) {
        w = geom_values<SHAPE>(g.geo + 8 * E0, g.tab, 0, lane, b);
    } else {
#pragma unroll
        for (int k = 0; k < C::NV; k++) b[k] = T(0);
    }
    if (lane < NE) {
        us[2 * lane] = ux;
        us[2 * lane + 1] = uy;
    }
    __syncthreads();
    double x[3] = {0.0, 0.0, 0.0};
    if (valid) {
        double e3[3];
        strain_fmt<SHAPE, FMT>(b, us + el * C::CE, e3);
        if constexpr (TAN) {
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
                double alpha = 0.0, d9[9];
                int mt, br;
                point_sigma<true>(e3, ep, alpha, mt, br, mc, w, x, d9);
#pragma unroll
                for (int k = 0; k < 9; k++) dep[k * npad + P] = d9[k];
            } else if (!(OP == EL_CERTIFIED && certified_elastic(e3, ep, mc, w, x))) {
                double alpha = 0.0;
                int mt, br;
                point_sigma<false>(e3, ep, alpha, mt, br, mc, w, x, nullptr);
            }
        }
    }
    // node rj of element re: its x and y columns, in the half that holds the node
    const int re = lane / NSH, rj = lane - re * NSH;
    const bool task = lane < NE && re < nv;
    const bool first = rj < H / 2;
    dv2 f = {0.0, 0.0};
    if (slot) bt_cols<SHAPE, FMT, 0, H>(b, x, lds + lane * H);
    __syncthreads();
    if (task && first) {
        const T* L = lds + re * C::NIP * H + 2 * rj;
        T fx = L[0], fy = L[1];
#pragma unroll
        for (int ip = 1; ip < C::NIP; ip++) {
            fx = fx + L[ip * H];
            fy = fy + L[ip * H + 1];
        }
        f = dv2{double(fx), double(fy)};
    }
    __syncthreads();
    if (slot) bt_cols<SHAPE, FMT, H, C::CE>(b, x, lds + lane * H2);
    __syncthreads();
    if (task && !first) {
        const T* L = lds + re * C::NIP * H2 + 2 * rj - H;
        T fx = L[0], fy = L[1];
#pragma unroll
        for (int ip = 1; ip < C::NIP; ip++) {
            fx = fx + L[ip * H2];
            fy = fy + L[ip * H2 + 1];
        }
        f = dv2{double(fx), double(fy)};
    }
    if (task) ef[N0 + lane] = f;
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
    __shared__ double sh[256];
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
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) sh[threadIdx.x] = sh[threadIdx.x] + sh[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = sh[0];
}

template <int FMT, int OP>
void elem(int shape, const SplitDev& g, const double* u, const PointState& st, double* dep, const float* dep32,
          int64_t npad, const CgBeta& cg, double* ef, hipStream_t s) {
    dispatch_shape(shape, [&](auto sc) {
        constexpr int S = decltype(sc)::value;
        hipLaunchKernelGGL((k_elem<S, FMT, OP>), dim3((unsigned)g.ntiles), dim3(kWave), 0, s, g, u, st, dep, dep32,
                           npad, cg, reinterpret_cast<dv2*>(ef));
    });
}

}  // namespace

void launch_elem_residual(int fmt, int shape, bool fast, const SplitDev& g, const double* u, const PointState& st,
                          double* ef, hipStream_t s) {
    if (g.ntiles == 0) return;
    if (fmt == FMT_G64) {
        if (fast)
            elem<FMT_G64, EL_CERTIFIED>(shape, g, u, st, nullptr, nullptr, 0, CgBeta{}, ef, s);
        else
            elem<FMT_G64, EL_RESIDUAL>(shape, g, u, st, nullptr, nullptr, 0, CgBeta{}, ef, s);
    } else if (fmt == FMT_G32) {
        if (fast)
            elem<FMT_G32, EL_CERTIFIED>(shape, g, u, st, nullptr, nullptr, 0, CgBeta{}, ef, s);
        else
            elem<FMT_G32, EL_RESIDUAL>(shape, g, u, st, nullptr, nullptr, 0, CgBeta{}, ef, s);
    }
}

void launch_elem_dep(int shape, const SplitDev& g, const double* u, const PointState& st, double* dep, int64_t npad,
                     double* ef, hipStream_t s) {
    if (g.ntiles) elem<FMT_G64, EL_DEP>(shape, g, u, st, dep, nullptr, npad, CgBeta{}, ef, s);
}

void launch_elem_tangent(int fmt, int shape, const SplitDev& g, const double* v, const CgBeta& cg, double* dep,
                         const float* dep32, int64_t npad, double* ef, hipStream_t s) {
    if (g.ntiles == 0) return;
    const PointState none{};
    if (fmt == FMT_G64) {
        if (cg.rz_old)
            elem<FMT_G64, EL_CG>(shape, g, v, none, dep, dep32, npad, cg, ef, s);
        else
            elem<FMT_G64, EL_TANGENT>(shape, g, v, none, dep, dep32, npad, cg, ef, s);
    } else if (fmt == FMT_G32) {
        if (cg.rz_old)
            elem<FMT_G32, EL_CG>(shape, g, v, none, dep, dep32, npad, cg, ef, s);
        else
            elem<FMT_G32, EL_TANGENT>(shape, g, v, none, dep, dep32, npad, cg, ef, s);
    }
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
