// ipf_fmt.h -- building blocks of the element kernels, shared by the colored
// launches (ipf_kernels_fmt.hip) and the element / node launches
// (ipf_split.hip): workgroup -> tile mapping, the B formats' loads, strains
// and B^T products.
#pragma once

#include "ipf_geometry.h"
#include "ipf_kernels.h"

namespace ipf {

namespace {

constexpr int kWave = 64;

// Workgroup -> tile (patch) of a launch of n workgroups.  The hardware deals
// consecutive workgroups of a dispatch to the 8 XCDs in turn, each with its
// own L2; this mapping gives XCD x one contiguous range of tiles -- ranges of
// q + 1 tiles for the first n mod 8 XCDs, q = n / 8 for the others -- so
// that neighbouring tiles, whose DoF, state and geometry arrays share cache
// lines at the tile boundaries, are read through the same L2.  A bijection
// of [0, n); the results do not depend on it (no two tiles of a launch write
// the same value).
__device__ __forceinline__ int64_t xcd_tile(int64_t b, int64_t n) {
    const int64_t q = n >> 3, r = n & 7, x = b & 7, k = b >> 3;
    return x < r ? x * (q + 1) + k : r * (q + 1) + (x - r) * q + k;
}

template <int FMT>
struct FmtTraits;
template <>
struct FmtTraits<FMT_D64> { using T = double; static constexpr bool COMPACT = false, GEOM = false; static constexpr int VEC = 2; };
template <>
struct FmtTraits<FMT_C64> { using T = double; static constexpr bool COMPACT = true, GEOM = false; static constexpr int VEC = 2; };
template <>
struct FmtTraits<FMT_D32> { using T = float; static constexpr bool COMPACT = false, GEOM = false; static constexpr int VEC = 4; };
template <>
struct FmtTraits<FMT_C32> { using T = float; static constexpr bool COMPACT = true, GEOM = false; static constexpr int VEC = 4; };
template <>
struct FmtTraits<FMT_G64> { using T = double; static constexpr bool COMPACT = true, GEOM = true; static constexpr int VEC = 2; };
template <>
struct FmtTraits<FMT_G32> { using T = float; static constexpr bool COMPACT = true, GEOM = true; static constexpr int VEC = 4; };

template <int SHAPE, int FMT>
struct FC {
    using F = FmtTraits<FMT>;
    using T = typename F::T;
    static constexpr int NIP = shape_nip(SHAPE);
    static constexpr int CE = shape_ce(SHAPE);
    static constexpr int ET = shape_et(SHAPE);
    static constexpr int TP = shape_tp(SHAPE);
    static constexpr int NV = format_values(SHAPE, FMT);  // stored values per point (padded)
    static constexpr int VEC = F::VEC;
    static constexpr int MIN_WAVES = F::COMPACT ? 4 : ((CE <= 8) ? 4 : (CE <= 18) ? 3 : 1);
};

template <class T>
__device__ __forceinline__ T ld_stream(const T* p) {
    return __builtin_nontemporal_load(p);
}

typedef double dv2 __attribute__((ext_vector_type(2)));
typedef float fv4 __attribute__((ext_vector_type(4)));

template <int SHAPE, int FMT>
__device__ __forceinline__ void load_values(const void* __restrict__ Bg, int64_t tile, int lane,
                                            typename FC<SHAPE, FMT>::T* b) {
    using C = FC<SHAPE, FMT>;
    if constexpr (C::VEC == 2) {
        const dv2* Bt = reinterpret_cast<const dv2*>(Bg) + tile * (int64_t)(C::NV / 2 * C::TP);
#pragma unroll
        for (int m = 0; m < C::NV / 2; m++) {
            const dv2 v = ld_stream(&Bt[m * C::TP + lane]);
            b[2 * m] = v.x;
            b[2 * m + 1] = v.y;
        }
    } else {
        const fv4* Bt = reinterpret_cast<const fv4*>(Bg) + tile * (int64_t)(C::NV / 4 * C::TP);
#pragma unroll
        for (int m = 0; m < C::NV / 4; m++) {
            const fv4 v = ld_stream(&Bt[m * C::TP + lane]);
            b[4 * m] = v.x;
            b[4 * m + 1] = v.y;
            b[4 * m + 2] = v.z;
            b[4 * m + 3] = v.w;
        }
    }
}

// Geometric format: the compact values (dN_a/dx, dN_a/dy) of the lane's point
// from its element's corners (Bg: 8 doubles per element slot of the group)
// and the shape table, computed in FP64 and stored as T (FP32: rounded);
// returns the weight w_q |det J|.
template <int SHAPE, class T>
__device__ __forceinline__ double geom_values(const double* __restrict__ Bg, const double* __restrict__ tab,
                                              int64_t tile, int lane, T* b) {
    using C = FC<SHAPE, FMT_G64>;
    const int el = lane / C::NIP, ip = lane - el * C::NIP;
    const dv2* Xv = reinterpret_cast<const dv2*>(Bg) + (tile * C::ET + el) * 4;
    double X[8];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const dv2 v = ld_stream(&Xv[c]);
        X[2 * c] = v.x;
        X[2 * c + 1] = v.y;
    }
    const double* xi = tab + C::NIP * C::CE;
    const QuadMap m = quad_map(X, xi[ip], xi[C::NIP + ip]);
    const dv2* dphi = reinterpret_cast<const dv2*>(tab) + ip * (C::CE / 2);
#pragma unroll
    for (int a = 0; a < C::CE / 2; a++) {
        const dv2 d = dphi[a];
        double gx, gy;
        quad_grad(m, d.x, d.y, gx, gy);
        b[2 * a] = T(gx);
        b[2 * a + 1] = T(gy);
    }
    return quad_weight(m, xi[2 * C::NIP + ip]);
}

// strain in the accumulation type T.  Dense: rows summed over columns j
// ascending.  Compact: the same sums with the zero terms left out.
template <int SHAPE, int FMT>
__device__ __forceinline__ void strain_fmt(const typename FC<SHAPE, FMT>::T* b, const double* ue, double* e3) {
    using C = FC<SHAPE, FMT>;
    using T = typename C::T;
    if constexpr (FmtTraits<FMT>::COMPACT) {
        // (the dense sums start from 0: a zero's sign apart, from the first term)
        T a0 = b[0] * T(ue[0]), a1 = b[1] * T(ue[0]), a2 = b[1] * T(ue[1]);
        a1 = a1 + b[0] * T(ue[1]);
#pragma unroll
        for (int a = 1; a < C::CE / 2; a++) {
            const T dx = b[2 * a], dy = b[2 * a + 1];
            const T ux = T(ue[2 * a]), uy = T(ue[2 * a + 1]);
            a0 = a0 + dx * ux;
            a1 = a1 + dy * ux;
            a1 = a1 + dx * uy;
            a2 = a2 + dy * uy;
        }
        e3[0] = double(a0);
        e3[1] = double(a1);
        e3[2] = double(a2);
    } else {
#pragma unroll
        for (int k = 0; k < 3; k++) {
            T acc = T(0);
#pragma unroll
            for (int j = 0; j < C::CE; j++) acc = acc + b[k * C::CE + j] * T(ue[j]);
            e3[k] = double(acc);
        }
    }
}

// Row stride of the staged partials: every lane writes its row of W values of
// B bytes in 16-byte pieces, eight lanes at a time, and reads pairs down the
// columns.  A stride of W put the rows of Q3 (16 FP64 values) on one bank in
// four (960 of 1,296 LDS cycles per wavefront were conflicts, and the LDS bound
// the launch); W rounded up to an odd multiple of 16 bytes spreads eight rows
// over all 64 banks.
constexpr int row_stride(int w, int bytes) {
    const int per = 16 / bytes;
    if (w % 2) return w;  // single values
    int q = (w + per - 1) / per;
    return (q % 2 ? q : q + 1) * per;
}

// The element launch of the residual with tangent parks B in LDS while the
// return map and the tangent fill the registers (a row of the lane's own, read
// back before the rows are staged): two wavefronts per SIMD at Q2 become three
// at 140 VGPRs; residual, tangent and K of 201x150 Q2 74 us, so 71 to 72.  Not at
// Q1, which has three anyway, nor at Q3, whose rows would take 17 KB per
// wavefront, nor in the launch per color, which spills at three (400x400 Q2
// 148 us, so 184).
constexpr bool park_B(int ce) { return ce > 8 && ce <= 20; }
template <int N, class T>
__device__ __forceinline__ void park(T* row, const T* b) {
#pragma unroll
    for (int k = 0; k < N; k++) row[k] = b[k];
    asm volatile("" ::: "memory");  // read back, not kept
}
template <int N, class T>
__device__ __forceinline__ void unpark(const T* row, T* b) {
    asm volatile("" ::: "memory");
#pragma unroll
    for (int k = 0; k < N; k++) b[k] = row[k];
}

// Columns [J0, J1) of one point's B^T (w sigma) partials into row[j - J0].
// Dense: rows summed in order per column; compact: the same sums without the
// zero terms.  The residual and tangent kernels stage half the columns at a
// time, which halves the LDS a wave holds (one wave per workgroup) so that
// registers, not LDS, bound the waves per CU.
template <int SHAPE, int FMT, int J0, int J1>
__device__ __forceinline__ void bt_cols(const typename FC<SHAPE, FMT>::T* b, const double* x,
                                        typename FC<SHAPE, FMT>::T* row) {
    using C = FC<SHAPE, FMT>;
    using T = typename C::T;
    const T x0 = T(x[0]), x1 = T(x[1]), x2 = T(x[2]);
#pragma unroll
    for (int j = J0; j < J1; j++) {
        T g;
        if constexpr (FmtTraits<FMT>::COMPACT) {
            const int a = j / 2;
            const T dx = b[2 * a], dy = b[2 * a + 1];
            if ((j & 1) == 0) {
                g = dx * x0;
                g = g + dy * x1;
            } else {
                g = dx * x1;
                g = g + dy * x2;
            }
        } else {
            g = b[j] * x0;
            g = g + b[C::CE + j] * x1;
            g = g + b[2 * C::CE + j] * x2;
        }
        row[j - J0] = g;
    }
}

// One lane's column sum: the partials L of element e's points in column jj of
// the staged half (rows W values apart), summed in point order and added negated to
// r[d] (TPZNumericalIntegrator::MultiplyTranspose's y = -B^T x); rv = r[d],
// read by the caller ahead of time.  Each lane owns one column sum per half
// (ET * W <= 64 for every shape), and the color's elements share no DoF, so
// no atomics.
template <int SHAPE, int FMT, int W>
__device__ __forceinline__ void reduce_lane(const typename FC<SHAPE, FMT>::T* L, int e, int jj, int d, double rv,
                                            double* __restrict__ r) {
    using C = FC<SHAPE, FMT>;
    using T = typename C::T;
    T f = L[(e * C::NIP) * W + jj];
#pragma unroll
    for (int ip = 1; ip < C::NIP; ip++) f = f + L[(e * C::NIP + ip) * W + jj];
    r[d] = rv + (-double(f));
}

}  // namespace

}  // namespace ipf
