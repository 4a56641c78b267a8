// ipf_assemble.hip -- tangent stiffness assembly into the symmetric CSR
// values (TPZNumericalIntegrator::KAssembly, TPZNumericalIntegrator.cpp:131-214,
// with ComputeTangentMatrix :236-270 and the per-color gather / add / scatter
// of :166-178).
//
// General blocks: one wavefront per element.  The element's dense B rows (3 x C per point),
// its points' w*Dep (3 x 3) and the products Dep.B are staged in LDS; the
// lanes then produce the packed upper triangle K_e(a, c), a <= c, row by row
// (the order of fColorLSequence), and add each entry to Kg at its CSR
// position.  Launched once per (color, shape) group in color order, so every
// Kg entry receives its element contributions color by color as in the
// reference, and the elements of one launch never share a CSR position (they
// share no DoF).
//
// Operation order per entry (the CPU restatement in the oracle uses the same):
//   DB[r][j]  = 0 + D[r][0] B[0][j] + D[r][1] B[1][j] + D[r][2] B[2][j]
//   K_e(a, c) = sum over points, in point order, of
//               (0 + B[0][a] DB[0][c] + B[1][a] DB[1][c] + B[2][a] DB[2][c])
//   Kg[l]     = Kg[l] + K_e(a, c)
#include "ipf_fmt.h"

namespace ipf {

namespace {

// Kg[l] = start + ke: an entry's first element in launch order (kFirstWrite
// on the position) starts from 0, so Kg needs no clear.
__device__ __forceinline__ void add_K(double* __restrict__ kg, int l, double old, double ke) {
    kg[l & kDofMask] = (l < 0 ? 0.0 : old) + ke;
}

template <int SHAPE>
__global__ void __launch_bounds__(kWave)
k_assemble_K(GroupDev g, const double* __restrict__ dep, int64_t npad, const int* __restrict__ lidx,
             double* __restrict__ kg) {
    constexpr int NIP = shape_nip(SHAPE);
    constexpr int CE = shape_ce(SHAPE);
    constexpr int ET = shape_et(SHAPE);
    constexpr int TP = shape_tp(SHAPE);
    constexpr int NB = 3 * CE;
    constexpr int NT = CE * (CE + 1) / 2;
    __shared__ double Bs[NIP * NB];
    __shared__ double Ds[NIP * 9];
    __shared__ double DBs[NIP * NB];
    const int lane = threadIdx.x;
    const int64_t elem = blockIdx.x;  // grid = g.nelem element slots
    const int64_t tile = elem / ET;
    const int el = (int)(elem - tile * ET);
    if (el >= tile_nvalid(g, tile)) return;  // padding slot
    // dense tile layout: value m of tile slot q at (m / 2) * 2 TP + 2 q + (m & 1)
    const double* Bt = g.B + tile * (int64_t)(NB * TP);
    for (int t = lane; t < NIP * NB; t += kWave) {
        const int ip = t / NB;
        const int m = t - ip * NB;
        const int q = el * NIP + ip;
        Bs[t] = Bt[(m >> 1) * (2 * TP) + 2 * q + (m & 1)];
    }
    const int64_t P0 = g.pt0 + tile * TP + el * NIP;
    for (int t = lane; t < NIP * 9; t += kWave) {
        const int ip = t / 9;
        const int rk = t - ip * 9;
        Ds[t] = dep[rk * npad + P0 + ip];
    }
    __syncthreads();
    for (int t = lane; t < NIP * NB; t += kWave) {
        const int ip = t / NB;
        const int rj = t - ip * NB;
        const int r = rj / CE;
        const int j = rj - r * CE;
        double acc = 0.;
#pragma unroll
        for (int k = 0; k < 3; k++) acc = acc + Ds[ip * 9 + 3 * r + k] * Bs[ip * NB + k * CE + j];
        DBs[t] = acc;
    }
    __syncthreads();
    const int* li = lidx + elem * (int64_t)NT;
    for (int t = lane; t < NT; t += kWave) {
        // packed row-major upper triangle: row a holds CE - a entries
        int a = 0, rem = t;
        while (rem >= CE - a) {
            rem -= CE - a;
            a++;
        }
        const int c = a + rem;
        double ke = 0.;
        for (int ip = 0; ip < NIP; ip++) {
            double acc = 0.;
#pragma unroll
            for (int k = 0; k < 3; k++) acc = acc + Bs[ip * NB + k * CE + a] * DBs[ip * NB + k * CE + c];
            ke = ke + acc;
        }
        const int l = li[t];
        add_K(kg, l, l < 0 ? 0.0 : kg[l], ke);
    }
}

// Where B has the 2D elasticity pattern (dN_a/dx, dN_a/dy): one wavefront for
// EPW elements, one lane for a pair of nodes a <= c, whose (up to) four entries
// K(2a + i, 2c + j) it sums over the points from four values of B in LDS and
// the point's w Dep.  The dense form above reads six LDS values per entry and
// point and was bound by that; here a pair reads four for four entries, and
// the terms with B's zeros are left out (the same sums).  GEOM: B from the
// element's corners, as the residual forms it, instead of 3 n_ip C_e stored
// values.  The positions and, behind them, the entries of Kg are requested
// first and arrive behind the products.
// Bound by the products (34 instructions per pair and point, 45 of 64 lanes at
// Q2, 136 of 192 at Q3) and the round trips position -> entry.  Residual,
// tangent and assembly, before (with the clear of Kg) -> now: 201x150 Q2
// 124 -> 66 us; 300x300 (from the stored dense B throughout) Q1 186 -> 84,
// Q2 586 -> 240, Q3 2,280 -> 728 us.
// Registers for seven wavefronts per SIMD where one element fills a wavefront:
// a color of a mesh of some ten thousand elements is then in flight at once
// (Q2 84 VGPRs, five wavefronts -> 44, eight: 201x150 Q2 71 -> 66 us; no
// spills).  Several elements share a wavefront's LDS rows at Q1, T1 and T2,
// which that bound would spill; Q3's LDS allows four anyway.
constexpr int pair_waves(int ce) { return ce * (ce + 2) / 8 > kWave / 2 ? 7 : 1; }
template <int SHAPE, bool GEOM>
__global__ void __launch_bounds__(kWave, pair_waves(shape_ce(SHAPE)))
k_assemble_pairs(GroupDev g, const double* __restrict__ geo, const double* __restrict__ dep, int64_t npad,
                 const int* __restrict__ lidx, double* __restrict__ kg) {
    constexpr int NIP = shape_nip(SHAPE), CE = shape_ce(SHAPE), ET = shape_et(SHAPE), TP = shape_tp(SHAPE);
    constexpr int NSH = CE / 2, NP = NSH * (NSH + 1) / 2, NT = CE * (CE + 1) / 2;
    constexpr int EPW = NP >= kWave ? 1 : (kWave / NP < ET ? kWave / NP : ET);  // elements per wavefront
    constexpr int ROUNDS = (NP + kWave - 1) / kWave;                            // of one element's pairs
    constexpr int NL = (EPW * NT + kWave - 1) / kWave;                          // positions per lane
    __shared__ dv2 Bs[EPW * NIP * NSH];
    __shared__ double Ks[EPW * NT];
    __shared__ double Js[EPW * NIP * 4];
    __shared__ double Ds[EPW > 1 ? EPW * NIP * 9 : 1];
    const int lane = threadIdx.x;
    const int64_t e0 = xcd_tile(blockIdx.x, gridDim.x) * EPW;  // first element slot of the wavefront
    auto real = [&](int64_t e) { return e < g.nelem && (int)(e % ET) < tile_nvalid(g, e / ET); };
    if (EPW == 1 && !real(e0)) return;
    int l[NL];
    double old[NL];
#pragma unroll
    for (int k = 0; k < NL; k++) {
        const int t = lane + k * kWave;
        const bool in = t < EPW * NT && real(e0 + t / NT);
        l[k] = in ? lidx[e0 * NT + t] : kFirstWrite;
    }
    // the points' maps, then every node's gradients (the entries as k_build_B writes them)
    if constexpr (GEOM) {
        for (int q = lane; q < EPW * NIP; q += kWave) {
            const int el = q / NIP, ip = q - el * NIP;
            const int64_t e = min(e0 + el, g.nelem - 1);
            double X[8];
#pragma unroll
            for (int c = 0; c < 8; c++) X[c] = geo[8 * e + c];
            const double* xi = g.tab + NIP * CE;
            const QuadMap m = quad_map(X, xi[ip], xi[NIP + ip]);
            Js[4 * q] = m.a;
            Js[4 * q + 1] = m.b;
            Js[4 * q + 2] = m.c;
            Js[4 * q + 3] = m.d;
        }
        __syncthreads();
        for (int t = lane; t < EPW * NIP * NSH; t += kWave) {
            const int q = t / NSH, a = t - q * NSH, ip = q % NIP;
            const dv2 d = reinterpret_cast<const dv2*>(g.tab)[ip * NSH + a];
            QuadMap m;
            m.a = Js[4 * q];
            m.b = Js[4 * q + 1];
            m.c = Js[4 * q + 2];
            m.d = Js[4 * q + 3];
            double x, y;
            quad_grad(m, d.x, d.y, x, y);
            Bs[t] = dv2{x, y};
        }
    } else {
        for (int t = lane; t < EPW * NIP * NSH; t += kWave) {
            const int el = t / (NIP * NSH), ip = (t - el * NIP * NSH) / NSH, a = t % NSH;
            const int64_t e = min(e0 + el, g.nelem - 1), tile = e / ET;
            const int q = (int)(e - tile * ET) * NIP + ip;
            const double* Bt = g.B + tile * (int64_t)(3 * CE * TP);
            auto at = [&](int m) { return Bt[(m >> 1) * (2 * TP) + 2 * q + (m & 1)]; };
            Bs[t] = dv2{at(2 * a), at(2 * CE + 2 * a + 1)};
        }
    }
    const int64_t P0 = g.pt0 + e0 / ET * TP + e0 % ET * NIP;  // EPW = 1: the element's first point
    if constexpr (EPW > 1) {
        for (int t = lane; t < EPW * NIP * 9; t += kWave) {
            const int k = t / (EPW * NIP), q = t - k * (EPW * NIP), el = q / NIP;
            const int64_t e = min(e0 + el, g.nelem - 1);
            Ds[q * 9 + k] = dep[k * npad + g.pt0 + e / ET * TP + e % ET * NIP + q - el * NIP];
        }
    }
#pragma unroll
    for (int k = 0; k < NL; k++) old[k] = l[k] < 0 ? 0.0 : kg[l[k]];
    __syncthreads();
#pragma unroll
    for (int rd = 0; rd < ROUNDS; rd++) {
        const int t = lane + rd * kWave;
        const int el = EPW == 1 ? 0 : t / NP, pr = t - el * NP;
        if (el < EPW && pr < NP) {
            int a = 0, c = pr;  // pair (a, c), a <= c, row by row
#pragma unroll
            for (int k = 0; k < NSH - 1; k++)
                if (a == k && c >= NSH - k) {
                    c -= NSH - k;
                    a = k + 1;
                }
            c += a;
            double k00 = 0., k01 = 0., k10 = 0., k11 = 0.;
            constexpr int UN = NIP % 4 == 0 ? 4 : 3;  // all points at once cost registers: 136 at Q2, 244 at Q3
#pragma unroll UN
            for (int ip = 0; ip < NIP; ip++) {
                const dv2 ba = Bs[(el * NIP + ip) * NSH + a], bc = Bs[(el * NIP + ip) * NSH + c];
                double D[9];
#pragma unroll
                for (int k = 0; k < 9; k++) D[k] = EPW == 1 ? dep[k * npad + P0 + ip] : Ds[(el * NIP + ip) * 9 + k];
                // columns 2c (dx, dy, 0) and 2c + 1 (0, dx, dy) of Dep B
                double x[3], y[3];
#pragma unroll
                for (int r = 0; r < 3; r++) {
                    x[r] = D[3 * r] * bc.x + D[3 * r + 1] * bc.y;
                    y[r] = D[3 * r + 1] * bc.x + D[3 * r + 2] * bc.y;
                }
                k00 = k00 + (ba.x * x[0] + ba.y * x[1]);
                k01 = k01 + (ba.x * y[0] + ba.y * y[1]);
                k10 = k10 + (ba.x * x[1] + ba.y * x[2]);
                k11 = k11 + (ba.x * y[1] + ba.y * y[2]);
            }
            // packed row-major upper triangle: row i starts at i CE - i (i - 1) / 2
            double* K = Ks + el * NT;
            const int r0 = 2 * a, r1 = r0 + 1;
            const int o0 = r0 * CE - r0 * (r0 - 1) / 2 - r0, o1 = r1 * CE - r1 * (r1 - 1) / 2 - r1;
            K[o0 + 2 * c] = k00;
            K[o0 + 2 * c + 1] = k01;
            if (a != c) K[o1 + 2 * c] = k10;
            K[o1 + 2 * c + 1] = k11;
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NL; k++) {
        const int t = lane + k * kWave;
        if (t < EPW * NT && real(e0 + t / NT)) add_K(kg, l[k], old[k], Ks[t]);
    }
}

}  // namespace

void launch_assemble_K(int shape, const GroupDev& g, const double* geo, bool pattern, const double* dep, int64_t npad,
                       const int* lidx, double* kg, hipStream_t s) {
    if (g.nelem == 0) return;
    if (pattern) {
        dispatch_shape(shape, [&](auto sc) {
            constexpr int S = decltype(sc)::value;
            constexpr int NSH = shape_ce(S) / 2, NP = NSH * (NSH + 1) / 2;
            constexpr int EPW = NP >= kWave ? 1 : (kWave / NP < shape_et(S) ? kWave / NP : shape_et(S));
            const dim3 grid((unsigned)((g.nelem + EPW - 1) / EPW));
            if (geo)
                hipLaunchKernelGGL((k_assemble_pairs<S, true>), grid, dim3(kWave), 0, s, g, geo, dep, npad, lidx, kg);
            else
                hipLaunchKernelGGL((k_assemble_pairs<S, false>), grid, dim3(kWave), 0, s, g, geo, dep, npad, lidx, kg);
        });
        return;
    }
    const dim3 grid((unsigned)g.nelem);
    dispatch_shape(shape, [&](auto sc) {
        constexpr int S = decltype(sc)::value;
        hipLaunchKernelGGL(k_assemble_K<S>, grid, dim3(kWave), 0, s, g, dep, npad, lidx, kg);
    });
}

}  // namespace ipf
