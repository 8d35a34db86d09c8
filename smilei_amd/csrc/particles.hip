// particles.hip -- the particle half of the PIC step on gfx950, FP64 form.
//
// k_particles<ND,ORDER,DEPOSIT>: one workgroup per 4-cell cluster of every
// patch (the reference's GPU cluster, Params.h:403-418).  The cluster's
// particles are contiguous in the cell-sorted list.  The workgroup
//   1. stages the six gathered field components of the cluster plus its
//      stencil halo in LDS,
//   2. per particle: gathers E and B_m (Interpolator{2D2,3D2,3D4}Order),
//      Boris-pushes (PusherBoris), tags the direction of motion against the
//      patch limits (internal_inf/sup), wraps periodic leavers
//      (Patch::prepareParticles), computes the destination cell key
//      (Cluster3D::CellKey) and, with DEPOSIT, adds the Esirkepov currents
//      (Projector{2D2,3D2,3D4}Order::currents) into an LDS tile with LDS
//      FP64 atomics,
//   3. flushes the J tile into the global arrays with FP64 atomics.
// Without DEPOSIT, gather and push use the reference's association order (the
// file is built with -ffp-contract=off); with it they are factorised and
// fused, as the current contributions are.
//
// k_det_deposit{3,2}: the same current contributions added in the reference's
// order into per-patch ghosted arrays; then the J ghost sum in x, y, z passes
// (SyncVectorPatch::sumAllComponents) and a copy of the patch interiors.
#include "kernels.h"
#include "ordered_deposit.h"
#include "pic_device.h"

namespace smi {

namespace {

using namespace dev;

// Esirkepov currents of one 3D particle into the cluster's LDS tile: old
// delta dold, new position in cell units pnn, old node ip; NT / NT - 1 window
// entries across / along the current (esirkepov3d_fact; NT = ORDER + 1: the
// node is unchanged on every axis).
template <int ORDER, int NT>
__device__ inline void deposit3_tile(double *sJ, const Geom &g, const int *G0, const double *dold, const double *pnn,
                                     const int *ip, double cw)
{
    using TL = Tile<ORDER>;
    constexpr int H = TL::H, JT = TL::JT;
    // J-tile strides: order-2 rows padded by one word (fp_cluster's layout)
    constexpr int JSY = ORDER == 2 ? JT + 1 : JT, JSX = JT * JSY, JSC = JT * JSX;
    double S0[3][ORDER + 2], DS[3][ORDER + 2];
    int w0[3] = {1, 1, 1};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        if constexpr (NT == ORDER + 1) {
            double s1[ORDER + 1];
            spline<ORDER>(dold[d], S0[d]);
            spline<ORDER>(pnn[d] - (double)ip[d], s1);
#pragma unroll
            for (int m = 0; m <= ORDER; ++m) DS[d][m] = s1[m] - S0[d][m];
        } else {
            esirkepov_window<ORDER>(dold[d], pnn[d], ip[d], S0[d], DS[d], w0[d]);
        }
    }
    const double cr[3] = {cw * g.dxdt[0], cw * g.dxdt[1], cw * g.dxdt[2]};
    // tile coords of stencil index 0 along each axis
    const int o0 = ip[0] - (H + 1) - (G0[0] - TL::JO);
    const int o1 = ip[1] - (H + 1) - (G0[1] - TL::JO);
    const int o2 = ip[2] - (H + 1) - (G0[2] - TL::JO);
    double *sJb = sJ + o0 * JSX + o1 * JSY + o2;
    esirkepov3d_fact<ORDER, NT, NT - 1>(S0, DS, w0, cr, [&](int c, int a, int b, int k, double v) {
        atomicAdd(&sJb[c * JSC + a * JSX + b * JSY + k], v);
    });
}

// The 2D J tile: rows of 12 words and four copies 112 words apart, the lane
// picking its copy: a cluster has 16 cells only, so that four neighbouring
// lanes of a wavefront share a cell (lane-interleaved storage) and met on the
// same words.  At one stencil offset the 64 lanes then spread two to a bank
// pair.
constexpr int kTile2Row = 12, kTile2Copy = 112, kTile2Copies = 4;

// 2D3V Esirkepov currents (Projector2D2Order.cpp:131-188) of one particle
// into its copy of the tile, transverse weights and current factors
// factorised as esirkepov3d_fact; NT = 3: the node is unchanged on both axes
// (21 adds), NT = 4 otherwise (40).  The walk of all 65 points with a test for
// zero at each, on one copy of the tile, took 594 us a step for 8.4e6
// particles, this 490.
template <int NT>
__device__ inline void deposit2_tile(double *sJ, const Geom &g, const int *G0, const double *dold, const double *pnn,
                                     const int *ip, double cw, double crz)
{
    constexpr int NA = NT - 1;
    double S0[2][4], DS[2][4];
    int w0[2] = {1, 1};
#pragma unroll
    for (int d = 0; d < 2; ++d) {
        if constexpr (NT == 3) {
            double s1[3];
            spline<2>(dold[d], S0[d]);
            spline<2>(pnn[d] - (double)ip[d], s1);
#pragma unroll
            for (int m = 0; m < 3; ++m) DS[d][m] = s1[m] - S0[d][m];
        } else {
            esirkepov_window<2>(dold[d], pnn[d], ip[d], S0[d], DS[d], w0[d]);
        }
    }
    constexpr int C = kTile2Copies * kTile2Copy;
    double *t = sJ + (threadIdx.x & (kTile2Copies - 1)) * kTile2Copy + (ip[0] - G0[0] + w0[0]) * kTile2Row +
                (ip[1] - G0[1] + w0[1]);
    const double cr[2] = {cw * g.dxdt[0], cw * g.dxdt[1]};
    double A[2][NA], M[2][NT];
#pragma unroll
    for (int d = 0; d < 2; ++d) {
        double ps = 0.;
#pragma unroll
        for (int r = 0; r < NA; ++r) {
            ps += DS[d][r];
            A[d][r] = -cr[d] * ps;
        }
#pragma unroll
        for (int m = 0; m < NT; ++m) M[d][m] = fma(0.5, DS[d][m], S0[d][m]);
    }
#pragma unroll
    for (int r = 0; r < NA; ++r)
#pragma unroll
        for (int m = 0; m < NT; ++m) {
            atomicAdd(&t[(r + 1) * kTile2Row + m], A[0][r] * M[1][m]);
            atomicAdd(&t[C + m * kTile2Row + r + 1], A[1][r] * M[0][m]);
        }
    // Jz: crz (S0y (S0x + S1x / 2) + S1y (S0x / 2 + S1x))
#pragma unroll
    for (int m = 0; m < NT; ++m) {
        const double u = crz * fma(0.5, DS[0][m], 1.5 * S0[0][m]), v = crz * fma(1.5, S0[0][m], DS[0][m]);
#pragma unroll
        for (int q = 0; q < NT; ++q)
            atomicAdd(&t[2 * C + m * kTile2Row + q], fma(S0[1][q], u, (S0[1][q] + DS[1][q]) * v));
    }
}

// ---------------------------------------------------------------------------
// Fused particle kernel.
// ---------------------------------------------------------------------------
// One workgroup runs the particles of every species of the launch
// (specs[0..ns)) of cluster `cluster` against one field tile (and, with
// DEPOSIT, one J tile).  Uniform across the workgroup; returns at once for
// an empty cluster.
// Inlined into its kernels: left to itself the compiler calls it (order 4),
// and the call's stack frame lives in scratch memory.
template <int ND, int ORDER, bool DEPOSIT>
__device__ __attribute__((always_inline)) inline void fp_cluster(const Geom &g, const FpSpecies *__restrict__ specs,
                                                                 int ns, const GatherFields &F, const JPtrs &J,
                                                                 int *__restrict__ err, int cluster)
{
    using TL = Tile<ORDER>;
    constexpr int H = TL::H, GT = TL::GT, JT = TL::JT, S = TL::S;
    constexpr int GT3 = ND == 3 ? GT * GT * GT : GT * GT;
    // 3D field tile x-stride: 68 doubles instead of 8*8, so that the four
    // x-planes of cells a wavefront covers do not share LDS banks
    constexpr int GSX = ND == 3 ? (ORDER == 2 ? 68 : GT * GT) : GT, GF = ND == 3 ? GT * GSX : GT3;
    constexpr int JT3 = ND == 3 ? JT * JT * JT : JT * JT;
    // 3D order 2: J rows padded by one word, so that the tile atomics of a
    // wavefront meet fewer LDS bank conflicts (the strides of deposit3_tile)
    constexpr int JSY = ND == 3 && ORDER == 2 ? JT + 1 : JT, JSX = JT * JSY,
                  JSC = ND == 3 ? JT * JSX : kTile2Copies * kTile2Copy;
    __shared__ double sF[6 * GF];
    __shared__ double sJ[DEPOSIT ? 3 * JSC : 1];
    __shared__ int sHist[kMaxMerged][64];  // destination-cell counts of this cluster's own cells
    // particles whose node changes on some axis are deposited in a second pass
    // over this queue (old delta, new position in cells, charge weight, old node
    // relative to the cluster), so that the main loop runs the narrow stencil
    // with all lanes.  Order 4: a short queue, so that the
    // workgroup's LDS (field and J tiles of 10^3 and 11^3 points) stays within
    // 80 KB and two workgroups fit a CU.
    constexpr int QCAP = DEPOSIT ? (ORDER == 4 ? 12 : 96) : 1;
    __shared__ double sQ[QCAP][8];
    __shared__ int sQn;

    const Cluster cl = decode_cluster(g, cluster);
    int total = 0;
    for (int q = 0; q < ns; ++q)
        total += specs[q].cell_off[cl.gbase + g.cells_per_cl] - specs[q].cell_off[cl.gbase];
    if (total == 0) return;  // uniform across the workgroup

    // ---- stage E, B_m of the cluster + halo
    const double *src[6] = {F.Ex, F.Ey, F.Ez, F.Bx, F.By, F.Bz};
    for (int t = threadIdx.x; t < GT3; t += blockDim.x) {
        int a, b, c;
        if constexpr (ND == 3) {
            a = t / (GT * GT);
            b = (t / GT) % GT;
            c = t % GT;
        } else {
            a = t / GT;
            b = t % GT;
            c = 0;
        }
        const int gi = wrapi(cl.G0[0] - TL::GO + a, g.N[0]);
        const int gj = wrapi(cl.G0[1] - TL::GO + b, g.N[1]);
        const int gk = ND == 3 ? wrapi(cl.G0[2] - TL::GO + c, g.N[2]) : 0;
        const int idx = (gi * g.N[1] + gj) * g.N[2] + gk;  // fewer than 2^27 cells
        const int so = ND == 3 ? a * GSX + b * GT + c : t;
#pragma unroll
        for (int f = 0; f < 6; ++f) sF[f * GF + so] = src[f][idx];
    }
    if constexpr (DEPOSIT)
        for (int t = threadIdx.x; t < 3 * JSC; t += blockDim.x) sJ[t] = 0.;
    for (int t = threadIdx.x; t < kMaxMerged * 64; t += blockDim.x) sHist[t / 64][t % 64] = 0;
    if (threadIdx.x == 0) sQn = 0;
    __syncthreads();

    double pmin[3], pmax[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        pmin[d] = (double)cl.pc[d] * g.plen[d];
        pmax[d] = (double)(cl.pc[d] + 1) * g.plen[d];
    }

    // A wavefront takes 64 consecutive slots of the cluster's range; stored
    // lane-interleaved by the sort, they hold particles of different cells,
    // so the lanes' LDS atomics rarely hit the same address.
    for (int sid = 0; sid < ns; ++sid) {
    const FpSpecies &Sp = specs[sid];
    const SpeciesK &sp = Sp.k;
    const GPart A = glb(Sp.A), B = glb(Sp.B);
    const gptr<const int32_t> perm = glb(Sp.perm);
    const gptr<uint32_t> keys = glb(Sp.keys);
    int32_t *__restrict__ counts = Sp.counts;
    const gptr<int32_t> rank = glb(Sp.rank);
    const bool stay = Sp.stay != nullptr;
    const int lay = Sp.lay;
    const gptr<double> scratch = glb(Sp.scratch);
    const int64_t cap = Sp.cap;
    const int s = Sp.cell_off[cl.gbase], e = Sp.cell_off[cl.gbase + g.cells_per_cl];
    const int N = e - s;
    // consecutive slots per wavefront (lanes in different cells when the
    // sort stored the cluster lane-interleaved)
    for (int rel = threadIdx.x; rel < N; rel += blockDim.x) {
        const int jslot = s + rel;
        const int i = perm[jslot];
        double x[3] = {A.x[i], A.y[i], ND == 3 ? A.z[i] : 0.};
        double u[3] = {A.px[i], A.py[i], A.pz[i]};
        const double w = A.w[i];

        // ---- gather (Interpolator*::coeffs + compute)
        double pn[3], cp[3][5], cd[3][5], dold[3];
        int ip[3], id[3];
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            pn[d] = x[d] * g.dinv[d];
            ip[d] = (int)round(pn[d]);
            dold[d] = pn[d] - (double)ip[d];
            spline<ORDER>(dold[d], cp[d]);
            id[d] = (int)round(pn[d] + 0.5);
            spline<ORDER>(pn[d] - (double)id[d] + 0.5, cd[d]);
        }
        int lp[3], ld[3];
        bool inside = true;
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            lp[d] = ip[d] - (cl.G0[d] - TL::GO);
            ld[d] = id[d] - (cl.G0[d] - TL::GO);
            inside &= lp[d] >= H && lp[d] <= GT - 1 - H && ld[d] >= H && ld[d] <= GT - 1 - H;
        }
        if (!inside) {
            // not in this cluster (corrupt state): leave it untouched, flag it
            atomicOr(err, 1);
            keys[jslot] = ((stay ? kPlaceAtomic : 13u) << 27) | (uint32_t)(cl.gbase);
            atomicAdd(&counts[cl.gbase], 1);
            B.x[jslot] = x[0];
            B.y[jslot] = x[1];
            if constexpr (ND == 3) B.z[jslot] = x[2];
            B.px[jslot] = u[0];
            B.py[jslot] = u[1];
            B.pz[jslot] = u[2];
            B.w[jslot] = w;
            if constexpr (!DEPOSIT) {
                for (int d = 0; d < 3; ++d) {
                    scratch[d * cap + jslot] = d < ND ? x[d] : 0.;
                    scratch[(3 + d) * cap + jslot] = d < ND ? x[d] : 0.;
                }
                scratch[6 * cap + jslot] = 1.0;
            }
            continue;
        }
        // DEPOSIT (the atomic form, whose sums have no fixed order): the fused
        // gather and push; else the reference's association order, bit for bit
        double Ep[3], Bp[3];
        auto gather = [&](int f, int dual) {
            const double *c[3];
            int l[3];
#pragma unroll
            for (int d = 0; d < ND; ++d) {
                c[d] = (dual >> d) & 1 ? cd[d] : cp[d];
                l[d] = (dual >> d) & 1 ? ld[d] : lp[d];
            }
            if constexpr (ND == 3 && DEPOSIT) return gather3_fused<H, GT, GSX>(c[0], c[1], c[2], sF + f * GF, l[0], l[1], l[2]);
            else if constexpr (ND == 3) return gather3<H, GT, GSX>(c[0], c[1], c[2], sF + f * GF, l[0], l[1], l[2]);
            else if constexpr (DEPOSIT) return gather2_fused<H, GT>(c[0], c[1], sF + f * GF, l[0], l[1]);
            else return gather2<H, GT>(c[0], c[1], sF + f * GF, l[0], l[1]);
        };
        Ep[0] = gather(0, 1);
        Ep[1] = gather(1, 2);
        Ep[2] = gather(2, 4);
        Bp[0] = gather(3, 6);
        Bp[1] = gather(4, 5);
        Bp[2] = gather(5, 3);

        // ---- push
        double dxp[3], invgf;
        if constexpr (DEPOSIT) boris_fused(sp.qmh, g.dt, Ep, Bp, u, dxp, invgf);
        else boris(sp.qmh, g.dt, Ep, Bp, u, dxp, invgf);
        double xn[3];
#pragma unroll
        for (int d = 0; d < ND; ++d) xn[d] = x[d] + dxp[d];

        // ---- boundary tag, periodic wrap, destination key
        int m[3] = {0, 0, 0}, dpc[3] = {cl.pc[0], cl.pc[1], cl.pc[2]};
        double xw[3] = {xn[0], ND > 1 ? xn[1] : 0., ND > 2 ? xn[2] : 0.};
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            if (xn[d] < pmin[d]) m[d] = -1;
            else if (xn[d] >= pmax[d]) m[d] = 1;
            dpc[d] = wrapi(cl.pc[d] + m[d], g.npatch[d]);
            if (m[d] == -1 && cl.pc[d] == 0 && xw[d] < 0.) xw[d] += g.xmax[d];
            if (m[d] == 1 && cl.pc[d] == g.npatch[d] - 1 && xw[d] >= g.xmax[d]) xw[d] -= g.xmax[d];
        }
        const int dp = (dpc[0] * g.npatch[1] + dpc[1]) * g.npatch[2] + dpc[2];
        const uint32_t gkey = (uint32_t)((int64_t)dp * g.cpp + cell_key<ND>(g, dpc, xw));
        // histogram of destination cells for the sort: own-cluster cells in
        // LDS, particles leaving the cluster straight to the global counts.
        // Top key bits: the direction of motion, or with `stay` the rank
        // among this cluster's stayers of the cell (placed by the sort).
        uint32_t tag = (uint32_t)((m[0] + 1) * 9 + (m[1] + 1) * 3 + (m[2] + 1));
        const int64_t rel_cell = (int64_t)gkey - cl.gbase;
        if (rel_cell >= 0 && rel_cell < g.cells_per_cl) {
            if (stay) {
                const int r = atomicAdd(&sHist[sid][rel_cell], 1);
                tag = r < (int)kPlaceMax ? (uint32_t)r : kPlaceAtomic;
            } else {
                atomicAdd(&sHist[sid][rel_cell], 1);
            }
        } else {
            atomicAdd(&counts[gkey], 1);
            if (stay) tag = kPlaceAtomic;
            // cell-major position of this input particle, the tie-break of
            // the canonical in-cell order at the next sort: only read for
            // the particles that leave their cluster (the sort computes it
            // for the others)
            if (rank) rank[jslot] = s + (lay ? cluster_rank(rel, N) : rel);  // layouts 0 and 1 (FP64 form)
        }
        keys[jslot] = (tag << 27) | gkey;
        B.x[jslot] = xw[0];
        B.y[jslot] = xw[1];
        if constexpr (ND == 3) B.z[jslot] = xw[2];
        B.px[jslot] = u[0];
        B.py[jslot] = u[1];
        B.pz[jslot] = u[2];
        B.w[jslot] = w;

        if constexpr (!DEPOSIT) {
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                scratch[d * cap + jslot] = d < ND ? x[d] : 0.;
                scratch[(3 + d) * cap + jslot] = d < ND ? xn[d] : 0.;
            }
            scratch[6 * cap + jslot] = invgf;
        } else {
            // ---- Esirkepov currents into the LDS tile
            const double cw = sp.cw_scale * w;
            const double crz = ND == 2 ? cw * kThird * u[2] * invgf : 0.;
            double pnn[3];
            int moved = 0;
#pragma unroll
            for (int d = 0; d < ND; ++d) {
                pnn[d] = xn[d] * g.dinv[d];
                moved |= (int)round(pnn[d]) - ip[d];
            }
            if (moved == 0) {
                if constexpr (ND == 3) deposit3_tile<ORDER, ORDER + 1>(sJ, g, cl.G0, dold, pnn, ip, cw);
                else deposit2_tile<3>(sJ, g, cl.G0, dold, pnn, ip, cw, crz);
            }
            const uint64_t gm = __ballot(moved != 0);
            if (gm) {
                const int lane = threadIdx.x & 63;
                const int leader = __ffsll((unsigned long long)gm) - 1;
                int base = 0;
                if (lane == leader) base = atomicAdd(&sQn, __popcll(gm));
                base = __shfl(base, leader, 64);
                if (moved != 0) {
                    const int pos = base + __popcll(gm & ((1ull << lane) - 1));
                    if (pos < QCAP) {
                        int packed = 0;
#pragma unroll
                        for (int d = 0; d < ND; ++d) {
                            sQ[pos][d] = dold[d];
                            sQ[pos][3 + d] = pnn[d];
                            packed |= (ip[d] - cl.G0[d]) << (4 * d);
                        }
                        if constexpr (ND == 2) sQ[pos][2] = crz;
                        sQ[pos][6] = cw;
                        sQ[pos][7] = (double)packed;
                    } else if constexpr (ND == 3) {
                        deposit3_tile<ORDER, ORDER + 2>(sJ, g, cl.G0, dold, pnn, ip, cw);
                    } else {
                        deposit2_tile<4>(sJ, g, cl.G0, dold, pnn, ip, cw, crz);
                    }
                }
            }
        }
    }

    }  // species

    __syncthreads();
    for (int t = threadIdx.x; t < ns * 64; t += blockDim.x) {
        const int c = t % 64 < g.cells_per_cl ? sHist[t / 64][t % 64] : 0;
        if (c) {
            const FpSpecies &S = specs[t / 64];
            atomicAdd(&S.counts[cl.gbase + t % 64], c);
            if (S.stay) S.stay[cl.gbase + t % 64] = (uint8_t)(c < (int)kPlaceMax ? c : (int)kPlaceMax);
        }
    }
    if constexpr (DEPOSIT) {
        const int nq = sQn < QCAP ? sQn : QCAP;
        for (int t = threadIdx.x; t < nq; t += blockDim.x) {
            const double dold[3] = {sQ[t][0], sQ[t][1], sQ[t][2]};
            const double pnn[3] = {sQ[t][3], sQ[t][4], sQ[t][5]};
            const int packed = (int)sQ[t][7];
            const int ip[3] = {cl.G0[0] + (packed & 15), cl.G0[1] + ((packed >> 4) & 15),
                               cl.G0[2] + ((packed >> 8) & 15)};
            if constexpr (ND == 3) deposit3_tile<ORDER, ORDER + 2>(sJ, g, cl.G0, dold, pnn, ip, sQ[t][6]);
            else deposit2_tile<4>(sJ, g, cl.G0, dold, pnn, ip, sQ[t][6], sQ[t][2]);
        }
        __syncthreads();
        // one tile position per thread and pass, its grid index computed once
        // for the three components (32-bit: the engine holds fewer than 2^27
        // cells)
        const gptr<double> dstJ[3] = {glb(J.Jx), glb(J.Jy), glb(J.Jz)};
        for (int r = threadIdx.x; r < JT3; r += blockDim.x) {
            int a, b, k;
            if constexpr (ND == 3) {
                a = r / (JT * JT);
                b = (r / JT) % JT;
                k = r % JT;
            } else {
                a = r / JT;
                b = r % JT;
                k = 0;
            }
            const int gi = wrapi(cl.G0[0] - TL::JO + a, g.N[0]);
            const int gj = wrapi(cl.G0[1] - TL::JO + b, g.N[1]);
            const int gk = ND == 3 ? wrapi(cl.G0[2] - TL::JO + k, g.N[2]) : 0;
            const int idx = (gi * g.N[1] + gj) * g.N[2] + gk;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                double v;
                if constexpr (ND == 3) {
                    v = sJ[c * JSC + a * JSX + b * JSY + k];
                } else {
                    v = 0.;
#pragma unroll
                    for (int q = 0; q < kTile2Copies; ++q) v += sJ[c * JSC + q * kTile2Copy + a * kTile2Row + b];
                }
                if (v != 0.) unsafeAtomicAdd((double *)(dstJ[c] + idx), v);
            }
        }
    }
}

// One workgroup per cluster of the grid (xcd: XCD-aware cluster order).
template <int ND, int ORDER, bool DEPOSIT>
__global__ void __launch_bounds__(ND == 3 && ORDER == 4 ? 256 : 512, ND == 3 && ORDER == 4 ? 2 : 3)
k_particles(Geom g, const FpSpecies *__restrict__ specs, int ns, GatherFields F, JPtrs J, int *__restrict__ err,
            int xcd)
{
    fp_cluster<ND, ORDER, DEPOSIT>(g, specs, ns, F, J, err, xcd ? xcd_cluster(blockIdx.x, gridDim.x) : blockIdx.x);
}

// Persistent form: a grid sized to the resident workgroups pulls clusters
// from the work list (the non-empty clusters, wcount[0] of them) through the
// queue head wcount[1]; every workgroup leaves once the list is exhausted.
template <int ND, int ORDER, bool DEPOSIT>
__global__ void __launch_bounds__(ND == 3 && ORDER == 4 ? 256 : 512, ND == 3 && ORDER == 4 ? 2 : 3)
k_particles_list(Geom g, const FpSpecies *__restrict__ specs, int ns, GatherFields F, JPtrs J, int *__restrict__ err,
                 const int *__restrict__ work, int *__restrict__ wcount)
{
    __shared__ int sItem;
    const int nwork = wcount[0];
    for (;;) {
        __syncthreads();  // the previous cluster is done with the LDS tiles
        if (threadIdx.x == 0) sItem = atomicAdd(&wcount[1], 1);
        __syncthreads();
        const int item = sItem;
        if (item >= nwork) break;
        fp_cluster<ND, ORDER, DEPOSIT>(g, specs, ns, F, J, err, work[item]);
    }
}

// Work list of the clusters holding particles of any species of the launch
// (order irrelevant); wcount[0..1] must be zero.
__global__ void k_fp_worklist(Geom g, const FpSpecies *__restrict__ specs, int ns, int *__restrict__ work,
                              int *__restrict__ wcount)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    int total = 0;
    if (c < g.npatches * g.clpp) {
        const int64_t gbase = (int64_t)(c / g.clpp) * g.cpp + (int64_t)(c % g.clpp) * g.cells_per_cl;
        for (int q = 0; q < ns; ++q) total += specs[q].cell_off[gbase + g.cells_per_cl] - specs[q].cell_off[gbase];
    }
    const uint64_t m = __ballot(total > 0);
    if (!m) return;
    const int lane = threadIdx.x & 63;
    const int leader = __ffsll((unsigned long long)m) - 1;
    int base = 0;
    if (lane == leader) base = atomicAdd(&wcount[0], __popcll(m));
    base = __shfl(base, leader, 64);
    if (total > 0) work[base + __popcll(m & ((1ull << lane) - 1))] = c;
}

// ---------------------------------------------------------------------------
// Deterministic deposit (reference order) into per-patch ghosted J.
// ---------------------------------------------------------------------------
struct PJLayout {
    int dims[3][3];   // dims of Jx, Jy, Jz
    int64_t off[3];   // offsets of Jx, Jy, Jz inside a patch block
    int64_t per;      // doubles per patch
};

__host__ __device__ inline PJLayout pj_layout(const Geom &g)
{
    PJLayout L;
    int np[3];
    for (int d = 0; d < 3; ++d) np[d] = d < g.nd ? g.n[d] + 2 * g.os + 1 : 1;
    for (int c = 0; c < 3; ++c)
        for (int d = 0; d < 3; ++d) L.dims[c][d] = np[d] + ((d == c && d < g.nd) ? 1 : 0);
    int64_t o = 0;
    for (int c = 0; c < 3; ++c) {
        L.off[c] = o;
        o += (int64_t)L.dims[c][0] * L.dims[c][1] * L.dims[c][2];
    }
    L.per = o;
    return L;
}

// 3D: one workgroup per tile of 4^3 points of a patch's ghosted arrays
// (ordered_deposit.h).  A cluster q along an axis reaches the tiles q, q + 1
// and q + 2, so a tile walks the clusters t - 2 .. t per axis in the patch's
// (cluster-major) particle order; the clusters of one z row are contiguous.
// Every point is written once, so the arrays need not be cleared.  32^3
// cells, 8^3 patches, 524,288 particles: 23.2 ms with one wavefront per
// patch, 1.4 ms here.
template <int ORDER>
__global__ void __launch_bounds__(kOrdThreads)
k_det_deposit3(Geom g, const DetSpecies *__restrict__ species, int nspecies, double *__restrict__ pj, int *__restrict__ err)
{
    __shared__ OrdShared<ORDER> sh;
    const PJLayout L = pj_layout(g);
    int nt[3];
    for (int d = 0; d < 3; ++d) nt[d] = (g.n[d] + 2 * g.os + 2 + 3) / 4;
    // tile-major: a tile's work depends on its place in the patch (the inner
    // ones meet the most clusters), and workgroups go round-robin to the 8
    // XCDs, so patch-major order would put the same tiles of all patches on
    // one XCD (measured 3.8 ms)
    const int p = blockIdx.x % g.npatches, t = blockIdx.x / g.npatches;
    int tc[3] = {t / (nt[1] * nt[2]), (t / nt[2]) % nt[1], t % nt[2]};
    // and the inner tiles first, so that the longest walks do not start last
    // (1,592 us in index order, 1,402 so)
    for (int d = 0; d < 3; ++d) tc[d] = tc[d] == nt[d] - 1 ? tc[d] : (tc[d] == nt[d] - 2 ? 0 : tc[d] + 1);
    const int pc[3] = {p / (g.npatch[1] * g.npatch[2]), (p / g.npatch[2]) % g.npatch[1], p % g.npatch[2]};
    int t0[3], dom[3], c0[3], c1[3];
    for (int d = 0; d < 3; ++d) {
        t0[d] = 4 * tc[d];
        dom[d] = pc[d] * g.n[d] - g.os;
        c0[d] = tc[d] - 2 < 0 ? 0 : tc[d] - 2;
        c1[d] = tc[d] < g.ncl[d] - 1 ? tc[d] : g.ncl[d] - 1;
    }
    const int lane = threadIdx.x & 63, c = threadIdx.x >> 6;
    const int pt[3] = {lane >> 4, (lane >> 2) & 3, lane & 3};
    const double dxdt[3] = {g.dx[0] / g.dt, g.dx[1] / g.dt, g.dx[2] / g.dt};
    double acc = 0.;
    for (int s = 0; s < nspecies; ++s) {
        const DetSpecies ds = species[s];
        auto load = [&](int64_t j) {
            OrdParticle q;
            q.ok = true;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const double pn = ds.scratch[d * ds.cap + j] * g.dinv[d];
                q.node[d] = (int)round(pn);
                q.io[d] = q.node[d] - dom[d];
                q.dold[d] = pn - (double)q.node[d];
                q.pnn[d] = ds.scratch[(3 + d) * ds.cap + j] * g.dinv[d];
                const int step = (int)round(q.pnn[d]) - q.node[d];
                // old node within the patch, move below one cell
                q.ok &= q.io[d] >= g.os && q.io[d] <= g.os + g.n[d] && step >= -1 && step <= 1;
            }
            q.cw = ds.sp.cw_scale * ds.w[j];
            if (!q.ok) atomicOr(err, 1);
            return q;
        };
        int pending = 0;
        for (int a = c0[0]; a <= c1[0]; ++a)
            for (int b = c0[1]; b <= c1[1]; ++b) {
                const int64_t row = (int64_t)p * g.cpp + (int64_t)(a * g.ncl[1] + b) * g.ncl[2] * 64;
                ordered_range<ORDER>(sh, pending, ds.cell_off[row + c0[2] * 64], ds.cell_off[row + (c1[2] + 1) * 64],
                                     a == c1[0] && b == c1[1], t0, pt, dxdt, load, acc);
            }
    }
    int idx[3];
    bool in = true;
    for (int d = 0; d < 3; ++d) {
        idx[d] = t0[d] + pt[d];
        in &= idx[d] < L.dims[c][d];
    }
    if (in) pj[p * L.per + L.off[c] + ((int64_t)idx[0] * L.dims[c][1] + idx[1]) * L.dims[c][2] + idx[2]] = acc;
}

// 2D: one wavefront per patch.  Each particle's contributions are split over
// the lanes by (component, transverse column); every J point receives at most
// one add per particle, and particles are processed strictly in order: the
// adds are L2 atomics and the barrier after each particle waits for them, so
// every J point sums its contributions in the patch's particle order.
__global__ void __launch_bounds__(64) k_det_deposit2(Geom g, const DetSpecies *__restrict__ species,
                                                     int nspecies, double *__restrict__ pj, int *__restrict__ err)
{
    constexpr int ND = 2, ORDER = 2;
    const int p = blockIdx.x;
    const PJLayout L = pj_layout(g);
    double *Jc[3] = {pj + p * L.per + L.off[0], pj + p * L.per + L.off[1], pj + p * L.per + L.off[2]};
    const int pc[2] = {p / g.npatch[1], p % g.npatch[1]};
    int dom[2];
    for (int d = 0; d < 2; ++d) dom[d] = pc[d] * g.n[d] - g.os;
    const int lane = threadIdx.x;

    for (int s = 0; s < nspecies; ++s) {
        const DetSpecies ds = species[s];
        const int a0 = ds.cell_off[(int64_t)p * g.cpp], a1 = ds.cell_off[(int64_t)(p + 1) * g.cpp];
        for (int j = a0; j < a1; ++j) {
            double xo[2], xn[2];
            for (int d = 0; d < 2; ++d) {
                xo[d] = ds.scratch[d * ds.cap + j];
                xn[d] = ds.scratch[(3 + d) * ds.cap + j];
            }
            const double cw = ds.sp.cw_scale * ds.w[j];
            double S0[3][7], S1[3][7], DS[3][7];
            int io[3];
            bool ok = true;
            for (int d = 0; d < ND; ++d) {
                const double pn = xo[d] * g.dinv[d];
                const int ipo = (int)round(pn);
                io[d] = ipo - dom[d];
                const int ipn = (int)round(xn[d] * g.dinv[d]);
                // old node within the patch, move below one cell
                ok &= io[d] >= g.os && io[d] <= g.os + g.n[d] && ipn - ipo >= -1 && ipn - ipo <= 1;
                esirkepov_shapes<ORDER>(pn - (double)ipo, xn[d] * g.dinv[d], ipo, S0[d], S1[d], DS[d]);
            }
            if (!ok) {
                if (lane == 0) atomicOr(err, 1);
                __syncthreads();
                continue;
            }
            const double crx = cw * (g.dx[0] / g.dt), cry = cw * (g.dx[1] / g.dt);
            const double crz = cw * kThird * ds.pz[j] * ds.scratch[6 * ds.cap + j];
            // lanes: 0..4 Jx columns j, 5..9 Jy rows i, 10..34 Jz points
            if (lane < 5) {
                const int jj = lane;
                double acc = 0.;
                for (int i = 1; i < 5; ++i) {
                    if (jj == 0) acc -= crx * DS[0][i - 1] * (0.5 * DS[1][0]);
                    else acc -= crx * DS[0][i - 1] * (S0[1][jj] + 0.5 * DS[1][jj]);
                    const int ii = io[0] - 2 + i, yy = io[1] - 2 + jj;
                    unsafeAtomicAdd(&Jc[0][(int64_t)ii * L.dims[0][1] + yy], acc);
                }
            } else if (lane < 10) {
                const int ii = lane - 5;
                const double ty = S0[0][ii] + 0.5 * DS[0][ii];
                double acc = 0.;
                for (int jj = 1; jj < 5; ++jj) {
                    acc -= cry * DS[1][jj - 1] * ty;
                    const int xx = io[0] - 2 + ii, yy = io[1] - 2 + jj;
                    unsafeAtomicAdd(&Jc[1][(int64_t)xx * L.dims[1][1] + yy], acc);
                }
            } else if (lane < 35) {
                const int ii = (lane - 10) / 5, jj = (lane - 10) % 5;
                double h2, h3;
                if (ii == 0) {
                    h2 = 0.5 * S1[0][0];
                    h3 = S1[0][0];
                } else {
                    h2 = 0.5 * S1[0][ii] + S0[0][ii];
                    h3 = 0.5 * S0[0][ii] + S1[0][ii];
                }
                const double v = jj == 0 ? crz * (S1[1][0] * h3) : crz * (S0[1][jj] * h2 + S1[1][jj] * h3);
                const int xx = io[0] - 2 + ii, yy = io[1] - 2 + jj;
                unsafeAtomicAdd(&Jc[2][(int64_t)xx * L.dims[2][1] + yy], v);
            }
            __syncthreads();
        }
    }
}

// Ghost sum along dimension d for the three components:
// low[n + a] += this[a]; this[a] = low[n + a], a in [0, 1 + 2*os + dual).
// The component is the workgroup's (blockIdx.y), the patch too (`blocks` of
// them per slab), so that extents and offsets are scalars: picked per thread
// they were arrays in scratch memory, 18 us a pass over 8 patches of 32^3
// cells against 5.5.
__global__ void __launch_bounds__(256) k_ghost_sum(Geom g, int d, int blocks, double *__restrict__ pj)
{
    const int c = blockIdx.y, p = blockIdx.x / blocks;
    int r = (int)(blockIdx.x - p * blocks) * 256 + threadIdx.x;
    int np[3], dm[3], ext[3];
    int64_t off = 0, per = 0;
#pragma unroll
    for (int e = 0; e < 3; ++e) {
        np[e] = e < g.nd ? g.n[e] + 2 * g.os + 1 : 1;
        dm[e] = np[e] + (e == c && e < g.nd ? 1 : 0);
        ext[e] = e == d ? 1 + 2 * g.os + (c == d ? 1 : 0) : dm[e];
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        int64_t sz = 1;
#pragma unroll
        for (int e = 0; e < 3; ++e) sz *= np[e] + (e == q && e < g.nd ? 1 : 0);
        if (q < c) off += sz;
        per += sz;
    }
    const int row = ext[1] * ext[2];
    const int i = r / row;
    if (i >= ext[0]) return;
    r -= i * row;
    const int j = r / ext[2], k = r - j * ext[2];
    int pc[3] = {p / (g.npatch[1] * g.npatch[2]), (p / g.npatch[2]) % g.npatch[1], p % g.npatch[2]};
#pragma unroll
    for (int e = 0; e < 3; ++e)
        if (e == d) pc[e] = wrapi(pc[e] - 1, g.npatch[e]);
    const int lp = (pc[0] * g.npatch[1] + pc[1]) * g.npatch[2] + pc[2];
    const int64_t b = ((int64_t)i * dm[1] + j) * dm[2] + k;
    const int64_t step = d == 0 ? (int64_t)dm[1] * dm[2] : (d == 1 ? dm[2] : 1);
    const int nd = d == 0 ? g.n[0] : (d == 1 ? g.n[1] : g.n[2]);
    double *me = pj + p * per + off, *lo = pj + lp * per + off;
    const int64_t a = b + nd * step;
    const double sum = lo[a] + me[b];
    lo[a] = sum;
    me[b] = sum;
}

// Global J[g] = owning patch's ghost-summed value.
__global__ void k_fold_interior(Geom g, const double *__restrict__ pj, JPtrs J)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= g.ncells) return;
    const PJLayout L = pj_layout(g);
    const int gk = (int)(t % g.N[2]);
    const int gj = (int)((t / g.N[2]) % g.N[1]);
    const int gi = (int)(t / ((int64_t)g.N[2] * g.N[1]));
    const int gg[3] = {gi, gj, gk};
    int pc[3], l[3];
    for (int d = 0; d < 3; ++d) {
        pc[d] = gg[d] / g.n[d];
        l[d] = gg[d] - pc[d] * g.n[d] + (d < g.nd ? g.os : 0);
    }
    const int p = (pc[0] * g.npatch[1] + pc[1]) * g.npatch[2] + pc[2];
    double *dst[3] = {J.Jx, J.Jy, J.Jz};
    for (int c = 0; c < 3; ++c) {
        const int *dm = L.dims[c];
        dst[c][t] = pj[(int64_t)p * L.per + L.off[c] + ((int64_t)l[0] * dm[1] + l[1]) * dm[2] + l[2]];
    }
}

}  // namespace

int64_t patch_j_size(const Geom &g) { return pj_layout(g).per; }

void launch_particles(const Geom &g, const FpSpecies *specs, int ns, const GatherFields &F, const JPtrs &J,
                      bool deposit, int *err, int threads, bool xcd, int persistent_blocks, int *work, int *wcount,
                      hipStream_t st)
{
    if (threads != 64 && threads != 128 && threads != 256 && threads != 512)
        throw Error(-1, "particle-kernel workgroup size must be 64, 128, 256 or 512");
    if (threads > particle_max_threads(g, false))
        throw Error(-1, "workgroup size above the particle kernel's limit for this geometry and order");
    if (ns < 1 || ns > kMaxMerged) throw Error(-1, "bad species count of a merged particle launch");
    const int nb = g.npatches * g.clpp;
    const dim3 block(threads);
    if (persistent_blocks > 0) {
        // the work list, then as many workgroups as fit at once
        launch_fill_i32(wcount, 2, 0, st);
        hipLaunchKernelGGL(k_fp_worklist, dim3((nb + 255) / 256), dim3(256), 0, st, g, specs, ns, work, wcount);
        SMI_LAUNCH_CHECK();
    }
    const dim3 grid(persistent_blocks > 0 ? std::min(nb, persistent_blocks) : nb);
#define SMI_PK(ND, O, D)                                                                                          \
    do {                                                                                                          \
        if (persistent_blocks > 0)                                                                                \
            hipLaunchKernelGGL((k_particles_list<ND, O, D>), grid, block, 0, st, g, specs, ns, F, J, err,         \
                               (const int *)work, wcount);                                                         \
        else                                                                                                      \
            hipLaunchKernelGGL((k_particles<ND, O, D>), grid, block, 0, st, g, specs, ns, F, J, err, xcd ? 1 : 0); \
    } while (0)
    if (g.nd == 3 && g.order == 2) {
        if (deposit) SMI_PK(3, 2, true);
        else SMI_PK(3, 2, false);
    } else if (g.nd == 3 && g.order == 4) {
        if (deposit) SMI_PK(3, 4, true);
        else SMI_PK(3, 4, false);
    } else if (g.nd == 2 && g.order == 2) {
        if (deposit) SMI_PK(2, 2, true);
        else SMI_PK(2, 2, false);
    } else {
        throw Error(-1, "unsupported (ndim, order) for the particle kernel");
    }
#undef SMI_PK
    SMI_LAUNCH_CHECK();
}

int fp_persistent_blocks(const Geom &g, bool deposit, int threads)
{
    int dev = 0, cus = 0, per_cu = 0;
    SMI_HIP(hipGetDevice(&dev));
    SMI_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const void *fn = nullptr;
    if (g.nd == 3 && g.order == 2)
        fn = deposit ? (const void *)k_particles_list<3, 2, true> : (const void *)k_particles_list<3, 2, false>;
    else if (g.nd == 3 && g.order == 4)
        fn = deposit ? (const void *)k_particles_list<3, 4, true> : (const void *)k_particles_list<3, 4, false>;
    else
        fn = deposit ? (const void *)k_particles_list<2, 2, true> : (const void *)k_particles_list<2, 2, false>;
    SMI_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, threads, 0));
    return std::max(1, cus * std::max(per_cu, 1));
}

int particle_max_threads(const Geom &g, bool mixed)
{
    // the 3D order-4 FP64 kernel needs the full register file of one wave
    return !mixed && g.nd == 3 && g.order == 4 ? 256 : 512;
}

void launch_det_deposit(const Geom &g, const DetSpecies *species, int nspecies, double *pj, int *err,
                        hipStream_t st)
{
    int64_t tiles = 1;
    for (int d = 0; d < 3; ++d) tiles *= (g.n[d] + 2 * g.os + 2 + 3) / 4;
    const dim3 grid((unsigned)(tiles * g.npatches)), block(kOrdThreads);
    if (g.nd == 3 && g.order == 2) {
        hipLaunchKernelGGL(k_det_deposit3<2>, grid, block, 0, st, g, species, nspecies, pj, err);
    } else if (g.nd == 3 && g.order == 4) {
        hipLaunchKernelGGL(k_det_deposit3<4>, grid, block, 0, st, g, species, nspecies, pj, err);
    } else if (g.nd == 2 && g.order == 2) {
        launch_fill(pj, pj_layout(g).per * g.npatches, 0.0, st);
        hipLaunchKernelGGL(k_det_deposit2, dim3(g.npatches), dim3(64), 0, st, g, species, nspecies, pj, err);
    } else {
        throw Error(-1, "unsupported (ndim, order) for the deterministic deposit");
    }
    SMI_LAUNCH_CHECK();
}

void launch_ghost_sum(const Geom &g, double *pj, hipStream_t st)
{
    const PJLayout L = pj_layout(g);
    for (int d = 0; d < g.nd; ++d) {
        int64_t slab = 0;  // the largest component's
        for (int c = 0; c < 3; ++c) {
            const int gsp = 1 + 2 * g.os + (c == d ? 1 : 0);
            int64_t sz = 1;
            for (int e = 0; e < 3; ++e) sz *= (e == d ? gsp : L.dims[c][e]);
            slab = sz > slab ? sz : slab;
        }
        const int64_t blocks = (slab + 255) / 256;
        hipLaunchKernelGGL(k_ghost_sum, dim3((unsigned)(blocks * g.npatches), 3), dim3(256), 0, st, g, d, (int)blocks,
                           pj);
        SMI_LAUNCH_CHECK();
    }
}

void launch_ghost_sum_and_fold(const Geom &g, double *pj, const JPtrs &J, hipStream_t st)
{
    launch_ghost_sum(g, pj, st);
    hipLaunchKernelGGL(k_fold_interior, dim3((unsigned)((g.ncells + 255) / 256)), dim3(256), 0, st, g,
                       (const double *)pj, J);
    SMI_LAUNCH_CHECK();
}

}  // namespace smi
