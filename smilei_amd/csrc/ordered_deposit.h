// ordered_deposit.h -- Esirkepov currents summed in particle order (3D).
//
// Every point of a ghosted patch array is the sum of its particles'
// contributions in the order the CPU operator adds them, so two points are
// independent and only the adds of one point are a chain.  One workgroup owns
// a tile of 4^3 points of the three components, one wavefront per component
// and one lane per point, its sum in a register.  The workgroup walks the
// particles whose stencil can reach the tile, in order: 192 at a time are
// tested and the ones that reach the tile appended to a list in LDS; for each
// 64 of the list the three wavefronts build the shapes (one axis each) in LDS
// and every lane then adds the particles' contributions to its point, one
// after the other.  The contributions round exactly as esirkepov3d's.
//
// What bounds it is the lanes' arithmetic (about 45 instructions per particle,
// tile and component); a particle reaches 5 to 8 tiles.  Adding a particle's
// contributions to L2 with atomics, a barrier after each particle, takes one
// wavefront per patch about 2 microseconds a particle instead.
#pragma once

#include "pic_device.h"

namespace smi {
namespace dev {

constexpr int kOrdThreads = 192, kOrdBatch = 64;

// A particle as the ordered deposit reads it.
struct OrdParticle {
    double dold[3];  // old offset from the old node
    double pnn[3];   // new position in cells (global)
    int node[3];     // old node, global
    int io[3];       // old node's index in the patch array
    double cw;       // charge weight
    bool ok;
};

template <int ORDER>
struct OrdShared {
    static constexpr int S = ORDER + 3;
    // (S0, DS) of axis d at stencil entry m; rows padded so that the entries
    // of one particle, which the lanes of a wavefront read together, lie in
    // different banks
    double2 sd[3][S][kOrdBatch + 1];
    double pre[3][S - 1][kOrdBatch];   // prefix factors of component c (DS; times the current factor at order 4)
    double cr[3][kOrdBatch];
    int base[kOrdBatch];               // stencil origin relative to the tile, 5 bits per axis, offset by 16
    int list[kOrdBatch + kOrdThreads];
    int wcount[kOrdThreads / 64];
};

template <int ORDER, int C>
__device__ inline void ordered_add(const OrdShared<ORDER> &sh, int count, const int *pt, double &acc)
{
    constexpr int S = ORDER + 3, BX = (C + 1) % 3, EX = (C + 2) % 3;
    // four particles at a time, straight-line: their LDS reads overlap (the
    // entries after the last particle of a batch hit nothing)
    for (int m0 = 0; m0 < count; m0 += 4) {
        double val[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int m = m0 + k;
            const int pk = sh.base[m];
            const int o[3] = {(pk & 31) - 16, ((pk >> 5) & 31) - 16, ((pk >> 10) & 31) - 16};
            const int r = pt[C] - o[C], b = pt[BX] - o[BX], e = pt[EX] - o[EX];
            const bool hit = r >= 1 && r < S && b >= 0 && b < S && e >= 0 && e < S;
            const double2 vb = sh.sd[BX][b < 0 ? 0 : (b < S ? b : S - 1)][m];
            const double2 ve = sh.sd[EX][e < 0 ? 0 : (e < S ? e : S - 1)][m];
            const double W = vb.x * ve.x + 0.5 * vb.y * ve.x + 0.5 * ve.y * vb.x + kThird * vb.y * ve.y;
            const double t = ORDER == 2 ? sh.cr[C][m] * W : W;
            double v = 0.;
#pragma unroll
            for (int q = 0; q < S - 1; ++q) {
                const double n = v - sh.pre[C][q][m] * t;
                v = q < r ? n : v;
            }
            val[k] = hit ? v : 0.;
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) acc += val[k];
    }
}

// Particles [beg, end) in order; pending particles stay in the list for the
// next range.  load(j) gives particle j; dxdt = dx / dt.
template <int ORDER, class Load>
__device__ inline void ordered_range(OrdShared<ORDER> &sh, int &pending, int64_t beg, int64_t end, bool last,
                                     const int *t0, const int *pt, const double *dxdt, Load load, double &acc)
{
    constexpr int H = ORDER / 2, S = ORDER + 3;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int64_t j0 = beg; j0 < end || last; j0 += kOrdThreads) {
        const int64_t j = j0 + threadIdx.x;
        bool reach = false;
        if (j < end) {
            const OrdParticle p = load(j);
            reach = p.ok;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                // S0 and DS are zero at the first stencil entry unless the
                // node moves down
                const int lo = p.io[d] - (H + 1) + ((int)round(p.pnn[d]) < p.node[d] ? 0 : 1);
                reach &= lo <= t0[d] + 3 && p.io[d] + H + 1 >= t0[d];
            }
        }
        const uint64_t mask = __ballot(reach);
        if (lane == 0) sh.wcount[wave] = __popcll(mask);
        __syncthreads();
        int at = pending, total = 0;
#pragma unroll
        for (int w = 0; w < kOrdThreads / 64; ++w) {
            const int k = __builtin_amdgcn_readfirstlane(sh.wcount[w]);
            if (w < wave) at += k;
            total += k;
        }
        if (reach) sh.list[at + __popcll(mask & ((1ull << lane) - 1))] = (int)j;
        pending += total;
        __syncthreads();
        const bool flush = last && j0 + kOrdThreads >= end;
        int head = 0;
        while (pending - head >= kOrdBatch || (flush && pending > head)) {
            const int count = pending - head < kOrdBatch ? pending - head : kOrdBatch;
            if (lane < count) {
                // this wavefront's axis of the particle
                const OrdParticle p = load(sh.list[head + lane]);
                double S0[S], S1[S], DS[S];
                const double dold = wave == 0 ? p.dold[0] : (wave == 1 ? p.dold[1] : p.dold[2]);
                const double pnn = wave == 0 ? p.pnn[0] : (wave == 1 ? p.pnn[1] : p.pnn[2]);
                const int node = wave == 0 ? p.node[0] : (wave == 1 ? p.node[1] : p.node[2]);
                esirkepov_shapes<ORDER>(dold, pnn, node, S0, S1, DS);
                const double cr = p.cw * (wave == 0 ? dxdt[0] : (wave == 1 ? dxdt[1] : dxdt[2]));
#pragma unroll
                for (int m = 0; m < S; ++m) sh.sd[wave][m][lane] = make_double2(S0[m], DS[m]);
#pragma unroll
                for (int m = 0; m < S - 1; ++m) sh.pre[wave][m][lane] = ORDER == 2 ? DS[m] : cr * DS[m];
                sh.cr[wave][lane] = cr;
                if (wave == 0) {
                    int pk = 0;
#pragma unroll
                    for (int d = 0; d < 3; ++d) pk |= (p.io[d] - (H + 1) - t0[d] + 16) << (5 * d);
                    sh.base[lane] = pk;
                }
            }
            if (wave == 0 && lane >= count) sh.base[lane] = 0x7FFF;  // no point of the tile
            __syncthreads();
            if (wave == 0) ordered_add<ORDER, 0>(sh, count, pt, acc);
            else if (wave == 1) ordered_add<ORDER, 1>(sh, count, pt, acc);
            else ordered_add<ORDER, 2>(sh, count, pt, acc);
            head += count;
            __syncthreads();
        }
        // the rest (fewer than a batch) to the front of the list
        const int rest = pending - head;
        int keep = 0;
        if (head && (int)threadIdx.x < rest) keep = sh.list[head + threadIdx.x];
        __syncthreads();
        if (head && (int)threadIdx.x < rest) sh.list[threadIdx.x] = keep;
        pending = rest;
        __syncthreads();
        if (flush) break;
    }
}

}  // namespace dev
}  // namespace smi
