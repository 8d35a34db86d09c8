// seams.hip -- per-operator entry points for the remaining reference seams:
//
//  * smi_current_deposition_3d / smi_density_deposition_3d keep the argument
//    lists of the reference's own C seams currentDeposition3DOnDevice and
//    densityDeposition3DOnDevice (src/Projector/Projector3D2OrderGPU.cpp:
//    55-120): one patch, particles binned by 4^3 cluster (bin_index = the
//    clusters' cumulative ends, Particles::last_index), per-particle int16
//    charge, SmileiMPI scratch iold/deltaold with stride n;
//  * smi_density_3d / smi_density_2d: Projector3D2Order / 3D4Order /
//    2D2Order ::basic, type 0 (the charge density of diagnostic steps and of
//    frozen species);
//  * smi_maxwell_ampere_2d / smi_maxwell_faraday_2d (MA_Solver2D_norm,
//    MF_Solver2D_Yee) on one patch;
//  * smi_sum_j_ghosts / smi_exchange_b: SyncVectorPatch::sumAllComponents and
//    exchangeB over all patches of a device, held in one patch-major array;
//  * smi_sort_exchange: the particle exchange between patches and the cell
//    sort of one species (Patch::exchParticles / importAndSortParticles,
//    Species::sortParticles) on one device.
#include <cstdio>
#include <vector>

#include "../../include/smilei_amd.h"
#include "kernels.h"
#include "pic_device.h"
#include "seams_internal.h"
#include "workspace.h"

using namespace smi;
using namespace smi::dev;
using namespace smi::seams;

int smi::seams::op_fail(int code, const std::string &m)
{
    set_error(m);
    return code;
}

namespace {

inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

#define SEAM_CHECK()                                                              \
    do {                                                                          \
        hipError_t e_ = hipGetLastError();                                        \
        if (e_ != hipSuccess) return op_fail(SMI_ERR_HIP, hipGetErrorString(e_)); \
    } while (0)

// ---------------------------------------------------------------------------
// Cluster-tiled deposits of the reference seams.  One workgroup per 4^3
// cluster of the patch (bins in the reference's x-major order); the cluster's
// tile spans the 9 array points [4c, 4c+9) per axis: the order-2 stencils
// (old nearest node +-2) of every particle binned in the cluster.  A particle
// whose stencil would leave the tile (not binned where bin_index says, or
// moved more than one cell) is skipped and flagged.
// ---------------------------------------------------------------------------
constexpr int kCT = 9, kCT3 = kCT * kCT * kCT;
// strides of the tile in LDS: rows padded by one word, fewer bank conflicts
constexpr int kCY = kCT + 1, kCX = kCT * kCY, kCC = kCT * kCX;

struct SeamArgs {
    double *out[3];     // Jx, Jy, Jz (currents) or rho (density)
    int64_t size[3];    // their sizes in doubles
    const double *pos[3];
    const short *charge;
    const double *weight;
    const int *bin_index;
    int nb[3];
    const int *iold;
    const double *dold;
    int64_t n;          // stride of iold / deltaold
    double icv, dinv[3], dxdt[3];
    int dom[3], nprimy, nprimz, not_spectral, cell_sorting;
    int *err;
};

__device__ inline int bin_coords(const SeamArgs &a, int b, int *bc)
{
    bc[0] = b / (a.nb[1] * a.nb[2]);
    bc[1] = (b / a.nb[2]) % a.nb[1];
    bc[2] = b % a.nb[2];
    return b;
}

// Calls f(i) for this thread's particles of bin b: with cell_sorting runs of
// neighbours (mostly of one cell) per thread, a strided walk otherwise
// (Projector3D2OrderGPUKernelCUDAHIP.cu:237-256 picks such a pair of orders).
// Only the order of the tile atomics differs.  The runs go to the lanes of
// different wavefronts in turn, so that the lanes of one wavefront mostly lie in
// different cells: with neighbouring runs on neighbouring lanes their atomics met
// on the same words (currents of 16 particles per cell 44.5 us against 42.3).
// A run is four particles at most, 1,024 of the bin at a time, where there are
// more bins than the caches hold the lines of: each thread of a run reads 8 bytes
// of its own line of 13 arrays.  Both seams, 64 particles per cell, few movers
// / many: 512 bins 656 / 666 us with one run a thread, 305 / 420 with runs of
// four; 4,096 bins 4,887 / 4,944 and 2,372 / 2,977; but 64 bins 179 / 214 and 192
// / 249, 128 bins (of 128 per cell) 372 / 421 and 369 / 523, 256 690 / 699 and
// 372 / 528.
constexpr int kSeamThreads = 256, kSeamRun = 4, kSeamFewBins = 128;

template <class F>
__device__ inline void for_bin(const SeamArgs &a, int b, F f)
{
    int64_t first = b == 0 ? 0 : a.bin_index[b - 1], last = a.bin_index[b];
    first = first < 0 ? 0 : (first > a.n ? a.n : first);
    last = last < first ? first : (last > a.n ? a.n : last);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t once = !a.cell_sorting ? kSeamThreads
                                         : (gridDim.x <= kSeamFewBins ? last - first : kSeamRun * kSeamThreads);
    const int place = a.cell_sorting ? lane * (kSeamThreads / 64) + wave : threadIdx.x;
    for (int64_t i0 = first; i0 < last; i0 += once) {
        const int64_t end = i0 + once < last ? i0 + once : last;
        const int per = (int)((end - i0 + kSeamThreads - 1) / kSeamThreads);
        const int64_t mine = i0 + (int64_t)place * per;
        for (int64_t i = mine; i < mine + per && i < end; ++i) f(i);
    }
}

// Old node and new position of particle i; false when its stencil leaves the
// tile or it moved more than one cell.  o: tile index of stencil point 0.
__device__ inline bool seam_particle(const SeamArgs &a, int64_t i, const int *bc, int *o, int *node, int *sh, double *pn)
{
    bool ok = true;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int io = a.iold[d * a.n + i];
        pn[d] = a.pos[d][i] * a.dinv[d];
        node[d] = io + a.dom[d];
        sh[d] = (int)round(pn[d]) - node[d];
        o[d] = io - 2 - 4 * bc[d];
        ok &= sh[d] >= -1 && sh[d] <= 1 && o[d] >= 0 && o[d] <= kCT - 5;
    }
    return ok;
}

// Currents of one particle on the tile: the stencil of a particle that keeps
// its node (WIDE = false) or the whole window.
template <bool WIDE>
__device__ inline void seam_deposit(const SeamArgs &a, int64_t i, const int *o, const int *node, const double *pn,
                                    double *sJ)
{
    double S0[3][4], DS[3][4];
    int w0[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) esirkepov_window<2>(a.dold[d * a.n + i], pn[d], node[d], S0[d], DS[d], w0[d]);
    // charge_weight and cr_p as Projector3D2OrderGPUKernelCUDAHIP.cu:281-284
    const double cw = a.icv * (double)a.charge[i] * a.weight[i];
    const double cr[3] = {cw * a.dxdt[0], cw * a.dxdt[1], cw * a.dxdt[2]};
    double *t = sJ + o[0] * kCX + o[1] * kCY + o[2];
    auto add = [&](int c, int u, int v, int k, double val) { atomicAdd(&t[c * kCC + u * kCX + v * kCY + k], val); };
    if constexpr (WIDE) {
        esirkepov3d_fact<2, 4, 3>(S0, DS, w0, cr, add);
    } else {
        const int one[3] = {1, 1, 1};
        esirkepov3d_fact<2, 3, 2>(S0, DS, one, cr, add);
    }
}

// Bound by the tile atomics and the FP64 arithmetic: a particle that keeps
// its node adds 54 points (300 walked with a test for zero before: 84 us for
// 524,288 particles in 512 bins, 42 now); the others are queued and
// deposited by a second pass, so that the lanes of the first agree.
__global__ void __launch_bounds__(kSeamThreads) k_seam_currents(SeamArgs a)
{
    constexpr int QCAP = 256;
    __shared__ double sJ[3 * kCC];
    __shared__ int64_t sQ[QCAP];
    __shared__ int sQn;
    const int b = blockIdx.x;
    int bc[3];
    bin_coords(a, b, bc);
    for (int t = threadIdx.x; t < 3 * kCC; t += blockDim.x) sJ[t] = 0.;
    if (threadIdx.x == 0) sQn = 0;
    __syncthreads();
    for_bin(a, b, [&](int64_t i) {
        int o[3], node[3], sh[3];
        double pn[3];
        if (!seam_particle(a, i, bc, o, node, sh, pn)) {
            atomicOr(a.err, 1);
            return;
        }
        if ((sh[0] | sh[1] | sh[2]) == 0) {
            seam_deposit<false>(a, i, o, node, pn, sJ);
            return;
        }
        const int q = atomicAdd(&sQn, 1);
        if (q < QCAP) sQ[q] = i;
        else seam_deposit<true>(a, i, o, node, pn, sJ);
    });
    __syncthreads();
    const int nq = sQn < QCAP ? sQn : QCAP;
    for (int q = threadIdx.x; q < nq; q += blockDim.x) {
        int o[3], node[3], sh[3];
        double pn[3];
        seam_particle(a, sQ[q], bc, o, node, sh, pn);
        seam_deposit<true>(a, sQ[q], o, node, pn, sJ);
    }
    __syncthreads();
    // flush: Jy and Jz are dual along y / z when not_spectral (their rows are
    // one point longer), as the reference's flush indexing encodes
    for (int t = threadIdx.x; t < kCT3; t += blockDim.x) {
        const int u = t / (kCT * kCT), v = (t / kCT) % kCT, k = t % kCT;
        const int gx = 4 * bc[0] + u, gy = 4 * bc[1] + v, gz = 4 * bc[2] + k;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const double val = sJ[c * kCC + u * kCX + v * kCY + k];
            if (val == 0.) continue;
            int64_t idx = ((int64_t)gx * a.nprimy + gy) * a.nprimz + gz;
            if (c == 1) idx += (int64_t)a.not_spectral * gx * a.nprimz;
            if (c == 2) idx += (int64_t)a.not_spectral * ((int64_t)gx * a.nprimy + gy);
            if (idx < 0 || idx >= a.size[c]) {
                atomicOr(a.err, 2);
                continue;
            }
            unsafeAtomicAdd(&a.out[c][idx], val);
        }
    }
}

__global__ void __launch_bounds__(kSeamThreads) k_seam_density(SeamArgs a)
{
    __shared__ double sR[kCC];
    const int b = blockIdx.x;
    int bc[3];
    bin_coords(a, b, bc);
    for (int t = threadIdx.x; t < kCC; t += blockDim.x) sR[t] = 0.;
    __syncthreads();
    for_bin(a, b, [&](int64_t i) {
        int o[3], node[3], sh[3];
        double pn[3], S1[3][3];
        if (!seam_particle(a, i, bc, o, node, sh, pn)) {
            atomicOr(a.err, 1);
            return;
        }
        // S1: the new position's weights on the 5-point window of the old
        // node (init_S1, Projector3D2OrderGPUKernelCUDAHIP.cu:116-131), whose
        // three non-zero entries start at 1 + the node change
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            spline2(pn[d] - (double)(node[d] + sh[d]), S1[d]);
            o[d] += 1 + sh[d];
        }
        const double cw = a.icv * (double)a.charge[i] * a.weight[i];
        double *r = sR + o[0] * kCX + o[1] * kCY + o[2];
#pragma unroll
        for (int u = 0; u < 3; ++u)
#pragma unroll
            for (int v = 0; v < 3; ++v) {
                const double t = cw * S1[0][u] * S1[1][v];
#pragma unroll
                for (int k = 0; k < 3; ++k) atomicAdd(&r[u * kCX + v * kCY + k], t * S1[2][k]);
            }
    });
    __syncthreads();
    for (int t = threadIdx.x; t < kCT3; t += blockDim.x) {
        const int u = t / (kCT * kCT), v = (t / kCT) % kCT, k = t % kCT;
        const double val = sR[u * kCX + v * kCY + k];
        if (val == 0.) continue;
        const int64_t idx = ((int64_t)(4 * bc[0] + u) * a.nprimy + 4 * bc[1] + v) * a.nprimz + 4 * bc[2] + k;
        if (idx < 0 || idx >= a.size[0]) {
            atomicOr(a.err, 2);
            continue;
        }
        unsafeAtomicAdd(&a.out[0][idx], val);
    }
}

// Checks shared by both seams; fills SeamArgs.  Returns SMI_OK or an error.
int seam_args(SeamArgs &a, const int *bin_index, unsigned nbx, unsigned nby, unsigned nbz, const int *iold,
              const double *deltaold, unsigned n, double inv_cell_volume, double dx_inv, double dy_inv,
              double dz_inv, double dx_ov_dt, double dy_ov_dt, double dz_ov_dt, int i_dom, int j_dom, int k_dom,
              int nprimy, int nprimz, int not_spectral, bool cell_sorting)
{
    if (nbx == 0 || nby == 0 || nbz == 0 || (uint64_t)nbx * nby * nbz > (1u << 30))
        return op_fail(SMI_ERR_INVALID, "bin counts must be positive");
    if (nprimy < 9 || nprimz < 9) return op_fail(SMI_ERR_INVALID, "nprimy and nprimz must hold a 9-point tile");
    if (4 * (int64_t)(nby - 1) + kCT > nprimy || 4 * (int64_t)(nbz - 1) + kCT > nprimz)
        return op_fail(SMI_ERR_INVALID, "bin counts do not fit the patch arrays (4 cells per bin + 5 ghost points)");
    if (not_spectral != 0 && not_spectral != 1) return op_fail(SMI_ERR_INVALID, "not_spectral must be 0 or 1");
    if (n > 0 && (!bin_index || !iold || !deltaold)) return op_fail(SMI_ERR_INVALID, "null particle scratch");
    a.bin_index = bin_index;
    a.nb[0] = (int)nbx;
    a.nb[1] = (int)nby;
    a.nb[2] = (int)nbz;
    a.iold = iold;
    a.dold = deltaold;
    a.n = n;
    a.icv = inv_cell_volume;
    a.dinv[0] = dx_inv;
    a.dinv[1] = dy_inv;
    a.dinv[2] = dz_inv;
    a.dxdt[0] = dx_ov_dt;
    a.dxdt[1] = dy_ov_dt;
    a.dxdt[2] = dz_ov_dt;
    a.dom[0] = i_dom;
    a.dom[1] = j_dom;
    a.dom[2] = k_dom;
    a.nprimy = nprimy;
    a.nprimz = nprimz;
    a.not_spectral = not_spectral;
    a.cell_sorting = cell_sorting ? 1 : 0;
    return SMI_OK;
}

// Runs one seam kernel on the null stream with a fresh error flag, waits for
// it (the reference's launcher synchronises the device after the kernel) and
// reports skipped particles.
template <class Kernel>
int run_seam(Kernel k, SeamArgs &a)
{
    int *err = nullptr;
    if (hipMalloc(&err, sizeof(int)) != hipSuccess) return op_fail(SMI_ERR_HIP, "hipMalloc of the error flag failed");
    try {
        launch_fill_i32(err, 1, 0, nullptr);
    } catch (const std::exception &ex) {
        (void)hipFree(err);
        return op_fail(SMI_ERR_HIP, ex.what());
    }
    a.err = err;
    hipLaunchKernelGGL(k, dim3((unsigned)(a.nb[0] * a.nb[1] * a.nb[2])), dim3(256), 0, nullptr, a);
    hipError_t e = hipGetLastError();
    int h = 0;
    if (e == hipSuccess) e = hipMemcpy(&h, err, sizeof(int), hipMemcpyDeviceToHost);
    (void)hipFree(err);
    if (e != hipSuccess) return op_fail(SMI_ERR_HIP, hipGetErrorString(e));
    if (h & 1)
        return op_fail(SMI_ERR_INVALID, "a particle's stencil leaves its bin's tile (not binned by bin_index, or moved "
                                        "more than one cell); it was skipped");
    if (h & 2) return op_fail(SMI_ERR_INVALID, "a tile point falls outside the output array (sizes too small)");
    return SMI_OK;
}

// ---------------------------------------------------------------------------
// Projector::basic type 0 (charge density at the particles' positions), one
// thread per particle, FP64 atomics into the patch array.
// ---------------------------------------------------------------------------
struct BasicArgs {
    double *rho;
    int np[3];
    int dom[3];
    double dinv[3];
    double cw_scale;  // inv_cell_volume * charge
    int64_t n;
    const double *pos[3];
    const double *w;
    int *err;
};

template <int ND, int ORDER>
__global__ void __launch_bounds__(256) k_basic(BasicArgs a)
{
    constexpr int H = ORDER / 2, W = 2 * H + 1;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    double S[3][5];
    int o[3] = {0, 0, 0};
    bool ok = true;
    for (int d = 0; d < ND; ++d) {
        const double pn = a.pos[d][i] * a.dinv[d];
        const int ip = (int)round(pn);
        spline<ORDER>(pn - (double)ip, S[d]);
        o[d] = ip - a.dom[d] - H;
        ok &= o[d] >= 0 && o[d] + W <= a.np[d];
    }
    if (!ok) {
        atomicOr(a.err, 1);
        return;
    }
    const double cw = a.cw_scale * a.w[i];
    if constexpr (ND == 3) {
        for (int u = 0; u < W; ++u)
            for (int v = 0; v < W; ++v)
                for (int k = 0; k < W; ++k)
                    unsafeAtomicAdd(&a.rho[((int64_t)(o[0] + u) * a.np[1] + (o[1] + v)) * a.np[2] + (o[2] + k)],
                                    cw * S[0][u] * S[1][v] * S[2][k]);
    } else {
        for (int u = 0; u < W; ++u)
            for (int v = 0; v < W; ++v)
                unsafeAtomicAdd(&a.rho[(int64_t)(o[0] + u) * a.np[1] + (o[1] + v)], cw * S[0][u] * S[1][v]);
    }
}

int run_basic(int nd, int order, BasicArgs &a, hipStream_t st)
{
    int *err = nullptr;
    if (hipMalloc(&err, sizeof(int)) != hipSuccess) return op_fail(SMI_ERR_HIP, "hipMalloc of the error flag failed");
    try {
        launch_fill_i32(err, 1, 0, st);
    } catch (const std::exception &ex) {
        (void)hipFree(err);
        return op_fail(SMI_ERR_HIP, ex.what());
    }
    a.err = err;
    const dim3 grid(nblk(a.n, 256)), block(256);
    if (nd == 3 && order == 2) hipLaunchKernelGGL((k_basic<3, 2>), grid, block, 0, st, a);
    else if (nd == 3) hipLaunchKernelGGL((k_basic<3, 4>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((k_basic<2, 2>), grid, block, 0, st, a);
    hipError_t e = hipGetLastError();
    int h = 0;
    if (e == hipSuccess) e = hipMemcpyAsync(&h, err, sizeof(int), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    (void)hipFree(err);
    if (e != hipSuccess) return op_fail(SMI_ERR_HIP, hipGetErrorString(e));
    if (h) return op_fail(SMI_ERR_INVALID, "a particle's stencil leaves the patch arrays; it was skipped");
    return SMI_OK;
}

// ---------------------------------------------------------------------------
// MA_Solver2D_norm / MF_Solver2D_Yee on one patch (same arithmetic and
// association as MA_Solver2D_norm.cpp:54-105, MF_Solver2D_Yee.cpp:50-99).
// ---------------------------------------------------------------------------
__global__ void k_ma2d_patch(double *Ex, double *Ey, double *Ez, const double *Bx, const double *By,
                             const double *Bz, const double *Jx, const double *Jy, const double *Jz, int nxp, int nyp,
                             double dt, double dtx, double dty)
{
    const int64_t nxd = nxp + 1, nyd = nyp + 1;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nEx = nxd * nyp, nEy = (int64_t)nxp * nyd, nEz = (int64_t)nxp * nyp;
    if (t < nEx) {
        const int64_t x = t / nyp, y = t % nyp;
        Ex[t] += -dt * Jx[t] + dty * (Bz[x * nyd + y + 1] - Bz[x * nyd + y]);
    } else if (t < nEx + nEy) {
        const int64_t e = t - nEx, x = e / nyd, y = e % nyd;
        Ey[e] += -dt * Jy[e] - dtx * (Bz[(x + 1) * nyd + y] - Bz[x * nyd + y]);
    } else if (t < nEx + nEy + nEz) {
        const int64_t e = t - nEx - nEy, x = e / nyp, y = e % nyp;
        Ez[e] += -dt * Jz[e] + dtx * (By[(x + 1) * nyp + y] - By[x * nyp + y]) -
                 dty * (Bx[x * nyd + y + 1] - Bx[x * nyd + y]);
    }
}

__global__ void k_mf2d_patch(double *Bx, double *By, double *Bz, const double *Ex, const double *Ey,
                             const double *Ez, int nxp, int nyp, double dtx, double dty)
{
    const int64_t nxd = nxp + 1, nyd = nyp + 1;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nBx = (int64_t)nxp * nyd, nBy = nxd * nyp, nBz = nxd * nyd;
    if (t < nBx) {
        const int64_t x = t / nyd, y = t % nyd;
        if (y < 1 || y >= nyd - 1) return;
        Bx[t] -= dty * (Ez[x * nyp + y] - Ez[x * nyp + y - 1]);
    } else if (t < nBx + nBy) {
        const int64_t e = t - nBx, x = e / nyp, y = e % nyp;
        if (x < 1 || x >= nxd - 1) return;
        By[e] += dtx * (Ez[x * nyp + y] - Ez[(x - 1) * nyp + y]);
    } else if (t < nBx + nBy + nBz) {
        const int64_t e = t - nBx - nBy, x = e / nyd, y = e % nyd;
        if (x < 1 || x >= nxd - 1 || y < 1 || y >= nyd - 1) return;
        Bz[e] += dty * (Ex[x * nyp + y] - Ex[x * nyp + y - 1]) - dtx * (Ey[x * nyd + y] - Ey[(x - 1) * nyd + y]);
    }
}

// ---------------------------------------------------------------------------
// B exchange between the patches of a patch-major array (exchangeB,
// SyncVectorPatch.cpp:667, 1441-1830), one pass per axis d: for each B
// component dual along d, this patch's planes [0, os) <- the low neighbour's
// [n, n+os), and the low neighbour's [n+os+2, n+2os+2) <- this patch's
// [os+2, 2os+2).  Within a pass no point is both read and written.
// ---------------------------------------------------------------------------
__device__ inline int low_patch(const Geom &g, int p, int d)
{
    int pc[3] = {p / (g.npatch[1] * g.npatch[2]), (p / g.npatch[2]) % g.npatch[1], p % g.npatch[2]};
#pragma unroll
    for (int e = 0; e < 3; ++e)
        if (e == d) pc[e] = wrapi(pc[e] - 1, g.npatch[e]);
    return (pc[0] * g.npatch[1] + pc[1]) * g.npatch[2] + pc[2];
}

// Work item: point of an os-plane slab of a component dual along d
// (blockIdx.y: B_c is dual along every axis but c) of a patch (`blocks`
// workgroups per slab), so that extents and offsets are scalars.
__global__ void __launch_bounds__(256) k_exchange_b(Geom g, int d, int blocks, double *__restrict__ B)
{
    const int c = (d + 1 + blockIdx.y) % 3, p = blockIdx.x / blocks;
    int r = (int)(blockIdx.x - p * blocks) * 256 + threadIdx.x;
    int np[3], dm[3], ext[3];
    int64_t off = 0, per = 0;
#pragma unroll
    for (int e = 0; e < 3; ++e) {
        np[e] = e < g.nd ? g.n[e] + 2 * g.os + 1 : 1;
        dm[e] = np[e] + (e != c && e < g.nd ? 1 : 0);
        ext[e] = e == d ? g.os : dm[e];
    }
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        int64_t sz = 1;
#pragma unroll
        for (int e = 0; e < 3; ++e) sz *= np[e] + (e != q && e < g.nd ? 1 : 0);
        if (q < c) off += sz;
        per += sz;
    }
    const int row = ext[1] * ext[2];
    const int i = r / row;
    if (i >= ext[0]) return;
    r -= i * row;
    const int j = r / ext[2], k = r - j * ext[2];
    double *me = B + p * per + off, *lo = B + (int64_t)low_patch(g, p, d) * per + off;
    const int64_t at = ((int64_t)i * dm[1] + j) * dm[2] + k;
    const int64_t step = d == 0 ? (int64_t)dm[1] * dm[2] : (d == 1 ? dm[2] : 1);
    const int nd = d == 0 ? g.n[0] : (d == 1 ? g.n[1] : g.n[2]);
    const int gsp = g.os + 2;
    me[at] = lo[at + nd * step];
    lo[at + (nd + gsp) * step] = me[at + gsp * step];
}

}  // namespace

// ---------------------------------------------------------------------------
// Geometry of the per-device entry points (the checks of smi_create).
// ---------------------------------------------------------------------------
int smi::seams::make_geom(int ndim, int order, const int n_cells[3], const int patch_size[3], const double *cell_length,
              Geom &g)
{
    if (ndim != 2 && ndim != 3) return op_fail(SMI_ERR_INVALID, "ndim must be 2 or 3");
    if (order != 2 && order != 4) return op_fail(SMI_ERR_INVALID, "order must be 2 or 4");
    if (ndim == 2 && order != 2) return op_fail(SMI_ERR_INVALID, "2D order must be 2");
    g = Geom{};
    g.nd = ndim;
    g.order = order;
    g.os = order;
    int64_t ncells = 1;
    for (int d = 0; d < 3; ++d) {
        if (d < ndim) {
            if (n_cells[d] <= 0 || patch_size[d] <= 0 || !(cell_length[d] > 0))
                return op_fail(SMI_ERR_INVALID, "n_cells, patch_size and cell_length must be positive");
            if (patch_size[d] % 4) return op_fail(SMI_ERR_INVALID, "patch_size must be a multiple of 4");
            if (n_cells[d] % patch_size[d]) return op_fail(SMI_ERR_INVALID, "patch_size must divide n_cells");
            if (patch_size[d] < 2 * g.os + 2)
                return op_fail(SMI_ERR_INVALID, "patch_size must be >= 2*oversize+2 for the ghost sum");
            g.N[d] = n_cells[d];
            g.n[d] = patch_size[d];
            g.dx[d] = cell_length[d];
        } else {
            g.N[d] = 1;
            g.n[d] = 1;
            g.dx[d] = 1.0;
        }
        g.npatch[d] = g.N[d] / g.n[d];
        g.ncl[d] = d < ndim ? g.n[d] / 4 : 1;
        g.dinv[d] = 1.0 / g.dx[d];
        g.plen[d] = (double)g.n[d] * g.dx[d];
        g.xmax[d] = g.dx[d] * (double)g.N[d];
        ncells *= g.N[d];
    }
    if (ncells >= (1ll << 27)) return op_fail(SMI_ERR_INVALID, "at most 2^27 cells");
    g.ncells = ncells;
    g.cpp = g.n[0] * g.n[1] * g.n[2];
    g.clpp = g.ncl[0] * g.ncl[1] * g.ncl[2];
    g.cells_per_cl = ndim == 3 ? 64 : 16;
    g.npatches = g.npatch[0] * g.npatch[1] * g.npatch[2];
    g.dt = 1.0;
    return SMI_OK;
}

// ---------------------------------------------------------------------------
// Particle exchange + cell sort of one species over all patches of a device.
// ---------------------------------------------------------------------------
namespace {

// Periodic wrap of Patch::prepareParticles (Patch.cpp:624-668): a position
// that left the box by less than its length re-enters on the other side;
// one farther out is flagged and left alone.  Then its cell key and the
// histogram of the cells, lanes with one cell in a row sharing an atomic: 39
// us for 4.2e6 particles in one pass over the positions, 216 in three with an
// atomic per particle.
template <int ND>
__global__ void __launch_bounds__(256)
k_wrap_bin(Geom g, double *x, double *y, double *z, int64_t n, uint32_t *__restrict__ keys, int32_t *__restrict__ counts,
           int *err)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t key = ~0u;
    if (i < n) {
        double *p[3] = {x, y, z};
        double v[3] = {0., 0., 0.};
        bool ok = true;
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            const double was = p[d][i];
            v[d] = was;
            if (!ok) continue;
            double w = was;
            if (w < 0.) w += g.xmax[d];
            else if (w >= g.xmax[d]) w -= g.xmax[d];
            // a tiny negative position can round to xmax itself: kept, and
            // clamped into the last cell by the key like the reference's
            ok = w >= 0. && w <= g.xmax[d];
            if (ok && w != was) p[d][i] = v[d] = w;
        }
        if (!ok) atomicOr(err, 1);
        key = position_key<ND>(g, v);
        keys[i] = (13u << 27) | key;
    }
    int head, len;
    key_run(key, head, len);
    if ((int)(threadIdx.x & 63) == head && i < n) atomicAdd(&counts[key], len);
}

// Particle arrays that are reordered together: up to kMoveMax of 8-byte
// elements, the charges, and the keys that the first pass writes out.
constexpr int kMoveMax = 8;
struct MoveSet {
    double *a[kMoveMax];  // null beyond the last one
    int16_t *charge, *charge_stage;
    int32_t *key;
};

// Sorted slot i of every array into the staging area, one thread per particle:
// the particles lie almost in order, so what bounds it is the number of loads
// in flight, and all arrays' loads depend on the one load of perm only.
// 4.2e6 particles of 7 arrays, charges and keys (660 MB, in two passes): 137 us,
// against 163 us one array at a time, and 4 launches instead of 17.
__global__ void __launch_bounds__(256) k_gather_set(Geom g, MoveSet M, const int32_t *__restrict__ perm,
                                                    const uint32_t *__restrict__ keys, double *__restrict__ stage,
                                                    int64_t stage_len, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int32_t p = perm[i];
    double v[kMoveMax];
    int16_t q = 0;
    uint32_t k = 0;
#pragma unroll
    for (int j = 0; j < kMoveMax; ++j) v[j] = M.a[j] ? M.a[j][p] : 0.;
    if (M.charge) q = M.charge[p];
    if (M.key) k = keys[p];
#pragma unroll
    for (int j = 0; j < kMoveMax; ++j)
        if (M.a[j]) stage[j * stage_len + i] = v[j];
    if (M.charge) M.charge_stage[i] = q;
    // in-patch cell key of the slot
    if (M.key) M.key[i] = (int32_t)((k & ((1u << 27) - 1)) % (uint32_t)g.cpp);
}

// And back: blockIdx.y the array, after the last one the charges; kMovePer
// elements a thread.
constexpr int kMovePer = 4;
__global__ void __launch_bounds__(256) k_unstage_set(MoveSet M, int arrays, const double *__restrict__ stage,
                                                     int64_t stage_len, int64_t n)
{
    const int64_t i0 = (int64_t)blockIdx.x * (256 * kMovePer) + threadIdx.x;
    const int j = blockIdx.y;
    if (j == arrays) {
#pragma unroll
        for (int k = 0; k < kMovePer; ++k)
            if (i0 + 256 * k < n) M.charge[i0 + 256 * k] = M.charge_stage[i0 + 256 * k];
        return;
    }
    double *__restrict__ a = M.a[j];
    const double *__restrict__ s = stage + j * stage_len;
    double v[kMovePer];
#pragma unroll
    for (int k = 0; k < kMovePer; ++k) v[k] = i0 + 256 * k < n ? s[i0 + 256 * k] : 0.;
#pragma unroll
    for (int k = 0; k < kMovePer; ++k)
        if (i0 + 256 * k < n) a[i0 + 256 * k] = v[k];
}

// Per-patch particle counts and, per patch, the cumulative ends of its
// clusters relative to the patch's first particle (Particles::last_index).
__global__ void k_bins_out(Geom g, const int32_t *__restrict__ cell_off, int32_t *__restrict__ patch_count,
                           int32_t *__restrict__ bin_index)
{
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)g.npatches * g.clpp) return;
    const int p = (int)(t / g.clpp), b = (int)(t % g.clpp);
    const int64_t c0 = (int64_t)p * g.cpp;
    if (bin_index) bin_index[t] = cell_off[c0 + (int64_t)(b + 1) * g.cells_per_cl] - cell_off[c0];
    if (patch_count && b == 0) patch_count[p] = cell_off[c0 + g.cpp] - cell_off[c0];
}

// Device memory of one call: from the stream's pool, or allocated where there
// is none (Workspace); `least` bytes where there is no room for `bytes`.
struct CallMemory {
    Workspace ws;
    void *own = nullptr;
    size_t bytes;
    CallMemory(size_t want, size_t least, hipStream_t st) : ws(want, st), bytes(want)
    {
        if (ws.p) return;
        if (hipMalloc(&own, want) == hipSuccess) return;
        (void)hipGetLastError();
        bytes = least;
        if (hipMalloc(&own, least) != hipSuccess) own = nullptr;
    }
    ~CallMemory() { (void)hipFree(own); }
    void *get() const { return ws.p ? ws.p : own; }
};

constexpr int64_t kAlignWords = 64;

int64_t align_words(int64_t w) { return (w + kAlignWords - 1) / kAlignWords * kAlignWords; }

}  // namespace

int64_t smi::seams::sort_scratch_words(const Geom &g, int64_t n, int nstage)
{
    const int64_t nc = g.ncells, m = n > 0 ? n : 1;
    return align_words(nc) + align_words(nc + 1) + 2 * align_words(m) + align_words(m / 17 + 1) + align_words(3) +
           align_words(sort_bsum_size(nc)) + align_words((nc + 3) / 4) + align_words(nc / g.cells_per_cl) +
           align_words(m) + nstage * align_words(2 * m) + align_words(1);
}

int smi::seams::sort_stage_arrays(const Geom &g, int64_t n, int64_t words)
{
    int k = kMoveMax;
    while (k > 1 && sort_scratch_words(g, n, k) > words) --k;
    return k;
}

SortScratch smi::seams::carve_sort_scratch(const Geom &g, int64_t n, int32_t *base, int nstage)
{
    const int64_t nc = g.ncells, m = n > 0 ? n : 1;
    SortScratch s{};
    int32_t *p = base;
    auto take = [&](int64_t words) {
        int32_t *r = p;
        p += align_words(words);
        return r;
    };
    s.sb.counts = take(nc);
    s.sb.cell_off = take(nc + 1);
    s.sb.perm = take(m);
    s.sb.tmp = take(m);
    s.sb.big = take(m / 17 + 1);
    s.sb.nbig = take(3);
    s.sb.nbsum = sort_bsum_size(nc);
    s.sb.bsum = take(s.sb.nbsum);
    s.sb.stay = (uint8_t *)take((nc + 3) / 4);
    s.sb.clus_old = take(nc / g.cells_per_cl);
    s.sb.rank = nullptr;
    s.keys = (uint32_t *)take(m);
    s.nstage = nstage;
    s.stage_len = align_words(2 * m) / 2;
    s.stage = (double *)take(2 * s.stage_len * nstage);
    s.err = take(1);
    return s;
}

int smi::seams::sort_exchange_impl(const Geom &g, int64_t n, const SortArrays &A, SortScratch &s, hipStream_t st)
{
    launch_fill_i32(s.sb.counts, g.ncells, 0, st);
    launch_fill_i32((int32_t *)s.sb.stay, (g.ncells + 3) / 4, 0, st);
    launch_fill_i32(s.err, 1, 0, st);
    if (n > 0) {
        const dim3 grid(nblk(n, 256)), block(256);
        if (g.nd == 3)
            hipLaunchKernelGGL(k_wrap_bin<3>, grid, block, 0, st, g, A.x, A.y, A.z, n, s.keys, s.sb.counts, s.err);
        else
            hipLaunchKernelGGL(k_wrap_bin<2>, grid, block, 0, st, g, A.x, A.y, A.z, n, s.keys, s.sb.counts, s.err);
        SEAM_CHECK();
    }
    launch_sort(g, s.keys, n, s.sb, st, /*counted=*/true, /*in_cell_order=*/true, /*interleaved=*/false,
                /*tie=*/nullptr, /*placed=*/false);
    if (n > 0) {
        // the arrays that the staging area holds at a time; the charges take the place of one
        double *arrs[7] = {A.x, A.y, A.px, A.py, A.pz, A.w, A.z};
        const int na = g.nd == 3 ? 7 : 6;
        bool charge = A.charge != nullptr, key = A.key != nullptr;
        for (int next = 0; next < na || charge || key;) {
            MoveSet M{};
            int used = 0;
            while (next < na && used < s.nstage && used < kMoveMax) M.a[used++] = arrs[next++];
            if (charge && next == na && used < s.nstage) {
                M.charge = A.charge;
                M.charge_stage = (int16_t *)(s.stage + used * s.stage_len);
                charge = false;
            }
            if (key) M.key = A.key;
            key = false;
            hipLaunchKernelGGL(k_gather_set, dim3(nblk(n, 256)), dim3(256), 0, st, g, M, (const int32_t *)s.sb.perm,
                               (const uint32_t *)s.keys, s.stage, s.stage_len, n);
            SEAM_CHECK();
            hipLaunchKernelGGL(k_unstage_set, dim3(nblk(n, 256 * kMovePer), used + (M.charge ? 1 : 0)), dim3(256), 0,
                               st, M, used, (const double *)s.stage, s.stage_len, n);
            SEAM_CHECK();
        }
    }
    if (A.patch_count || A.bin_index) {
        hipLaunchKernelGGL(k_bins_out, dim3(nblk((int64_t)g.npatches * g.clpp, 256)), dim3(256), 0, st, g,
                           (const int32_t *)s.sb.cell_off, A.patch_count, A.bin_index);
        SEAM_CHECK();
    }
    int h = 0;
    hipError_t e = hipMemcpyAsync(&h, s.err, sizeof(int), hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e != hipSuccess) return op_fail(SMI_ERR_HIP, hipGetErrorString(e));
    if (h) return op_fail(SMI_ERR_INVALID, "a particle lies farther than one box length outside the box");
    return SMI_OK;
}

int smi::seams::sort_exchange_args(int ndim, const int n_cells[3], const int patch_size[3], const double cell_length[3],
                       int64_t n, const SortArrays &A, Geom &g)
{
    if (!n_cells || !patch_size || !cell_length) return op_fail(SMI_ERR_INVALID, "null geometry");
    int rc = make_geom(ndim, 2, n_cells, patch_size, cell_length, g);
    if (rc) return rc;
    if (n < 0 || n >= (1ll << 31)) return op_fail(SMI_ERR_INVALID, "particle count out of range");
    if (n > 0 && (!A.x || !A.y || (ndim == 3 && !A.z) || !A.px || !A.py || !A.pz || !A.w))
        return op_fail(SMI_ERR_INVALID, "null particle array");
    return SMI_OK;
}

extern "C" {

int smi_current_deposition_3d(double *Jx, double *Jy, double *Jz, int Jx_size, int Jy_size, int Jz_size,
                              const double *particle_position_x, const double *particle_position_y,
                              const double *particle_position_z, const short *particle_charge,
                              const double *particle_weight, const int *bin_index, unsigned int x_dimension_bin_count,
                              unsigned int y_dimension_bin_count, unsigned int z_dimension_bin_count,
                              const double *invgf, const int *iold, const double *deltaold,
                              unsigned int number_of_particles, double inv_cell_volume, double dx_inv, double dy_inv,
                              double dz_inv, double dx_ov_dt, double dy_ov_dt, double dz_ov_dt, int i_domain_begin,
                              int j_domain_begin, int k_domain_begin, int nprimy, int nprimz, int not_spectral,
                              bool cell_sorting)
{
    (void)invgf;  // read by the 2D/AM projectors only
    SeamArgs a{};
    int rc = seam_args(a, bin_index, x_dimension_bin_count, y_dimension_bin_count, z_dimension_bin_count, iold,
                       deltaold, number_of_particles, inv_cell_volume, dx_inv, dy_inv, dz_inv, dx_ov_dt, dy_ov_dt,
                       dz_ov_dt, i_domain_begin, j_domain_begin, k_domain_begin, nprimy, nprimz, not_spectral,
                       cell_sorting);
    if (rc) return rc;
    if (!Jx || !Jy || !Jz) return op_fail(SMI_ERR_INVALID, "null current array");
    if (number_of_particles > 0 &&
        (!particle_position_x || !particle_position_y || !particle_position_z || !particle_charge || !particle_weight))
        return op_fail(SMI_ERR_INVALID, "null particle array");
    a.out[0] = Jx;
    a.out[1] = Jy;
    a.out[2] = Jz;
    a.size[0] = Jx_size;
    a.size[1] = Jy_size;
    a.size[2] = Jz_size;
    a.pos[0] = particle_position_x;
    a.pos[1] = particle_position_y;
    a.pos[2] = particle_position_z;
    a.charge = particle_charge;
    a.weight = particle_weight;
    return run_seam(k_seam_currents, a);
}

int smi_density_deposition_3d(double *rho, int rho_size, const double *particle_position_x,
                              const double *particle_position_y, const double *particle_position_z,
                              const short *particle_charge, const double *particle_weight, const int *bin_index,
                              unsigned int x_dimension_bin_count, unsigned int y_dimension_bin_count,
                              unsigned int z_dimension_bin_count, const double *invgf, const int *iold,
                              const double *deltaold, unsigned int number_of_particles, double inv_cell_volume,
                              double dx_inv, double dy_inv, double dz_inv, double dx_ov_dt, double dy_ov_dt,
                              double dz_ov_dt, int i_domain_begin, int j_domain_begin, int k_domain_begin, int nprimy,
                              int nprimz, int not_spectral, bool cell_sorting)
{
    (void)invgf;
    SeamArgs a{};
    int rc = seam_args(a, bin_index, x_dimension_bin_count, y_dimension_bin_count, z_dimension_bin_count, iold,
                       deltaold, number_of_particles, inv_cell_volume, dx_inv, dy_inv, dz_inv, dx_ov_dt, dy_ov_dt,
                       dz_ov_dt, i_domain_begin, j_domain_begin, k_domain_begin, nprimy, nprimz, not_spectral,
                       cell_sorting);
    if (rc) return rc;
    if (!rho) return op_fail(SMI_ERR_INVALID, "null density array");
    if (number_of_particles > 0 &&
        (!particle_position_x || !particle_position_y || !particle_position_z || !particle_charge || !particle_weight))
        return op_fail(SMI_ERR_INVALID, "null particle array");
    a.out[0] = rho;
    a.size[0] = rho_size;
    a.pos[0] = particle_position_x;
    a.pos[1] = particle_position_y;
    a.pos[2] = particle_position_z;
    a.charge = particle_charge;
    a.weight = particle_weight;
    return run_seam(k_seam_density, a);
}

int smi_density_3d(int order, double *rho, const int np[3], const int dom_begin[3], const double cell_length[3],
                   double charge, int64_t n, const double *x, const double *y, const double *z, const double *w,
                   void *stream)
{
    if (order != 2 && order != 4) return op_fail(SMI_ERR_INVALID, "order must be 2 or 4");
    if (n <= 0) return SMI_OK;
    if (!rho || !x || !y || !z || !w) return op_fail(SMI_ERR_INVALID, "null array");
    BasicArgs a{};
    a.rho = rho;
    double cell_volume = 1.0;
    for (int d = 0; d < 3; ++d) {
        a.np[d] = np[d];
        a.dom[d] = dom_begin[d];
        a.dinv[d] = 1.0 / cell_length[d];
        cell_volume *= cell_length[d];
    }
    a.cw_scale = (1. / cell_volume) * charge;
    a.n = n;
    a.pos[0] = x;
    a.pos[1] = y;
    a.pos[2] = z;
    a.w = w;
    return run_basic(3, order, a, (hipStream_t)stream);
}

int smi_density_2d(int order, double *rho, const int np[2], const int dom_begin[2], const double cell_length[2],
                   double charge, int64_t n, const double *x, const double *y, const double *w, void *stream)
{
    if (order != 2) return op_fail(SMI_ERR_INVALID, "2D order must be 2");
    if (n <= 0) return SMI_OK;
    if (!rho || !x || !y || !w) return op_fail(SMI_ERR_INVALID, "null array");
    BasicArgs a{};
    a.rho = rho;
    double cell_volume = 1.0;
    for (int d = 0; d < 2; ++d) {
        a.np[d] = np[d];
        a.dom[d] = dom_begin[d];
        a.dinv[d] = 1.0 / cell_length[d];
        cell_volume *= cell_length[d];
    }
    a.np[2] = 1;
    a.cw_scale = (1. / cell_volume) * charge;
    a.n = n;
    a.pos[0] = x;
    a.pos[1] = y;
    a.pos[2] = nullptr;
    a.w = w;
    return run_basic(2, 2, a, (hipStream_t)stream);
}

int smi_maxwell_ampere_2d(double *Ex, double *Ey, double *Ez, const double *Bx, const double *By, const double *Bz,
                          const double *Jx, const double *Jy, const double *Jz, const int np[2], double timestep,
                          const double cell_length[2], void *stream)
{
    if (np[0] < 2 || np[1] < 2) return op_fail(SMI_ERR_INVALID, "patch arrays too small");
    const int64_t tot = (int64_t)(np[0] + 1) * np[1] + (int64_t)np[0] * (np[1] + 1) + (int64_t)np[0] * np[1];
    hipLaunchKernelGGL(k_ma2d_patch, dim3(nblk(tot, 256)), dim3(256), 0, (hipStream_t)stream, Ex, Ey, Ez, Bx, By, Bz,
                       Jx, Jy, Jz, np[0], np[1], timestep, timestep / cell_length[0], timestep / cell_length[1]);
    SEAM_CHECK();
    return SMI_OK;
}

int smi_maxwell_faraday_2d(double *Bx, double *By, double *Bz, const double *Ex, const double *Ey, const double *Ez,
                           const int np[2], double timestep, const double cell_length[2], void *stream)
{
    if (np[0] < 2 || np[1] < 2) return op_fail(SMI_ERR_INVALID, "patch arrays too small");
    const int64_t tot = (int64_t)np[0] * (np[1] + 1) + (int64_t)(np[0] + 1) * np[1] + (int64_t)(np[0] + 1) * (np[1] + 1);
    hipLaunchKernelGGL(k_mf2d_patch, dim3(nblk(tot, 256)), dim3(256), 0, (hipStream_t)stream, Bx, By, Bz, Ex, Ey, Ez,
                       np[0], np[1], timestep / cell_length[0], timestep / cell_length[1]);
    SEAM_CHECK();
    return SMI_OK;
}

int smi_sum_j_ghosts(int ndim, int order, const int n_cells[3], const int patch_size[3], double *J, void *stream)
{
    if (!n_cells || !patch_size || !J) return op_fail(SMI_ERR_INVALID, "null argument");
    const double unit[3] = {1., 1., 1.};
    Geom g;
    int rc = make_geom(ndim, order, n_cells, patch_size, unit, g);
    if (rc) return rc;
    try {
        launch_ghost_sum(g, J, (hipStream_t)stream);
    } catch (const std::exception &e) {
        return op_fail(SMI_ERR_HIP, e.what());
    }
    return SMI_OK;
}

int smi_exchange_b(int ndim, int order, const int n_cells[3], const int patch_size[3], double *B, void *stream)
{
    if (!n_cells || !patch_size || !B) return op_fail(SMI_ERR_INVALID, "null argument");
    const double unit[3] = {1., 1., 1.};
    Geom g;
    int rc = make_geom(ndim, order, n_cells, patch_size, unit, g);
    if (rc) return rc;
    for (int d = 0; d < g.nd; ++d) {
        int64_t slab = 0;  // the larger component's
        for (int c = 0; c < 3; ++c) {
            if (c == d) continue;
            int64_t sz = 1;
            for (int e = 0; e < g.nd; ++e) sz *= e == d ? g.os : g.n[e] + 2 * g.os + 1 + (e != c ? 1 : 0);
            slab = sz > slab ? sz : slab;
        }
        const int64_t blocks = (slab + 255) / 256;
        hipLaunchKernelGGL(k_exchange_b, dim3((unsigned)(blocks * g.npatches), 2), dim3(256), 0, (hipStream_t)stream, g,
                           d, (int)blocks, B);
        SEAM_CHECK();
    }
    return SMI_OK;
}

int smi_sort_exchange(int ndim, const int n_cells[3], const int patch_size[3], const double cell_length[3], int64_t n,
                      double *x, double *y, double *z, double *px, double *py, double *pz, double *w, int16_t *charge,
                      int32_t *key, int32_t *patch_count, int32_t *bin_index, void *stream)
{
    const SortArrays A{x, y, z, px, py, pz, w, charge, key, patch_count, bin_index};
    Geom g;
    int rc = sort_exchange_args(ndim, n_cells, patch_size, cell_length, n, A, g);
    if (rc) return rc;
    // as many arrays staged at a time as fit into what the pool keeps between
    // calls: beyond it, each call would wait for its memory to be mapped
    int nstage = sort_stage_arrays(g, n, kWorkspaceKeep / 4);
    const size_t want = (size_t)sort_scratch_words(g, n, nstage) * 4, least = (size_t)sort_scratch_words(g, n) * 4;
    const CallMemory mem(want, least, (hipStream_t)stream);
    if (!mem.get()) return op_fail(SMI_ERR_HIP, "hipMalloc of the sort scratch failed");
    if (mem.bytes < want) nstage = 1;
    SortScratch s = carve_sort_scratch(g, n, (int32_t *)mem.get(), nstage);
    try {
        rc = sort_exchange_impl(g, n, A, s, (hipStream_t)stream);
    } catch (const std::exception &e) {
        rc = op_fail(SMI_ERR_HIP, e.what());
    }
    (void)hipStreamSynchronize((hipStream_t)stream);
    return rc;
}

}  // extern "C"
