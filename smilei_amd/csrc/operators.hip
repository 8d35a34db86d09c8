// operators.hip -- per-operator entry points in the reference's per-patch
// memory layout (ghosted Field3D/Field2D arrays, SoA particles and the
// SmileiMPI dynamics_* scratch with stride n).  A reference build that keeps
// its own orchestration calls these from its operator classes in place of
// the OpenMP-target loops and of currentDeposition3DOnDevice
// (src/Projector/Projector3D2OrderGPU.cpp:55-88).
#include "../../include/smilei_amd.h"
#include "kernels.h"
#include "pic_device.h"
#include "workspace.h"

using namespace smi;
using namespace smi::dev;

namespace {

inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

struct Ints3 {
    int v[3];
};
struct Dbl3 {
    double v[3];
};

// Interpolator3D{2,4}Order::fieldsWrapper, one thread per particle.
// (launched with 256 threads: the bound leaves the compiler 256 registers
// instead of the 128 of a 1024-thread default; the six gathers are kept apart,
// so that their loads in flight fit in them)
template <int ORDER, class O>
__global__ void __launch_bounds__(256, ORDER == 4 ? 3 : 4) k_interp3d(const double *Ex, const double *Ey, const double *Ez, const double *Bx, const double *By,
                           const double *Bz, Ints3 np, Ints3 dom, Dbl3 dinv, int64_t n, const double *x,
                           const double *y, const double *z, double *Ep, double *Bp, int32_t *iold, double *dold)
{
    constexpr int H = ORDER / 2;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double pos[3] = {x[i], y[i], z[i]};
    double cp[3][5], cd[3][5], dp[3];
    int ip[3], id[3];
    for (int d = 0; d < 3; ++d) {
        const double pn = pos[d] * dinv.v[d];
        ip[d] = (int)round(pn);
        dp[d] = pn - (double)ip[d];
        spline<ORDER>(dp[d], cp[d]);
        id[d] = (int)round(pn + 0.5);
        spline<ORDER>(pn - (double)id[d] + 0.5, cd[d]);
        ip[d] -= dom.v[d];
        id[d] -= dom.v[d];
    }
    bool ok = true;
    for (int d = 0; d < 3; ++d)
        ok &= ip[d] >= H && ip[d] + H <= np.v[d] - 1 && id[d] >= H && id[d] + H <= np.v[d];
    if (!ok) {  // position outside the patch: no memory access, NaN result
        for (int c = 0; c < 3; ++c) Ep[c * n + i] = Bp[c * n + i] = __builtin_nan("");
        return;
    }
    const int ny = np.v[1], nz = np.v[2];
    Ep[i] = gather3s<H, O>(cd[0], cp[1], cp[2], Ex, id[0], ip[1], ip[2], ny, nz);
    Bp[n + i] = gather3s<H, O>(cd[0], cp[1], cd[2], By, id[0], ip[1], id[2], ny, nz + 1);
    Ep[n + i] = gather3s<H, O>(cp[0], cd[1], cp[2], Ey, ip[0], id[1], ip[2], ny + 1, nz);
    Bp[i] = gather3s<H, O>(cp[0], cd[1], cd[2], Bx, ip[0], id[1], id[2], ny + 1, nz + 1);
    Ep[2 * n + i] = gather3s<H, O>(cp[0], cp[1], cd[2], Ez, ip[0], ip[1], id[2], ny, nz + 1);
    Bp[2 * n + i] = gather3s<H, O>(cd[0], cd[1], cp[2], Bz, id[0], id[1], ip[2], ny + 1, nz);
    for (int d = 0; d < 3; ++d) {
        iold[d * n + i] = ip[d];
        dold[d * n + i] = dp[d];
    }
}

// Interpolator2D2Order::fieldsWrapper.
__global__ void k_interp2d(const double *Ex, const double *Ey, const double *Ez, const double *Bx, const double *By,
                           const double *Bz, Ints3 np, Ints3 dom, Dbl3 dinv, int64_t n, const double *x,
                           const double *y, double *Ep, double *Bp, int32_t *iold, double *dold)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double pos[2] = {x[i], y[i]};
    double cp[2][5], cd[2][5], dp[2];
    int ip[2], id[2];
    for (int d = 0; d < 2; ++d) {
        const double pn = pos[d] * dinv.v[d];
        ip[d] = (int)round(pn);
        dp[d] = pn - (double)ip[d];
        spline2(dp[d], cp[d]);
        id[d] = (int)round(pn + 0.5);
        spline2(pn - (double)id[d] + 0.5, cd[d]);
        ip[d] -= dom.v[d];
        id[d] -= dom.v[d];
    }
    bool ok = true;
    for (int d = 0; d < 2; ++d) ok &= ip[d] >= 1 && ip[d] + 1 <= np.v[d] - 1 && id[d] >= 1 && id[d] + 1 <= np.v[d];
    if (!ok) {
        for (int c = 0; c < 3; ++c) Ep[c * n + i] = Bp[c * n + i] = __builtin_nan("");
        return;
    }
    const int ny = np.v[1];
    Ep[i] = gather2s<1>(cd[0], cp[1], Ex, id[0], ip[1], ny);
    Ep[n + i] = gather2s<1>(cp[0], cd[1], Ey, ip[0], id[1], ny + 1);
    Ep[2 * n + i] = gather2s<1>(cp[0], cp[1], Ez, ip[0], ip[1], ny);
    Bp[i] = gather2s<1>(cp[0], cd[1], Bx, ip[0], id[1], ny + 1);
    Bp[n + i] = gather2s<1>(cd[0], cp[1], By, id[0], ip[1], ny);
    Bp[2 * n + i] = gather2s<1>(cd[0], cd[1], Bz, id[0], id[1], ny + 1);
    for (int d = 0; d < 2; ++d) {
        iold[d * n + i] = ip[d];
        dold[d * n + i] = dp[d];
    }
}

// PusherBoris::operator().
__global__ void k_boris(int ndim, double qmh, double dt, int64_t n, double *x, double *y, double *z, double *px,
                        double *py, double *pz, const double *Ep, const double *Bp, double *invgf)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double E[3] = {Ep[i], Ep[n + i], Ep[2 * n + i]};
    const double B[3] = {Bp[i], Bp[n + i], Bp[2 * n + i]};
    double u[3] = {px[i], py[i], pz[i]}, dxp[3], g;
    boris(qmh, dt, E, B, u, dxp, g);
    invgf[i] = g;
    px[i] = u[0];
    py[i] = u[1];
    pz[i] = u[2];
    x[i] += dxp[0];
    if (ndim > 1) {
        y[i] += dxp[1];
        if (ndim > 2) z[i] += dxp[2];
    }
}

struct Proj3Args {
    double *J[3];
    int dims[3][3];
    Ints3 dom;
    Dbl3 dinv, cr_scale;  // cr = cw * dx/dt
    double cw_scale;
    int64_t n;
    const double *x[3];
    const double *w;
    const int32_t *iold;
    const double *dold;
};

// Returns false (and touches no J point) when the particle's stencil would
// leave the patch arrays or it moved by more than one cell.
template <int ORDER>
__device__ inline bool proj3_particle_shapes(const Proj3Args &a, int64_t i, double (&S0)[3][7], double (&S1)[3][7],
                                             double (&DS)[3][7], int *io)
{
    constexpr int H = ORDER / 2;
    bool ok = true;
    for (int d = 0; d < 3; ++d) {
        io[d] = a.iold[d * a.n + i];
        const double pn = a.x[d][i] * a.dinv.v[d];
        const int sh = (int)round(pn) - (io[d] + a.dom.v[d]);
        ok &= io[d] - (H + 1) >= 0 && io[d] + H + 1 <= a.dims[(d + 1) % 3][d] - 1 && sh >= -1 && sh <= 1;
        esirkepov_shapes<ORDER>(a.dold[d * a.n + i], pn, io[d] + a.dom.v[d], S0[d], S1[d], DS[d]);
    }
    return ok;
}

// Projector3D{2,4}Order::currents with FP64 atomics, one thread per particle.
// (launched with 128 threads; register budget as k_interp3d)
template <int ORDER>
__global__ void __launch_bounds__(128, 2) k_proj3d_atomic(Proj3Args a)
{
    constexpr int H = ORDER / 2;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    double S0[3][7], S1[3][7], DS[3][7];
    int io[3];
    if (!proj3_particle_shapes<ORDER>(a, i, S0, S1, DS, io)) return;
    const double cw = a.cw_scale * a.w[i];
    const double cr[3] = {cw * a.cr_scale.v[0], cw * a.cr_scale.v[1], cw * a.cr_scale.v[2]};
    esirkepov3d<ORDER>(S0, DS, cr, [&](int c, int u, int v, int k, double val) {
        if (val == 0.) return;
        const int *dm = a.dims[c];
        const int64_t idx = ((int64_t)(io[0] - (H + 1) + u) * dm[1] + (io[1] - (H + 1) + v)) * dm[2] +
                            (io[2] - (H + 1) + k);
        unsafeAtomicAdd(&a.J[c][idx], val);
    });
}

// The same currents over particles binned by their old node: bin = the 4^3
// nodes it lies in.  One workgroup per bin, or per share of a crowded one, sums
// its particles' stencils (a tile of 6 + 2H points per axis) in LDS and flushes
// the tile once, instead of adding 54 to 400 contributions per particle to global memory, which the
// memory-side FP64 atomics bound at 4e10 per second whatever the order of
// the particles.  The particles are not moved: the bins list their indices.
// The strides of the tile put the 64 nodes of a bin, at one stencil offset,
// two to a bank pair.
// Binning pays from this many particles on.  Sorted / unsorted arrays,
// microseconds, per-particle atomics against bins: order 2, 4,096 particles
// 20 / 31 against 22 / 22, 8,192 29 / 47 against 23 / 23, 32,768 88 / 160
// against 39 / 40, 2.1e6 4,000 / 7,222 against 180 / 481; order 4, 64
// particles 39 / 40 against 24 / 23, 512 54 / 79 against 24 / 24, 32,768 432 /
// 775 against 61 / 62, 2.1e6 19,020 / 34,860 against 622 / 670.
constexpr int64_t bin_min(int order) { return order == 2 ? 8192 : 64; }

// Up to this many particles one workgroup does all of the binning: four
// launches less against the work of one CU.  Whole call, one workgroup against
// many (sorted / unsorted): order 2, 8,192 particles 23 / 23 against 37 / 36,
// 12,288 27 / 28 against 37 / 36, 16,384 32 / 34 against 40 / 36, 32,768 49 / 55
// against 39 / 40; order 4, 64 particles 24 against 35, 12,288 46 / 44 against
// 45 / 42, 16,384 58 / 56 against 54 / 49.
constexpr int64_t bin_one_max(int order) { return order == 2 ? 12288 : 8192; }

template <int ORDER>
struct BinTile {
    static constexpr int H = ORDER / 2, T = 6 + 2 * H, SY = 10, SX = 104, SC = T * SX;
};

struct Bins {
    int nb[3];      // bins per axis
    int nbins, share;
    int *count;     // per bin
    int *start;     // per bin, and the total
    int *key, *rank, *list;  // per particle
    int2 *further;  // bin and number of the further shares of crowded bins
    int *nfurther;
};

// A crowded bin is worked on in equal shares of at most b.share particles, by
// as many workgroups: with one workgroup per bin a species that lies in a few
// bins was left to a few CUs (6e5 particles within 2^3 cells, order 4:
// interpolation 34 ms, projection 66 ms; 0.14 and 0.43 ms in shares).
__device__ inline int bin_shares(const Bins &b, int count) { return (count + b.share - 1) / b.share; }

// Work items: the first share of every bin, then the further ones; empty
// beyond them.
struct Share {
    int bin, first, last;  // its places in the list
};
__device__ inline Share bin_item(const Bins &b, int item)
{
    int bin = item, k = 0;
    if (item >= b.nbins) {
        if (item - b.nbins >= *b.nfurther) return Share{0, 0, 0};
        const int2 f = b.further[item - b.nbins];
        bin = f.x;
        k = f.y;
    }
    Share w{bin, b.start[bin], b.start[bin + 1]};
    const int count = w.last - w.first;
    if (count > b.share) {
        const int shares = bin_shares(b, count), per = (count + shares - 1) / shares;
        w.first += k * per;
        w.last = w.last - w.first < per ? w.last : w.first + per;
    }
    return w;
}

// Starts of all bins from their counts, and the further shares, by one
// workgroup, 4,096 bins at a time; keep: the starts take the counts' place too.
constexpr int kBinThreads = 1024;
__device__ inline void bin_scan(const Bins &b, int *count, bool keep)
{
    constexpr int WAVES = kBinThreads / 64;
    __shared__ int part[2][WAVES];
    __shared__ int nfurther;
    if (threadIdx.x == 0) nfurther = 0;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int before = 0;
    for (int q0 = 0, k = 0; q0 < b.nbins; q0 += 4 * kBinThreads, k ^= 1) {
        const int q = q0 + 4 * threadIdx.x, m = b.nbins - q;
        int c[4] = {0, 0, 0, 0};
        if (m >= 4) {
            const int4 v = *reinterpret_cast<const int4 *>(count + q);
            c[0] = v.x;
            c[1] = v.y;
            c[2] = v.z;
            c[3] = v.w;
        } else {
            for (int i = 0; i < m; ++i) c[i] = count[q + i];
        }
        const int sum = c[0] + c[1] + c[2] + c[3];
        int incl = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int t = __shfl_up(incl, o, 64);
            if (lane >= o) incl += t;
        }
        if (lane == 63) part[k][wave] = incl;
        __syncthreads();
        int at = before + incl - sum;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            if (w < wave) at += part[k][w];
            before += part[k][w];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (i >= m) break;
            b.start[q + i] = at;
            if (keep) count[q + i] = at;
            at += c[i];
            if (c[i] > b.share) {
                const int more = bin_shares(b, c[i]) - 1, f = atomicAdd(&nfurther, more);
                for (int j = 0; j < more; ++j) b.further[f + j] = make_int2(q + i, j + 1);
            }
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        b.start[b.nbins] = before;
        *b.nfurther = nfurther;
    }
}

// Bin of particle i by its old node, or -1 for one whose stencil would leave
// the arrays.
template <int ORDER>
struct NodeKey {
    Proj3Args a;
    __device__ int64_t n() const { return a.n; }
    __device__ int operator()(const Bins &b, int64_t i) const;
};

template <int ORDER>
__device__ inline int NodeKey<ORDER>::operator()(const Bins &b, int64_t i) const
{
    constexpr int H = ORDER / 2;
    int key = 0;
    bool ok = true;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        const int io = a.iold[d * a.n + i];
        ok &= io - (H + 1) >= 0 && io + H + 1 <= a.dims[(d + 1) % 3][d] - 1;
        key = key * b.nb[d] + (io >> 2);
    }
    return ok ? key : -1;
}

// Bin and place in the bin of every particle.  Lanes of a wavefront with
// equal bins in a row (particles in cell order) share one atomic.  For more
// bins than a workgroup counts in LDS.
template <class Key>
__global__ void __launch_bounds__(256) k_bin_count(Key of, Bins b)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & 63;
    const int key = i < of.n() ? of(b, i) : -1;
    int head, len;
    key_run((uint32_t)key, head, len);
    int first = 0;
    if (lane == head && key >= 0) first = atomicAdd(&b.count[key], len);
    first = __shfl(first, head, 64);
    if (i < of.n()) {
        b.key[i] = key;
        b.rank[i] = first + lane - head;
    }
}

// The same counted in LDS first, `per` particles a thread, and added to the
// bins' counts by one atomic per workgroup and bin: the atomics of one bin
// queue up otherwise (order 2, whole call, with k_bin_count: 2.6e5 particles
// 88 us in cell order and 131 shuffled, here 56 and 69; 2.1e6 307 and 558, here
// 211 and 473).
constexpr int kBinLds = 8192;

template <class Key>
__device__ inline void bin_count_lds(const Key &of, const Bins &b, int nbins, int64_t i0, int per, int *h)
{
    for (int q = threadIdx.x; q < nbins; q += kBinThreads) h[q] = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63;
#pragma unroll 4
    for (int k = 0; k < per; ++k) {
        const int64_t i = i0 + (int64_t)k * kBinThreads + threadIdx.x;
        const int key = i < of.n() ? of(b, i) : -1;
        int head, len;
        key_run((uint32_t)key, head, len);
        int first = 0;
        if (lane == head && key >= 0) first = atomicAdd(&h[key], len);
        first = __shfl(first, head, 64);
        if (i < of.n()) {
            b.key[i] = key;
            b.rank[i] = first + lane - head;
        }
    }
    __syncthreads();
}

template <class Key>
__global__ void __launch_bounds__(kBinThreads) k_bin_count_lds(Key of, Bins b, int nbins, int per)
{
    __shared__ int h[kBinLds];
    const int64_t i0 = (int64_t)blockIdx.x * per * kBinThreads;
    bin_count_lds(of, b, nbins, i0, per, h);
#pragma unroll 4
    for (int q = threadIdx.x; q < nbins; q += kBinThreads)
        if (h[q]) h[q] = atomicAdd(&b.count[q], h[q]);
    __syncthreads();
#pragma unroll 4
    for (int k = 0; k < per; ++k) {
        const int64_t i = i0 + (int64_t)k * kBinThreads + threadIdx.x;
        if (i < of.n() && b.key[i] >= 0) b.rank[i] += h[b.key[i]];
    }
}

// All of the binning by one workgroup: count, start of the bins and list, one
// launch instead of four.
template <class Key>
__global__ void __launch_bounds__(kBinThreads) k_bin_one(Key of, Bins b, int nbins, int per)
{
    __shared__ __align__(16) int h[kBinLds];
    bin_count_lds(of, b, nbins, 0, per, h);
    bin_scan(b, h, true);
    __syncthreads();
#pragma unroll 4
    for (int k = 0; k < per; ++k) {
        const int64_t i = (int64_t)k * kBinThreads + threadIdx.x;
        if (i < of.n() && b.key[i] >= 0) b.list[h[b.key[i]] + b.rank[i]] = (int)i;
    }
}

__global__ void __launch_bounds__(kBinThreads) k_bin_scan(Bins b)
{
    bin_scan(b, b.count, false);
}

__global__ void __launch_bounds__(256) k_bin_fill(Bins b, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int key = b.key[i];
    if (key >= 0) b.list[b.start[key] + b.rank[i]] = (int)i;
}

// Deposit of particle i on the tile: the narrow stencil for one that keeps
// its node on every axis, the wide one otherwise.  Returns false, without a
// deposit, for a particle whose node changes when wide is not set.
template <int ORDER, bool WIDE>
__device__ inline bool bin_deposit(const Proj3Args &a, int64_t i, double *sJ)
{
    using BT = BinTile<ORDER>;
    double S0[3][ORDER + 2], DS[3][ORDER + 2], pn[3], dold[3];
    int w0[3], io[3], moved = 0;
    bool ok = true;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
        io[d] = a.iold[d * a.n + i];
        dold[d] = a.dold[d * a.n + i];
        pn[d] = a.x[d][i] * a.dinv.v[d];
        const int sh = (int)round(pn[d]) - (io[d] + a.dom.v[d]);
        ok &= sh >= -1 && sh <= 1;
        moved |= sh;
    }
    if (!ok) return true;
    if (!WIDE && moved) return false;
#pragma unroll
    for (int d = 0; d < 3; ++d) esirkepov_window<ORDER>(dold[d], pn[d], io[d] + a.dom.v[d], S0[d], DS[d], w0[d]);
    const double cw = a.cw_scale * a.w[i];
    const double cr[3] = {cw * a.cr_scale.v[0], cw * a.cr_scale.v[1], cw * a.cr_scale.v[2]};
    double *t = sJ + (io[0] & 3) * BT::SX + (io[1] & 3) * BT::SY + (io[2] & 3);
    if constexpr (!WIDE) {
        const int one[3] = {1, 1, 1};
        esirkepov3d_fact<ORDER, ORDER + 1, ORDER>(S0, DS, one, cr, [&](int c, int u, int v, int k, double val) {
            atomicAdd(&t[c * BT::SC + u * BT::SX + v * BT::SY + k], val);
        });
    } else {
        esirkepov3d_fact<ORDER, ORDER + 2, ORDER + 1>(S0, DS, w0, cr, [&](int c, int u, int v, int k, double val) {
            atomicAdd(&t[c * BT::SC + u * BT::SX + v * BT::SY + k], val);
        });
    }
    return true;
}

// One workgroup per share of a bin.  The particles that change node are queued and
// deposited by a second pass, so that the first runs the narrow stencil with
// all lanes.  A lane takes a run of the bin's list and a wavefront every fourth
// place of its lanes' runs: neighbours in the list, mostly of one node where
// the arrays are in cell order, do not meet on the same words (order 4, 2.1e6
// particles in cell order 911 us with neighbours on neighbouring lanes, 622 so;
// in no order 668 / 670).
template <int ORDER>
__global__ void __launch_bounds__(256) k_proj3d_bins(Proj3Args a, Bins b)
{
    using BT = BinTile<ORDER>;
    constexpr int T = BT::T, QCAP = 256;
    __shared__ double sJ[3 * BT::SC];
    __shared__ int sQ[QCAP];
    __shared__ int sQn;
    const Share w = bin_item(b, blockIdx.x);
    const int n = w.last - w.first;
    if (n == 0) return;  // uniform across the workgroup
    for (int t = threadIdx.x; t < 3 * BT::SC; t += blockDim.x) sJ[t] = 0.;
    if (threadIdx.x == 0) sQn = 0;
    __syncthreads();
    const int per = (n + 63) / 64, first = (threadIdx.x & 63) * per;
    for (int k = threadIdx.x >> 6; k < per && first + k < n; k += blockDim.x >> 6) {
        const int i = b.list[w.first + first + k];
        if (bin_deposit<ORDER, false>(a, i, sJ)) continue;
        const int q = atomicAdd(&sQn, 1);
        if (q < QCAP) sQ[q] = i;
        else bin_deposit<ORDER, true>(a, i, sJ);
    }
    __syncthreads();
    const int nq = sQn < QCAP ? sQn : QCAP;
    for (int q = threadIdx.x; q < nq; q += blockDim.x) bin_deposit<ORDER, true>(a, sQ[q], sJ);
    __syncthreads();
    // array index of tile point 0: the bin's first node less H + 1
    const int bz = w.bin % b.nb[2], by = (w.bin / b.nb[2]) % b.nb[1], bx = w.bin / (b.nb[2] * b.nb[1]);
    const int o[3] = {4 * bx - BT::H - 1, 4 * by - BT::H - 1, 4 * bz - BT::H - 1};
    for (int t = threadIdx.x; t < T * T * T; t += blockDim.x) {
        const int q[3] = {t / (T * T), (t / T) % T, t % T};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const double v = sJ[c * BT::SC + q[0] * BT::SX + q[1] * BT::SY + q[2]];
            const int *dm = a.dims[c];
            const int i = o[0] + q[0], j = o[1] + q[1], k = o[2] + q[2];
            if (v == 0. || i < 0 || i >= dm[0] || j < 0 || j >= dm[1] || k < 0 || k >= dm[2]) continue;
            unsafeAtomicAdd(&a.J[c][((int64_t)i * dm[1] + j) * dm[2] + k], v);
        }
    }
}

// Same contributions in particle order: one wavefront, lanes over
// (component, transverse column), ordered L2 atomics and a barrier per
// particle; every J point sums in index order like the CPU operator.
template <int ORDER>
__global__ void __launch_bounds__(64) k_proj3d_ordered(Proj3Args a)
{
    constexpr int H = ORDER / 2, S = 2 * H + 3;
    for (int64_t i = 0; i < a.n; ++i) {
        double S0[3][7], S1[3][7], DS[3][7];
        int io[3];
        if (!proj3_particle_shapes<ORDER>(a, i, S0, S1, DS, io)) continue;  // uniform across the wavefront
        const double cw = a.cw_scale * a.w[i];
        const double cr[3] = {cw * a.cr_scale.v[0], cw * a.cr_scale.v[1], cw * a.cr_scale.v[2]};
        for (int task = threadIdx.x; task < 3 * S * S; task += 64) {
            const int c = task / (S * S), col = task % (S * S);
            const int u = col / S, v = col % S;
            const int *dm = a.dims[c];
            double W;
            if (c == 0) W = weight3(S0[1], DS[1], S0[2], DS[2], u, v);
            else if (c == 1) W = weight3(S0[2], DS[2], S0[0], DS[0], v, u);
            else W = weight3(S0[0], DS[0], S0[1], DS[1], u, v);
            const double t = cr[c] * W;
            double acc = 0.;
            for (int r = 1; r < S; ++r) {
                if constexpr (ORDER == 2) acc -= DS[c][r - 1] * t;
                else acc -= cr[c] * DS[c][r - 1] * W;
                int ii, jj, kk;
                if (c == 0) { ii = r; jj = u; kk = v; }
                else if (c == 1) { ii = u; jj = r; kk = v; }
                else { ii = u; jj = v; kk = r; }
                const int64_t idx = ((int64_t)(io[0] - (H + 1) + ii) * dm[1] + (io[1] - (H + 1) + jj)) * dm[2] +
                                    (io[2] - (H + 1) + kk);
                unsafeAtomicAdd(&a.J[c][idx], acc);
            }
        }
        __syncthreads();
    }
}

struct Proj2Args {
    double *J[3];
    int ny[3];  // second extent of Jx, Jy, Jz
    int nx;     // primal extent along x
    Ints3 dom;
    Dbl3 dinv, cr_scale;
    double cw_scale;
    int64_t n;
    const double *x, *y, *pz, *w, *invgf;
    const int32_t *iold;
    const double *dold;
};

__device__ inline bool proj2_particle(const Proj2Args &a, int64_t i, double (&S0)[3][7], double (&S1)[3][7],
                                      double (&DS)[3][7], int *io, double &crx, double &cry, double &crz)
{
    const double pos[2] = {a.x[i], a.y[i]};
    bool ok = true;
    for (int d = 0; d < 2; ++d) {
        io[d] = a.iold[d * a.n + i];
        const double pn = pos[d] * a.dinv.v[d];
        const int sh = (int)round(pn) - (io[d] + a.dom.v[d]);
        // Jz (p,p) has the primal extents: ny[2] along y, nprim_x along x
        const int ext = d == 0 ? a.nx : a.ny[2];
        ok &= io[d] - 2 >= 0 && io[d] + 2 <= ext - 1 && sh >= -1 && sh <= 1;
        esirkepov_shapes<2>(a.dold[d * a.n + i], pn, io[d] + a.dom.v[d], S0[d], S1[d], DS[d]);
    }
    const double cw = a.cw_scale * a.w[i];
    crx = cw * a.cr_scale.v[0];
    cry = cw * a.cr_scale.v[1];
    crz = cw * kThird * a.pz[i] * a.invgf[i];
    return ok;
}

__global__ void k_proj2d_atomic(Proj2Args a)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    double S0[3][7], S1[3][7], DS[3][7], crx, cry, crz;
    int io[2];
    if (!proj2_particle(a, i, S0, S1, DS, io, crx, cry, crz)) return;
    esirkepov2d(S0, S1, DS, crx, cry, crz, [&](int c, int u, int v, double val) {
        if (val == 0.) return;
        unsafeAtomicAdd(&a.J[c][(int64_t)(io[0] - 2 + u) * a.ny[c] + (io[1] - 2 + v)], val);
    });
}

__global__ void __launch_bounds__(64) k_proj2d_ordered(Proj2Args a)
{
    const int lane = threadIdx.x;
    for (int64_t i = 0; i < a.n; ++i) {
        double S0[3][7], S1[3][7], DS[3][7], crx, cry, crz;
        int io[2];
        if (!proj2_particle(a, i, S0, S1, DS, io, crx, cry, crz)) continue;  // uniform across the wavefront
        if (lane < 5) {
            const int jj = lane;
            double acc = 0.;
            for (int ii = 1; ii < 5; ++ii) {
                if (jj == 0) acc -= crx * DS[0][ii - 1] * (0.5 * DS[1][0]);
                else acc -= crx * DS[0][ii - 1] * (S0[1][jj] + 0.5 * DS[1][jj]);
                unsafeAtomicAdd(&a.J[0][(int64_t)(io[0] - 2 + ii) * a.ny[0] + (io[1] - 2 + jj)], acc);
            }
        } else if (lane < 10) {
            const int ii = lane - 5;
            const double ty = S0[0][ii] + 0.5 * DS[0][ii];
            double acc = 0.;
            for (int jj = 1; jj < 5; ++jj) {
                acc -= cry * DS[1][jj - 1] * ty;
                unsafeAtomicAdd(&a.J[1][(int64_t)(io[0] - 2 + ii) * a.ny[1] + (io[1] - 2 + jj)], acc);
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
            unsafeAtomicAdd(&a.J[2][(int64_t)(io[0] - 2 + ii) * a.ny[2] + (io[1] - 2 + jj)], v);
        }
        __syncthreads();
    }
}

// MA_Solver3D_norm on one patch array: each component over its own extent.
__global__ void k_ma3d_patch(double *Ex, double *Ey, double *Ez, const double *Bx, const double *By,
                             const double *Bz, const double *Jx, const double *Jy, const double *Jz, Ints3 np,
                             double dt, double dtx, double dty, double dtz)
{
    const int64_t nxp = np.v[0], nyp = np.v[1], nzp = np.v[2], nxd = nxp + 1, nyd = nyp + 1, nzd = nzp + 1;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nEx = nxd * nyp * nzp, nEy = nxp * nyd * nzp, nEz = nxp * nyp * nzd;
    if (t < nEx) {
        const int64_t i = t / (nyp * nzp), j = (t / nzp) % nyp, k = t % nzp;
        Ex[t] += -dt * Jx[t] + dty * (Bz[(i * nyd + j + 1) * nzp + k] - Bz[(i * nyd + j) * nzp + k]) -
                 dtz * (By[(i * nyp + j) * nzd + k + 1] - By[(i * nyp + j) * nzd + k]);
    } else if (t < nEx + nEy) {
        const int64_t e = t - nEx;
        const int64_t i = e / (nyd * nzp), j = (e / nzp) % nyd, k = e % nzp;
        Ey[e] += -dt * Jy[e] - dtx * (Bz[((i + 1) * nyd + j) * nzp + k] - Bz[(i * nyd + j) * nzp + k]) +
                 dtz * (Bx[(i * nyd + j) * nzd + k + 1] - Bx[(i * nyd + j) * nzd + k]);
    } else if (t < nEx + nEy + nEz) {
        const int64_t e = t - nEx - nEy;
        const int64_t i = e / (nyp * nzd), j = (e / nzd) % nyp, k = e % nzd;
        Ez[e] += -dt * Jz[e] + dtx * (By[((i + 1) * nyp + j) * nzd + k] - By[(i * nyp + j) * nzd + k]) -
                 dty * (Bx[(i * nyd + j + 1) * nzd + k] - Bx[(i * nyd + j) * nzd + k]);
    }
}

// MF_Solver3D_Yee on one patch array: interior of the dual axes only.
__global__ void k_mf3d_patch(double *Bx, double *By, double *Bz, const double *Ex, const double *Ey,
                             const double *Ez, Ints3 np, double dtx, double dty, double dtz)
{
    const int64_t nxp = np.v[0], nyp = np.v[1], nzp = np.v[2], nxd = nxp + 1, nyd = nyp + 1, nzd = nzp + 1;
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nBx = nxp * nyd * nzd, nBy = nxd * nyp * nzd, nBz = nxd * nyd * nzp;
    if (t < nBx) {
        const int64_t i = t / (nyd * nzd), j = (t / nzd) % nyd, k = t % nzd;
        if (j < 1 || j >= nyd - 1 || k < 1 || k >= nzd - 1) return;
        Bx[t] += -dty * (Ez[(i * nyp + j) * nzd + k] - Ez[(i * nyp + j - 1) * nzd + k]) +
                 dtz * (Ey[(i * nyd + j) * nzp + k] - Ey[(i * nyd + j) * nzp + k - 1]);
    } else if (t < nBx + nBy) {
        const int64_t e = t - nBx;
        const int64_t i = e / (nyp * nzd), j = (e / nzd) % nyp, k = e % nzd;
        if (i < 1 || i >= nxd - 1 || k < 1 || k >= nzd - 1) return;
        By[e] += -dtz * (Ex[(i * nyp + j) * nzp + k] - Ex[(i * nyp + j) * nzp + k - 1]) +
                 dtx * (Ez[(i * nyp + j) * nzd + k] - Ez[((i - 1) * nyp + j) * nzd + k]);
    } else if (t < nBx + nBy + nBz) {
        const int64_t e = t - nBx - nBy;
        const int64_t i = e / (nyd * nzp), j = (e / nzp) % nyd, k = e % nzp;
        if (i < 1 || i >= nxd - 1 || j < 1 || j >= nyd - 1) return;
        Bz[e] += -dtx * (Ey[(i * nyd + j) * nzp + k] - Ey[((i - 1) * nyd + j) * nzp + k]) +
                 dty * (Ex[(i * nyp + j) * nzp + k] - Ex[(i * nyp + j - 1) * nzp + k]);
    }
}

int op_fail(int code, const std::string &m)
{
    set_error(m);
    return code;
}

// Particles of a share: 1,024, more where a uniform plasma has more to a bin
// (a bin with four times the mean is split) as long as there are 2,048 shares.
// Uniform, 8.4e6 particles and 1,223 to a bin, order 4: interpolation 1,372 us
// in shares of 1,024, 1,320 unsplit.
int64_t share_size(int64_t nbins, int64_t n) { return std::max<int64_t>(1024, std::min(4 * n / nbins, n / 2048)); }

// Workgroups over the shares: there are at most n / share further ones, and a
// workgroup without one ends at its first load (2,048 of them beside the 6,859
// bins of 2.1e6 particles: nothing; the interpolation as a loop over the shares
// took 432 us instead of 407).
int64_t share_blocks(int64_t nbins, int64_t n) { return nbins + n / share_size(nbins, n); }

// 4-byte words of scratch of the binning.
int64_t bins_words(int64_t nbins, int64_t n) { return 2 * (n / share_size(nbins, n)) + 2 + 2 * nbins + 2 + 3 * n; }

// Lists the n particles by bin: b.start and b.list, in ws (bins_words).
template <class Key>
void launch_binning(const Key &of, Bins &b, int64_t nbins, int64_t n, int64_t one_max, int *ws, hipStream_t st)
{
    b.nbins = (int)nbins;
    b.share = (int)share_size(nbins, n);
    b.count = ws;  // (read four at a time)
    b.further = (int2 *)(b.count + (nbins + 1) / 2 * 2);
    b.nfurther = (int *)(b.further + n / b.share);
    b.start = b.nfurther + 2;
    b.key = b.start + nbins + 1;
    b.rank = b.key + n;
    b.list = b.rank + n;
    const dim3 wide(kBinThreads);
    if (nbins <= kBinLds && n <= one_max) {
        hipLaunchKernelGGL(k_bin_one<Key>, dim3(1), wide, 0, st, of, b, (int)nbins, (int)nblk(n, kBinThreads));
        return;
    }
    launch_fill_i32(b.count, nbins, 0, st);
    if (nbins <= kBinLds) {
        // a workgroup per CU where there are that many particles, 16 particles
        // a thread at most, and half a bin's worth a thread at least, as the
        // bins are cleared and added up once per workgroup
        const int64_t want = std::max<int64_t>(n / (256 * kBinThreads), nbins / (2 * kBinThreads));
        const int per = (int)std::min<int64_t>(std::max<int64_t>(want, 1), 16);
        hipLaunchKernelGGL(k_bin_count_lds<Key>, dim3(nblk(n, per * kBinThreads)), wide, 0, st, of, b, (int)nbins, per);
    } else {
        hipLaunchKernelGGL(k_bin_count<Key>, dim3(nblk(n, 256)), dim3(256), 0, st, of, b);
    }
    hipLaunchKernelGGL(k_bin_scan, dim3(1), wide, 0, st, b);
    hipLaunchKernelGGL(k_bin_fill, dim3(nblk(n, 256)), dim3(256), 0, st, b, n);
}

// The binned projection where it is the faster one and has its scratch;
// false otherwise.
bool launch_bins(int order, const Proj3Args &a, hipStream_t st)
{
    if (a.n < bin_min(order) || a.n >= (1ll << 31)) return false;
    Bins b{};
    int64_t nbins = 1;
    for (int d = 0; d < 3; ++d) {
        b.nb[d] = (a.dims[(d + 1) % 3][d] + 3) / 4;
        nbins *= b.nb[d];
    }
    // Sparse: a workgroup per bin for one particle, and at order 2 the launches of
    // the binning, which cost what the atomics of 5,000 particles do.  Order 2,
    // atomics against bins, cell order: 4,913 bins, 8,192 particles 37.5 / 35.2 us,
    // 10,000 42.3 / 38.2; 8,000 bins, 10,000 42.6 / 47.9, 14,000 55.1 / 56.5, 16,384
    // 62.8 / 56.7; 9,261 bins, 16,384 65.0 / 54.1; 15,625 bins, 22,000 82.7 / 72.8;
    // 17,576 bins, 18,000 70 / 78, 24,000 89.6 / 78.6; 35,937 bins, 42,500 158 /
    // 133; 274,625 bins, 280,000 1,007 / 1,004.  Order 4, 6,859 bins, 7,000 139 / 67.
    if (a.n < (order == 2 ? nbins + std::min<int64_t>(2 * nbins / 3, 5120) : nbins)) return false;
    if (share_blocks(nbins, a.n) >= (1ll << 24)) return false;  // 2^32 threads a launch
    const Workspace ws((size_t)bins_words(nbins, a.n) * sizeof(int), st);
    if (!ws.p) return false;
    const dim3 block(256), grid((unsigned)share_blocks(nbins, a.n));
    if (order == 2) {
        launch_binning(NodeKey<2>{a}, b, nbins, a.n, bin_one_max(2), (int *)ws.p, st);
        hipLaunchKernelGGL(k_proj3d_bins<2>, grid, block, 0, st, a, b);
    } else {
        launch_binning(NodeKey<4>{a}, b, nbins, a.n, bin_one_max(4), (int *)ws.p, st);
        hipLaunchKernelGGL(k_proj3d_bins<4>, grid, block, 0, st, a, b);
    }
    return true;
}

// Interpolation of particles binned by node: a bin's particles gather from a
// tile of the six fields in LDS (5 + 2H points per axis), by the same
// products and sums as k_interp3d, so to the same bits.  Gathered from global
// memory, a particle's rows come through the L1 (64 bytes a clock, half of what
// LDS gives) while its neighbours are near it, and through the L2 when the
// array is in no order.  The gathers are kept apart (scheduling barriers): 23
// registers spilled at three wavefronts per SIMD, 415 us for 2.1e6 particles
// against 438 without, and against 439 with two wavefronts and no spills.
struct Interp3Args {
    const double *F[6];  // Ex, Ey, Ez, Bx, By, Bz
    Ints3 np, dom;
    Dbl3 dinv;
    int64_t n;
    const double *x[3];
    double *Ep, *Bp;
    int32_t *iold;
    double *dold;
};

// Bin of particle i by its node; -1, and NaN as its result, for one outside
// the patch.
template <int ORDER>
struct PlaceKey {
    Interp3Args a;
    __device__ int64_t n() const { return a.n; }
    __device__ int operator()(const Bins &b, int64_t i) const
    {
        constexpr int H = ORDER / 2;
        int key = 0;
        bool ok = true;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const double pn = a.x[d][i] * a.dinv.v[d];
            const int ip = (int)round(pn) - a.dom.v[d], id = (int)round(pn + 0.5) - a.dom.v[d];
            ok &= ip >= H && ip + H <= a.np.v[d] - 1 && id >= H && id + H <= a.np.v[d];
            key = key * b.nb[d] + (ip >> 2);
        }
        if (!ok)
            for (int c = 0; c < 3; ++c) a.Ep[c * a.n + i] = a.Bp[c * a.n + i] = __builtin_nan("");
        return ok ? key : -1;
    }
};

template <int ORDER>
__global__ void __launch_bounds__(256, 3) k_interp3d_bins(Interp3Args a, Bins b)
{
    constexpr int H = ORDER / 2, T = 5 + 2 * H, SY = T, SX = T * T + 3, SF = T * SX;
    __shared__ double s[6 * SF];
    const Share w = bin_item(b, blockIdx.x);
    if (w.first == w.last) return;  // uniform across the workgroup
    // tile point 0 is point 4 q - H of an axis; points outside an array are read by no particle of the bin
    const int q[3] = {w.bin / (b.nb[1] * b.nb[2]) * 4 - H, w.bin / b.nb[2] % b.nb[1] * 4 - H,
                      w.bin % b.nb[2] * 4 - H};
    for (int t = threadIdx.x; t < T * T * T; t += blockDim.x) {
        const int l[3] = {t / (T * T), t / T % T, t % T};
#pragma unroll
        for (int f = 0; f < 6; ++f) {
            bool in = true;
            int64_t idx = 0;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const int m = a.np.v[d] + ((f < 3) == (f % 3 == d) ? 1 : 0), g = q[d] + l[d];
                in &= g >= 0 && g < m;
                idx = idx * m + g;
            }
            s[f * SF + l[0] * SX + l[1] * SY + l[2]] = in ? a.F[f][idx] : 0.;
        }
    }
    __syncthreads();
    for (int t = w.first + threadIdx.x; t < w.last; t += blockDim.x) {
        const int64_t i = b.list[t];
        double cp[3][5], cd[3][5];
        int lp[3], ld[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const double pn = a.x[d][i] * a.dinv.v[d];
            int ip = (int)round(pn), id = (int)round(pn + 0.5);
            const double dp = pn - (double)ip;
            spline<ORDER>(dp, cp[d]);
            spline<ORDER>(pn - (double)id + 0.5, cd[d]);
            ip -= a.dom.v[d];
            id -= a.dom.v[d];
            lp[d] = ip - q[d];
            ld[d] = id - q[d];
            a.iold[d * a.n + i] = ip;
            a.dold[d * a.n + i] = dp;
        }
        a.Ep[i] = gather3<H, SY, SX>(cd[0], cp[1], cp[2], s + 0 * SF, ld[0], lp[1], lp[2]);
        __builtin_amdgcn_sched_barrier(0);
        a.Ep[a.n + i] = gather3<H, SY, SX>(cp[0], cd[1], cp[2], s + 1 * SF, lp[0], ld[1], lp[2]);
        __builtin_amdgcn_sched_barrier(0);
        a.Ep[2 * a.n + i] = gather3<H, SY, SX>(cp[0], cp[1], cd[2], s + 2 * SF, lp[0], lp[1], ld[2]);
        __builtin_amdgcn_sched_barrier(0);
        a.Bp[i] = gather3<H, SY, SX>(cp[0], cd[1], cd[2], s + 3 * SF, lp[0], ld[1], ld[2]);
        __builtin_amdgcn_sched_barrier(0);
        a.Bp[a.n + i] = gather3<H, SY, SX>(cd[0], cp[1], cd[2], s + 4 * SF, ld[0], lp[1], ld[2]);
        __builtin_amdgcn_sched_barrier(0);
        a.Bp[2 * a.n + i] = gather3<H, SY, SX>(cd[0], cd[1], cp[2], s + 5 * SF, ld[0], ld[1], lp[2]);
    }
}

// Where binning pays: order 4, this many particles, and so many to a bin (the
// tile of a bin is 9^3 points of six fields).  Whole call, cell order / no order,
// k_interp3d against bins: 2.6e5 particles 83 / 205 us against 95 / 142; 5.1e5 159
// / 455 against 146 / 220; 1.0e6, 180 to a bin, 282 / 1,733 against 261 / 378;
// 2.1e6 524 / 4,002 against 415 / 853; but 5.2e5, 90 to a bin, 143 against 195 in
// cell order.  6e5 within 2^3 cells: 260 / 299 against 133 / 145.  Order 2, 2.1e6: 144 / 886 against 166 / 466, left as it is.
constexpr int64_t kInterpBinMin = 1 << 19, kInterpPerBin = 160;

bool launch_interp_bins(int order, const Interp3Args &a, hipStream_t st)
{
    if (order != 4 || a.n < kInterpBinMin || a.n >= (1ll << 31)) return false;
    Bins b{};
    int64_t nbins = 1;
    for (int d = 0; d < 3; ++d) {
        b.nb[d] = (a.np.v[d] + 3) / 4;
        nbins *= b.nb[d];
    }
    if (nbins < 1 || a.n < kInterpPerBin * nbins) return false;
    const Workspace ws((size_t)bins_words(nbins, a.n) * sizeof(int), st);
    if (!ws.p) return false;
    launch_binning(PlaceKey<4>{a}, b, nbins, a.n, bin_one_max(4), (int *)ws.p, st);
    hipLaunchKernelGGL(k_interp3d_bins<4>, dim3((unsigned)share_blocks(nbins, a.n)), dim3(256), 0, st, a, b);
    return true;
}

#define OP_CHECK()                                                              \
    do {                                                                        \
        hipError_t e_ = hipGetLastError();                                      \
        if (e_ != hipSuccess) return op_fail(SMI_ERR_HIP, hipGetErrorString(e_)); \
    } while (0)

}  // namespace

extern "C" {

int smi_interpolate_3d(int order, const double *Ex, const double *Ey, const double *Ez, const double *Bxm,
                       const double *Bym, const double *Bzm, const int np[3], const int dom_begin[3],
                       const double cell_length[3], int64_t n, const double *x, const double *y, const double *z,
                       double *Epart, double *Bpart, int32_t *iold, double *deltaold, void *stream)
{
    if (order != 2 && order != 4) return op_fail(SMI_ERR_INVALID, "order must be 2 or 4");
    if (n <= 0) return SMI_OK;
    Ints3 NP{{np[0], np[1], np[2]}}, D{{dom_begin[0], dom_begin[1], dom_begin[2]}};
    Dbl3 di{{1.0 / cell_length[0], 1.0 / cell_length[1], 1.0 / cell_length[2]}};
    hipStream_t st = (hipStream_t)stream;
    const dim3 grid(nblk(n, 256)), block(256);
    const Interp3Args a{{Ex, Ey, Ez, Bxm, Bym, Bzm}, NP, D, di, n, {x, y, z}, Epart, Bpart, iold, deltaold};
    try {
        if (launch_interp_bins(order, a, st)) {
            OP_CHECK();
            return SMI_OK;
        }
    } catch (const std::exception &e) {
        return op_fail(SMI_ERR_HIP, e.what());
    }
    const bool small = (int64_t)(np[0] + 1) * (np[1] + 1) * (np[2] + 1) < (1ll << 29);
#define SMI_INTERP(O, T)                                                                                             \
    hipLaunchKernelGGL((k_interp3d<O, T>), grid, block, 0, st, Ex, Ey, Ez, Bxm, Bym, Bzm, NP, D, di, n, x, y, z, Epart, \
                       Bpart, iold, deltaold)
    if (order == 2) {
        if (small) SMI_INTERP(2, uint32_t);
        else SMI_INTERP(2, uint64_t);
    } else {
        if (small) SMI_INTERP(4, uint32_t);
        else SMI_INTERP(4, uint64_t);
    }
#undef SMI_INTERP
    OP_CHECK();
    return SMI_OK;
}

int smi_interpolate_2d(int order, const double *Ex, const double *Ey, const double *Ez, const double *Bxm,
                       const double *Bym, const double *Bzm, const int np[2], const int dom_begin[2],
                       const double cell_length[2], int64_t n, const double *x, const double *y, double *Epart,
                       double *Bpart, int32_t *iold, double *deltaold, void *stream)
{
    if (order != 2) return op_fail(SMI_ERR_INVALID, "2D interpolation order must be 2");
    if (n <= 0) return SMI_OK;
    Ints3 NP{{np[0], np[1], 1}}, D{{dom_begin[0], dom_begin[1], 0}};
    Dbl3 di{{1.0 / cell_length[0], 1.0 / cell_length[1], 1.0}};
    hipLaunchKernelGGL(k_interp2d, dim3(nblk(n, 256)), dim3(256), 0, (hipStream_t)stream, Ex, Ey, Ez, Bxm, Bym, Bzm,
                       NP, D, di, n, x, y, Epart, Bpart, iold, deltaold);
    OP_CHECK();
    return SMI_OK;
}

int smi_push_boris(int ndim, double charge, double mass, double timestep, int64_t n, double *x, double *y, double *z,
                   double *px, double *py, double *pz, const double *Epart, const double *Bpart, double *invgf,
                   void *stream)
{
    if (!(mass > 0)) return op_fail(SMI_ERR_INVALID, "mass must be > 0");
    if (n <= 0) return SMI_OK;
    const double one_over_mass = 1.0 / mass, dts2 = timestep / 2.;
    const double qmh = charge * one_over_mass * dts2;
    hipLaunchKernelGGL(k_boris, dim3(nblk(n, 256)), dim3(256), 0, (hipStream_t)stream, ndim, qmh, timestep, n, x, y,
                       z, px, py, pz, Epart, Bpart, invgf);
    OP_CHECK();
    return SMI_OK;
}

int smi_currents_3d(int order, double *Jx, double *Jy, double *Jz, const int np[3], const int dom_begin[3],
                    const double cell_length[3], double timestep, double charge, int64_t n, const double *x,
                    const double *y, const double *z, const double *w, const int32_t *iold, const double *deltaold,
                    int deterministic, void *stream)
{
    if (order != 2 && order != 4) return op_fail(SMI_ERR_INVALID, "order must be 2 or 4");
    if (n <= 0) return SMI_OK;
    Proj3Args a;
    a.J[0] = Jx;
    a.J[1] = Jy;
    a.J[2] = Jz;
    for (int c = 0; c < 3; ++c)
        for (int d = 0; d < 3; ++d) a.dims[c][d] = np[d] + (c == d ? 1 : 0);
    for (int d = 0; d < 3; ++d) {
        a.dom.v[d] = dom_begin[d];
        a.dinv.v[d] = 1.0 / cell_length[d];
        a.cr_scale.v[d] = cell_length[d] / timestep;
    }
    double cell_volume = 1.0;
    for (int d = 0; d < 3; ++d) cell_volume *= cell_length[d];
    a.cw_scale = (1. / cell_volume) * charge;
    a.n = n;
    a.x[0] = x;
    a.x[1] = y;
    a.x[2] = z;
    a.w = w;
    a.iold = iold;
    a.dold = deltaold;
    hipStream_t st = (hipStream_t)stream;
    try {
        if (deterministic) {
            if (order == 2) hipLaunchKernelGGL(k_proj3d_ordered<2>, dim3(1), dim3(64), 0, st, a);
            else hipLaunchKernelGGL(k_proj3d_ordered<4>, dim3(1), dim3(64), 0, st, a);
        } else if (!launch_bins(order, a, st)) {
            if (order == 2) hipLaunchKernelGGL(k_proj3d_atomic<2>, dim3(nblk(n, 128)), dim3(128), 0, st, a);
            else hipLaunchKernelGGL(k_proj3d_atomic<4>, dim3(nblk(n, 128)), dim3(128), 0, st, a);
        }
    } catch (const std::exception &e) {
        return op_fail(SMI_ERR_HIP, e.what());
    }
    OP_CHECK();
    return SMI_OK;
}

int smi_currents_2d(int order, double *Jx, double *Jy, double *Jz, const int np[2], const int dom_begin[2],
                    const double cell_length[2], double timestep, double charge, int64_t n, const double *x,
                    const double *y, const double *pz, const double *w, const double *invgf, const int32_t *iold,
                    const double *deltaold, int deterministic, void *stream)
{
    if (order != 2) return op_fail(SMI_ERR_INVALID, "2D projection order must be 2");
    if (n <= 0) return SMI_OK;
    Proj2Args a;
    a.J[0] = Jx;
    a.J[1] = Jy;
    a.J[2] = Jz;
    a.ny[0] = np[1];
    a.ny[1] = np[1] + 1;
    a.ny[2] = np[1];
    a.nx = np[0];
    a.dom = Ints3{{dom_begin[0], dom_begin[1], 0}};
    a.dinv = Dbl3{{1.0 / cell_length[0], 1.0 / cell_length[1], 1.0}};
    a.cr_scale = Dbl3{{cell_length[0] / timestep, cell_length[1] / timestep, 0.}};
    double cell_volume = 1.0;
    cell_volume *= cell_length[0];
    cell_volume *= cell_length[1];
    a.cw_scale = (1. / cell_volume) * charge;
    a.n = n;
    a.x = x;
    a.y = y;
    a.pz = pz;
    a.w = w;
    a.invgf = invgf;
    a.iold = iold;
    a.dold = deltaold;
    hipStream_t st = (hipStream_t)stream;
    if (deterministic) hipLaunchKernelGGL(k_proj2d_ordered, dim3(1), dim3(64), 0, st, a);
    else hipLaunchKernelGGL(k_proj2d_atomic, dim3(nblk(n, 128)), dim3(128), 0, st, a);
    OP_CHECK();
    return SMI_OK;
}

int smi_maxwell_ampere_3d(double *Ex, double *Ey, double *Ez, const double *Bx, const double *By, const double *Bz,
                          const double *Jx, const double *Jy, const double *Jz, const int np[3], double timestep,
                          const double cell_length[3], void *stream)
{
    Ints3 NP{{np[0], np[1], np[2]}};
    const int64_t tot = (int64_t)(np[0] + 1) * np[1] * np[2] + (int64_t)np[0] * (np[1] + 1) * np[2] +
                        (int64_t)np[0] * np[1] * (np[2] + 1);
    hipLaunchKernelGGL(k_ma3d_patch, dim3(nblk(tot, 256)), dim3(256), 0, (hipStream_t)stream, Ex, Ey, Ez, Bx, By, Bz,
                       Jx, Jy, Jz, NP, timestep, timestep / cell_length[0], timestep / cell_length[1],
                       timestep / cell_length[2]);
    OP_CHECK();
    return SMI_OK;
}

int smi_maxwell_faraday_3d(double *Bx, double *By, double *Bz, const double *Ex, const double *Ey, const double *Ez,
                           const int np[3], double timestep, const double cell_length[3], void *stream)
{
    Ints3 NP{{np[0], np[1], np[2]}};
    const int64_t tot = (int64_t)np[0] * (np[1] + 1) * (np[2] + 1) + (int64_t)(np[0] + 1) * np[1] * (np[2] + 1) +
                        (int64_t)(np[0] + 1) * (np[1] + 1) * np[2];
    hipLaunchKernelGGL(k_mf3d_patch, dim3(nblk(tot, 256)), dim3(256), 0, (hipStream_t)stream, Bx, By, Bz, Ex, Ey, Ez,
                       NP, timestep / cell_length[0], timestep / cell_length[1], timestep / cell_length[2]);
    OP_CHECK();
    return SMI_OK;
}

}  // extern "C"
