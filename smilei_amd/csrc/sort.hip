// sort.hip -- per-step cell sort and inter-patch exchange of particles.
//
// Replaces the reference's leaving-particle extraction, neighbour exchange
// and per-patch sort (Particles::copyLeavingParticlesToBuffers
// Particles.cpp:1308, Patch::exchParticles/cornersParticles Patch.cpp:
// 670-801, nvidiaParticles::sortParticleByKey nvidiaParticles.cu:1217-1247)
// with one device-wide counting sort by destination cell, since the push
// kernel already computed every particle's destination patch and cell:
//   1. histogram of destination cells          (int32 atomics)
//   2. exclusive scan -> cell_off               (block scan in one to three launches)
//   3. scatter of slot indices into buckets     (atomic count-down, which
//      also returns the histogram to zero for the next step)
//   4. per-bucket rank sort by (direction of motion, source slot), the
//      canonical order of particles inside a cell.
// The particle data itself is not moved here: the next step's particle
// kernel reads its input through `perm`.
#include <algorithm>

#include "kernels.h"
#include "pic_device.h"

namespace smi {

namespace {

constexpr uint32_t kKeyMask = (1u << 27) - 1;

// One species of a sort launch; the species of a step share their launches
// (blockIdx.y): small simulations are bound by the number of launches.
struct SortOne {
    const uint32_t *keys;
    int64_t n;
    const int32_t *tie;   // or null
    int32_t *counts, *cell_off, *first, *perm, *tmp, *big, *nbig, *bsum, *clus_old;
    uint8_t *stay;        // or null
};
struct SortSet {
    SortOne s[kMaxMerged];
};

__global__ void k_hist(const uint32_t *__restrict__ keys, int64_t n, int32_t *__restrict__ counts)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t key = i < n ? keys[i] & kKeyMask : ~0u;
    int head, len;
    dev::key_run(key, head, len);
    if ((int)(threadIdx.x & 63) == head && i < n) atomicAdd(&counts[key], len);
}

constexpr int kScanThreads = 256;
constexpr int kScanItems = 16;
constexpr int kScanTile = kScanThreads * kScanItems;

// Block-wide exclusive scan of one int per thread; returns the block total.
__device__ inline int block_exclusive_scan(int v, int &total)
{
    __shared__ int warp_tot[kScanThreads / 64];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    int incl = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(incl, o, 64);
        if (lane >= o) incl += t;
    }
    if (lane == 63) warp_tot[wid] = incl;
    __syncthreads();
    int base = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < kScanThreads / 64; ++w) {
        if (w < wid) base += warp_tot[w];
        tot += warp_tot[w];
    }
    __syncthreads();
    total = tot;
    return base + incl - v;
}

__global__ void __launch_bounds__(kScanThreads) k_scan_reduce(SortSet set, int64_t n)
{
    const int32_t *__restrict__ in = set.s[blockIdx.y].counts;
    int32_t *__restrict__ bsum = set.s[blockIdx.y].bsum;
    const int64_t base = (int64_t)blockIdx.x * kScanTile;
    int s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const int64_t i = base + (int64_t)k * kScanThreads + threadIdx.x;
        if (i < n) s += in[i];
    }
    int tot;
    block_exclusive_scan(s, tot);
    if (threadIdx.x == 0) bsum[blockIdx.x] = tot;
}

// Single-block exclusive scan of the block sums (in place).
__global__ void __launch_bounds__(kScanThreads) k_scan_bsum(SortSet set, int64_t nb)
{
    int32_t *__restrict__ bsum = set.s[blockIdx.y].bsum;
    int carry = 0;
    for (int64_t b0 = 0; b0 < nb; b0 += kScanTile) {
        int v[kScanItems];
        int s = 0;
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) {
            const int64_t i = b0 + (int64_t)threadIdx.x * kScanItems + k;
            v[k] = i < nb ? bsum[i] : 0;
            s += v[k];
        }
        int tot;
        int ex = block_exclusive_scan(s, tot) + carry;
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) {
            const int64_t i = b0 + (int64_t)threadIdx.x * kScanItems + k;
            if (i < nb) bsum[i] = ex;
            ex += v[k];
        }
        carry += tot;
    }
}

// Where a block of k_scan_apply takes the sum of the tiles before its own
// from: kPrefScanned, bsum scanned by k_scan_bsum; kPrefSums, the tile sums
// of k_scan_reduce, added up by the block; kPrefCounts, the counts
// themselves.  A block adds up to 2,048 sums (kPrefSums) or 32,768 counts
// (kPrefCounts, eight L2 reads in flight per thread) in less time than the
// launches it replaces take: the scan of 32^3 cells and two species takes
// 10.6 us in one launch, 32.5 us in three per species.
constexpr int kPrefScanned = 0, kPrefSums = 1, kPrefCounts = 2;
constexpr int64_t kMaxPrefSums = 2048, kMaxPrefCounts = 8;  // tiles

// out[i] = sum of the tiles before + exclusive prefix inside the block;
// out[n] = total.  Each thread owns 16 consecutive entries, moved as four
// 16-byte vectors (the entries of a full tile are 64-byte aligned); the
// ragged last tile takes the scalar path.  stay (placed stayers, or null):
// in[i] -= stay[i] after the totals are read, leaving the count of the
// bucket's atomic places, and stay[i] = 0 (not with kPrefCounts: other blocks
// still read in).  clus_old (or null): the previous out[] of every cpcell-th
// entry (each cluster's first slot before this sort) is saved there before it
// is overwritten.  Block 0 clears the work list of crowded cells.
__global__ void __launch_bounds__(kScanThreads) k_scan_apply(SortSet set, int64_t n, int pref, int cpcell)
{
    const SortOne &S = set.s[blockIdx.y];
    int32_t *__restrict__ in = S.counts;
    int32_t *__restrict__ out = S.cell_off;
    const int32_t *__restrict__ bsum = S.bsum;
    uint8_t *__restrict__ stay = S.stay;
    int32_t *__restrict__ clus_old = S.clus_old;
    if (S.nbig && blockIdx.x == 0 && threadIdx.x < 3) S.nbig[threadIdx.x] = 0;
    int before = 0;
    if (pref == kPrefScanned) {
        before = bsum[blockIdx.x];
    } else {
        int s = 0;
        if (pref == kPrefSums) {
            for (int i = threadIdx.x; i < (int)blockIdx.x; i += kScanThreads) s += bsum[i];
        } else {
            const int4 *src = reinterpret_cast<const int4 *>(in);
            const int m = blockIdx.x * (kScanTile / 4);
#pragma unroll 8
            for (int i = threadIdx.x; i < m; i += kScanThreads) {
                const int4 t = src[i];
                s += (t.x + t.y) + (t.z + t.w);
            }
        }
        block_exclusive_scan(s, before);
    }
    const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
    const bool full = (int64_t)(blockIdx.x + 1) * kScanTile <= n;
    // (a cluster is 16 or 64 cells: it begins at the first of a thread's
    // entries if at any)
    if (clus_old && base < n && (base & (cpcell - 1)) == 0) clus_old[base >> __builtin_ctz(cpcell)] = out[base];
    int v[kScanItems];
    int s = 0;
    if (full) {
        const int4 *src = reinterpret_cast<const int4 *>(in + base);
#pragma unroll
        for (int q = 0; q < kScanItems / 4; ++q) {
            const int4 t = src[q];
            v[4 * q] = t.x;
            v[4 * q + 1] = t.y;
            v[4 * q + 2] = t.z;
            v[4 * q + 3] = t.w;
        }
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) v[k] = base + k < n ? in[base + k] : 0;
    }
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) s += v[k];
    int tot;
    int ex = block_exclusive_scan(s, tot) + before;
    int o[kScanItems];
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        o[k] = ex;
        ex += v[k];
    }
    if (full) {
        int4 *dst = reinterpret_cast<int4 *>(out + base);
#pragma unroll
        for (int q = 0; q < kScanItems / 4; ++q) dst[q] = make_int4(o[4 * q], o[4 * q + 1], o[4 * q + 2], o[4 * q + 3]);
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; ++k)
            if (base + k < n) out[base + k] = o[k];
    }
    // the grand total after the last entry
#pragma unroll
    for (int k = 0; k < kScanItems; ++k)
        if (base + k == n - 1) out[n] = o[k] + v[k];
    if (!stay) return;
    if (full) {
        uint4 *sp = reinterpret_cast<uint4 *>(stay + base);
        const uint4 t = *sp;
        const uint32_t wd[4] = {t.x, t.y, t.z, t.w};
        if (wd[0] | wd[1] | wd[2] | wd[3]) {
            int4 *dst = reinterpret_cast<int4 *>(in + base);
#pragma unroll
            for (int q = 0; q < kScanItems / 4; ++q)
                dst[q] = make_int4(v[4 * q] - (int)(wd[q] & 255u), v[4 * q + 1] - (int)((wd[q] >> 8) & 255u),
                                   v[4 * q + 2] - (int)((wd[q] >> 16) & 255u), v[4 * q + 3] - (int)(wd[q] >> 24));
            *sp = make_uint4(0u, 0u, 0u, 0u);
        }
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; ++k)
            if (base + k < n && stay[base + k]) {
                in[base + k] = v[k] - stay[base + k];
                stay[base + k] = 0;
            }
    }
}

// Scatter of slot indices into their cell buckets.  Consecutive slots mostly
// keep their cell, so lanes of a wavefront with equal keys form runs: the
// run head takes `run` places with one atomic and the lanes fill them in
// slot order.  The count-down returns the histogram to zero.  With the
// count c before a run's atomic, the run takes places [end - c, end - c +
// run) of its bucket [start, end): successive runs fill the top counts[g]
// places, the whole bucket without placed stayers.  placed: a key whose top
// bits hold a rank r < kPlaceAtomic goes to start + r with no atomic (its
// cluster's stayers, SortBufs::stay).  cpc > 0 (the cells per cluster): the
// cell-major place is stored at its lane-interleaved slot of the cluster
// (cluster_slot).  The slots are dealt to the workgroups in the XCD-aware
// order (xcd_cluster): consecutive slots, and so the writes into one
// cluster's range of perm, meet in one L2, where the partial lines merge
// before they are written back.  Each wavefront takes kScatItems groups of
// 64 consecutive slots and issues the loads, atomics and stores of the
// groups together: the kernel is bound by the latency of its dependent
// accesses (key, count-down, bucket offsets, store), not by bytes.  Six
// groups per wavefront measured best on the 1.08e9-particle beam-plasma
// (sort 5.13 ms per step; four groups 5.40, five 5.26, seven 5.16, eight
// 5.62).
constexpr int kScatThreads = 256, kScatItems = 6, kScatTile = kScatThreads * kScatItems;

__global__ void __launch_bounds__(kScatThreads) k_scatter(SortSet set, int cpc, int lay, int placed)
{
    const SortOne &S = set.s[blockIdx.y];
    const uint32_t *__restrict__ keys = S.keys;
    const int64_t n = S.n;
    const int32_t *__restrict__ cell_off = S.cell_off;
    int32_t *__restrict__ counts = S.counts;
    int32_t *__restrict__ perm = S.first;
    const int blocks = (int)((n + kScatTile - 1) / kScatTile);  // of this species; the grid is the largest's
    if ((int)blockIdx.x >= blocks) return;
    const int lane = threadIdx.x & 63;
    const int64_t i0 = (int64_t)dev::xcd_cluster(blockIdx.x, blocks) * kScatTile +
                       (int64_t)(threadIdx.x >> 6) * (64 * kScatItems) + lane;
    uint32_t kk[kScatItems];
#pragma unroll
    for (int j = 0; j < kScatItems; ++j) kk[j] = i0 + 64 * j < n ? keys[i0 + 64 * j] : 0u;
    int c[kScatItems], my_head[kScatItems];
#pragma unroll
    for (int j = 0; j < kScatItems; ++j) {
        const bool direct = placed && (kk[j] >> 27) < kPlaceAtomic;
        // lanes of the count-down; the others carry the sentinel
        const uint32_t g = i0 + 64 * j < n && !direct ? kk[j] & kKeyMask : 0xFFFFFFFFu;
        const uint32_t gp = __shfl_up(g, 1, 64);
        const bool head = lane == 0 || gp != g;
        const uint64_t heads = __ballot(head);
        const uint64_t above = lane == 63 ? 0ull : heads & (~0ull << (lane + 1));
        const int next = above ? __ffsll((unsigned long long)above) - 1 : 64;
        my_head[j] = 63 - __clzll((unsigned long long)(heads & (lane == 63 ? ~0ull : ((2ull << lane) - 1))));
        c[j] = 0;
        if (head && g != 0xFFFFFFFFu) c[j] = atomicSub(&counts[g], next - lane);
    }
#pragma unroll
    for (int j = 0; j < kScatItems; ++j) {
        const int ch = __shfl(c[j], my_head[j], 64);
        const int64_t i = i0 + 64 * j;
        if (i >= n) continue;
        const uint32_t tag = kk[j] >> 27;
        const bool direct = placed && tag < kPlaceAtomic;
        const uint32_t gc = kk[j] & kKeyMask;
        const int pos = direct ? cell_off[gc] + (int)tag : cell_off[gc + 1] - ch + (lane - my_head[j]);
        if (cpc) {
            const uint32_t cb = gc & ~(uint32_t)(cpc - 1);
            const int s = cell_off[cb];
            perm[s + layout_slot(lay, pos - s, cell_off[cb + cpc] - s)] = (int32_t)i;
        } else {
            perm[pos] = (int32_t)i;
        }
    }
}

// Canonical order inside a cell: by direction of motion, then source slot.
// A wavefront takes 16 to 64 cells, whose particles are one run of places, and works
// on as many whole cells at a time as fit into kFixBatch places: one lane per
// place, kFixPer places per lane in flight.  The keys are staged in LDS, and a
// lane's rank is the number of smaller (direction, slot) pairs of its cell; the
// pairs are distinct because slots are.  What bounds it is the chain place ->
// slot -> key of loads from memory, hence the places in flight, eight
// wavefronts per SIMD (64 registers, one of them spilled; at seven 72 against
// 54 us) and the 18 KB of LDS.  Cells of more than `most` particles (fix_most) go
// to the work lists of k_bucket_fix_big: a wavefront with many of them would
// work on them for long after the rest of the chip is done (16^3 cells of 130
// particles in a grid of 64^3, two species: 1,055 us a sort with cells of up to
// 256 ranked here, 140 so; of 300, 960 and 285).  The stores of a batch follow
// the loads of all its places, so the in-place case (dst == src) is safe.
// 2D plasma, 2 x 2.6e5 cells of 16 particles: 54 us; 118 us with a thread per
// cell of up to 16 particles and half a wavefront per cell of up to 32.
// 3D, 2.6e5 cells of 8: 69 -> 29 us; 2 x 4.2e6 cells of 8: 453 -> 378 us.
// The cell-major input is src; cpc == 0: sorted in place (dst == src);
// cpc > 0: every particle is written to its lane-interleaved slot of the
// cluster in dst.  The tie-break value of source slot v is tie[v] when tie
// is given, else v.
constexpr int kFixMid = 64;
constexpr int kFixPer = 8;
constexpr int kFixBatch = 64 * kFixPer;  // at least kFixWave: a batch holds one cell at least
constexpr int kFixAhead = 4;             // keys read per step of the ranking

// Where the tie-breaks come from: tie[v] (the cell-major position of slot
// v in the previous sorted order, recorded by the particle kernel), or v
// itself when tie is null.  With clus_old (each cluster's first slot in
// the previous order, stored lane-interleaved), the tie of a slot inside
// the previous range of the cell's own cluster -- a particle that stayed
// in its cluster, nearly all of them -- is computed (cluster_rank) instead
// of gathered.  Such a particle did not leave its patch, so its direction of
// motion is 13 (no patch face crossed) and its key need not be read either,
// unless some axis is one cluster wide (a periodic wrap lands in the same
// cluster): stay13 = 0 then.
struct TieGeom {
    int cpcell, ncl;
    int lay;  // layout of the previous order's clusters
    int stay13;
};
struct TieSrc {
    const int32_t *tie;
    const int32_t *clus_old;
    int cpcell, ncl;
    int lay;  // layout of the previous order's clusters
    int64_t n;
    int stay13;
    __device__ TieSrc(const SortOne &S, const TieGeom &G)
        : tie(S.tie), clus_old(S.clus_old), cpcell(G.cpcell), ncl(G.ncl), lay(G.lay), n(S.n), stay13(G.stay13)
    {
    }
    // previous range [cs, cs + cn) of the cluster of cell g (cn = 0: none)
    __device__ void range(int64_t g, int &cs, int &cn) const
    {
        cs = 0;
        cn = 0;
        if (!tie || !clus_old) return;
        const int b = (int)g >> __builtin_ctz(cpcell);  // 16 or 64 cells; fewer than 2^27 in all
        cs = clus_old[b];
        cn = (b + 1 < ncl ? clus_old[b + 1] : (int)n) - cs;
    }
};

__device__ inline uint64_t fix_key(const uint32_t *keys, const TieSrc &T, int32_t v, int cs, int cn)
{
    uint32_t t = (uint32_t)v;
    if (T.tie) {
        const int r = v - cs;
        if (r >= 0 && r < cn) {
            t = (uint32_t)(cs + layout_rank(T.lay, r, cn));
            if (T.stay13) return (13ull << 32) | t;
        } else {
            t = (uint32_t)T.tie[v];
        }
    }
    return ((uint64_t)(keys[v] >> 27) << 32) | t;
}

// Wave-aggregated append of the lanes with `want` to a counter: returns
// each such lane's index (one atomic per wavefront).
__device__ inline int wave_append(bool want, int32_t *counter)
{
    const uint64_t m = __ballot(want);
    if (!m) return 0;
    const int lane = threadIdx.x & 63;
    const int leader = __ffsll((unsigned long long)m) - 1;
    int base = 0;
    if (lane == leader) base = atomicAdd(counter, __popcll(m));
    base = __shfl(base, leader, 64);
    return base + __popcll(m & ((1ull << lane) - 1));
}

// The lists of crowded cells: more than kFixWave particles in S.big (at most n /
// 257 cells), up to kFixWave behind them (at most n / 65).
constexpr int kFixWave = 256;
static_assert(kFixBatch >= kFixWave, "a batch holds whole cells");
__device__ inline int32_t *mid_list(const SortOne &S) { return S.big + S.n / (kFixWave + 1) + 1; }

// Orders a wavefront's accesses to LDS that only it uses.
__device__ inline void lds_order()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Cells per wavefront for so many cells of all species: 64 where that still
// gives the chip the 8,192 wavefronts it holds, else 32 or 16.  Measured for
// 64 / 32 / 16 / 8 cells: 5.2e5 cells 63 / 65 / 67 / 78 us, 2.6e5 cells 42 / 32 /
// 33 / 38 us, 6.6e4 cells 22 / 14 / 10 / 11 us.
constexpr int64_t kFixWaves = 8192;

inline int fix_cells(int64_t cells)
{
    return cells >= 64 * kFixWaves ? 64 : cells >= 32 * kFixWaves ? 32 : 16;
}

// Largest cell that a wavefront of k_bucket_fix ranks (its `most`): 64, or where
// the mean cell is crowded itself twice the mean, as long as there are enough
// wavefronts for all cells to be ranked at once.  Uniform plasmas of 2 species, cells
// ranked there / listed, us: 8,192 wavefronts (64^3 cells), 64 particles per
// cell 980 / 1,249, 128 2,607 / 3,065, 200 5,119 / 4,698; 4,096 (32^3) 80 221 / 251,
// 100 301 / 289; 2,048 (128^2) 64 114 / 131, 80 150 / 126; 512 (16^3) 56 87 / 89, 64
// 106 / 94: the line lies at 48 particles and one more per 75 wavefronts.
inline int fix_most(int64_t n, int64_t ncells, int64_t waves)
{
    const int64_t mean = n / ncells;
    return (int)std::min<int64_t>(mean > 48 + waves / 75 ? kFixMid : std::max<int64_t>(2 * mean, kFixMid), kFixWave);
}

__global__ void __launch_bounds__(256, 8) k_bucket_fix(SortSet set, int64_t ncells, int wcells, int most, int cpc, int lay, TieGeom G)
{
    const SortOne &S = set.s[blockIdx.y];
    const uint32_t *__restrict__ keys = S.keys;
    const int32_t *__restrict__ cell_off = S.cell_off;
    int32_t *src = S.first, *dst = S.perm;
    const TieSrc T(S, G);
    __shared__ uint64_t sKey[4][kFixBatch + kFixAhead];
    __shared__ __align__(8) uint8_t sHead[4][kFixBatch];
    uint64_t *const sk = sKey[threadIdx.x >> 6];
    uint8_t *const sh = sHead[threadIdx.x >> 6];  // 1 + the lane whose cell begins at a place, else 0
    const int lane = threadIdx.x & 63;
    const int64_t g = ((int64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * wcells + lane;
    const bool mine = lane < wcells && g < ncells;
    const int a = mine ? cell_off[g] : 0;
    const int n = mine ? cell_off[g + 1] - a : 0;
    // range of the lane's cluster, now and before
    int cs = 0, cn = 0, ocs = 0, ocn = 0;
    if (n > 0) {
        if (cpc) {
            const int64_t cb = g & ~(int64_t)(cpc - 1);
            cs = cell_off[cb];
            cn = cell_off[cb + cpc] - cs;
        }
        T.range(g, ocs, ocn);
    }
    if (__ballot(n > most)) {
        const int iw = wave_append(n > most && n <= kFixWave, &S.nbig[2]);
        if (n > most && n <= kFixWave) mid_list(S)[iw] = (int32_t)g;
        const int ib = wave_append(n > kFixWave, &S.nbig[0]);
        if (n > kFixWave) S.big[ib] = (int32_t)g;
    }
    // places of the lane's cell in the wavefront's run (in place, a single
    // particle is where it belongs), and where they begin
    const int m = n > most || (n == 1 && !cpc) ? 0 : n;
    int end = m;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int e = __shfl_up(end, d, 64);
        if (lane >= d) end += e;
    }
    const int begin = end - m, total = __builtin_amdgcn_readlane(end, 63);
    for (int base = 0; base < total;) {
        // the cells that begin at base or later and end within the batch
        const int len = __builtin_amdgcn_readlane(end, 63 - __builtin_clzll(__ballot(end - base <= kFixBatch))) - base;
        static_assert(kFixBatch == 64 * 8, "a lane clears eight places");
        *reinterpret_cast<uint64_t *>(sh + 8 * lane) = 0;
        lds_order();
        if (m > 0 && begin >= base && end - base <= len) sh[begin - base] = (uint8_t)(lane + 1);
        lds_order();
        int32_t v[kFixPer];
        int c[kFixPer];  // the lane that holds the place's cell
        int last = 0;    // ... of the place before
#pragma unroll
        for (int q = 0; q < kFixPer; ++q) {
            v[q] = 0;
            c[q] = 0;
            if (64 * q >= len) continue;
            const int t = base + 64 * q + lane;
            const int head = sh[64 * q + lane];
            const uint64_t before = __ballot(head != 0) & (~0ull >> (63 - lane));
            const int at = __shfl(head - 1, before ? 63 - __builtin_clzll(before) : lane, 64);
            c[q] = before ? at : last;
            last = __builtin_amdgcn_readlane(c[q], 63);
            const int ac = __shfl(a - begin, c[q], 64);
            if (t - base < len) v[q] = src[ac + t];
        }
#pragma unroll
        for (int q = 0; q < kFixPer; ++q) {
            if (64 * q >= len) continue;
            const int oc = __shfl(ocs, c[q], 64), on = __shfl(ocn, c[q], 64);
            if (64 * q + lane < len) sk[64 * q + lane] = fix_key(keys, T, v[q], oc, on);
        }
        lds_order();
#pragma unroll
        for (int q = 0; q < kFixPer; ++q) {
            if (64 * q >= len) continue;
            const int s = __shfl(begin, c[q], 64) - base, mc = __shfl(m, c[q], 64), ac = __shfl(a, c[q], 64);
            const int ccs = __shfl(cs, c[q], 64), ccn = __shfl(cn, c[q], 64);
            if (64 * q + lane < len) {
                const uint64_t k = sk[64 * q + lane];
                int r = ac;
                for (int j = 0; j < mc; j += kFixAhead)
#pragma unroll
                    for (int i = 0; i < kFixAhead; ++i) r += j + i < mc && sk[s + j + i] < k ? 1 : 0;
                dst[cpc ? ccs + layout_slot(lay, r - ccs, ccn) : r] = v[q];
            }
        }
        lds_order();
        base += len;
    }
}

// The cells of the work lists.  Up to kFixWave particles (nbig[2] cells): a
// wavefront each, four places a lane, a place's rank counted over the cell's keys
// in LDS, which all lanes read at the same time.  More (nbig[0] cells, nbig[1] =
// 0 on entry): one workgroup per cell pulled from the list until it is
// exhausted.  Up to kBigLds particles: bitonic sort of the (key, slot) pairs in
// LDS.  More: each particle's rank = the number of smaller keys, counted over the
// cell in LDS-staged chunks, kBigLds target particles at a time (in place, cpc ==
// 0, the cell is first copied to scr so that no write can overtake a read).
// Every workgroup exits once the lists are exhausted.
constexpr int kBigThreads = 256;
constexpr int kBigLds = 4096;
constexpr int kBigPer = kBigLds / kBigThreads;
constexpr int kBigBlocks = 1024;

// Workgroups for the crowded cells of n particles, of which there are usually
// none: a workgroup that finds the lists empty ends at its first load
// (1,024 of them cost no more than 192 that each asked the list for work: 4.2e6
// particles 84.3 / 83.8 us a sort).
inline unsigned big_blocks(int64_t n)
{
    const int64_t b = (n + 2047) / 2048;
    return (unsigned)(b < kBigBlocks ? b : kBigBlocks);
}

// Order of the cell of n <= 64 * PER particles from place a on, by one wavefront;
// put(place, slot) stores; sk: 64 * PER keys of LDS.
template <int PER, class Key, class Put>
__device__ inline void rank_by_wave(const int32_t *src, int a, int n, uint64_t *sk, Key key, Put put)
{
    const int lane = threadIdx.x & 63;
    int32_t v[PER];
    uint64_t k[PER];
    int r[PER];
#pragma unroll
    for (int q = 0; q < PER; ++q) v[q] = 64 * q + lane < n ? src[a + 64 * q + lane] : 0;
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        k[q] = 64 * q + lane < n ? key(v[q]) : ~0ull;
        r[q] = 0;
        sk[64 * q + lane] = k[q];
    }
    lds_order();
    for (int j = 0; j < n; j += 2) {  // (an entry after the last is the largest key)
        const uint64_t k0 = sk[j], k1 = sk[j + 1];
#pragma unroll
        for (int q = 0; q < PER; ++q) r[q] += (k0 < k[q] ? 1 : 0) + (k1 < k[q] ? 1 : 0);
    }
    lds_order();
#pragma unroll
    for (int q = 0; q < PER; ++q)
        if (64 * q + lane < n) put(a + r[q], v[q]);
}

__global__ void __launch_bounds__(kBigThreads) k_bucket_fix_big(SortSet set, int cpc, int lay, TieGeom G)
{
    const SortOne &S = set.s[blockIdx.y];
    const uint32_t *__restrict__ keys = S.keys;
    const int32_t *__restrict__ cell_off = S.cell_off;
    int32_t *src = S.first, *dst = S.perm, *scr = S.tmp;
    const TieSrc T(S, G);
    const int32_t *__restrict__ big = S.big;
    int32_t *__restrict__ nbig = S.nbig;
    __shared__ uint64_t sK[kBigLds];
    __shared__ int32_t sV[kBigLds];
    __shared__ int sItem;
    const int nb = nbig[0], nm = nbig[2];
    if ((nb | nm) == 0) return;
    const int tid = threadIdx.x;
    const int32_t *mid = mid_list(S);
    for (int item = blockIdx.x * (kBigThreads / 64) + (tid >> 6); item < nm; item += gridDim.x * (kBigThreads / 64)) {
        const int g = mid[item], a = cell_off[g];
        int cs = 0, cn = 0, ocs, ocn;
        if (cpc) {
            const int cb = g & ~(cpc - 1);
            cs = cell_off[cb];
            cn = cell_off[cb + cpc] - cs;
        }
        T.range(g, ocs, ocn);
        const int n = cell_off[g + 1] - a;
        uint64_t *sk = sK + (tid >> 6) * kFixWave;
        auto key = [&](int32_t v) { return fix_key(keys, T, v, ocs, ocn); };
        auto put = [&](int pos, int32_t v) { dst[cpc ? cs + layout_slot(lay, pos - cs, cn) : pos] = v; };
        if (n <= 128) rank_by_wave<2>(src, a, n, sk, key, put);
        else rank_by_wave<4>(src, a, n, sk, key, put);
    }
    if (nb == 0) return;
    for (;;) {
        __syncthreads();  // the previous cell is done with the LDS arrays
        if (tid == 0) sItem = atomicAdd(&nbig[1], 1);
        __syncthreads();
        const int item = sItem;
        if (item >= nb) break;
        const int64_t g = big[item];
        const int a = cell_off[g], n = cell_off[g + 1] - a;
        int cs = 0, cn = 0;
        if (cpc) {
            const int64_t cb = g & ~(int64_t)(cpc - 1);
            cs = cell_off[cb];
            cn = cell_off[cb + cpc] - cs;
        }
        auto put = [&](int pos, int32_t v) { dst[cpc ? cs + layout_slot(lay, pos - cs, cn) : pos] = v; };
        int ocs, ocn;
        T.range(g, ocs, ocn);
        if (n <= kBigLds) {
            int P = 1;
            while (P < n) P <<= 1;
            for (int i = tid; i < P; i += kBigThreads) {
                const int32_t v = i < n ? src[a + i] : 0;
                sK[i] = i < n ? fix_key(keys, T, v, ocs, ocn) : ~0ull;
                sV[i] = v;
            }
            __syncthreads();
            for (int k = 2; k <= P; k <<= 1)
                for (int j = k >> 1; j > 0; j >>= 1) {
                    for (int i = tid; i < P; i += kBigThreads) {
                        const int l = i ^ j;
                        if (l > i && ((sK[i] > sK[l]) == ((i & k) == 0))) {
                            const uint64_t tk = sK[i];
                            sK[i] = sK[l];
                            sK[l] = tk;
                            const int32_t tv = sV[i];
                            sV[i] = sV[l];
                            sV[l] = tv;
                        }
                    }
                    __syncthreads();
                }
            for (int i = tid; i < n; i += kBigThreads) put(a + i, sV[i]);
            continue;
        }
        const int32_t *rd = src;
        if (!cpc) {
            for (int i = tid; i < n; i += kBigThreads) scr[a + i] = src[a + i];
            __threadfence_block();
            __syncthreads();
            rd = scr;
        }
        for (int t0 = 0; t0 < n; t0 += kBigLds) {
            uint64_t mk[kBigPer];
            int32_t mv[kBigPer];
            int rk[kBigPer];
#pragma unroll
            for (int m = 0; m < kBigPer; ++m) {
                const int i = t0 + tid + m * kBigThreads;
                mv[m] = i < n ? rd[a + i] : 0;
                mk[m] = i < n ? fix_key(keys, T, mv[m], ocs, ocn) : ~0ull;
                rk[m] = 0;
            }
            for (int c0 = 0; c0 < n; c0 += kBigLds) {
                const int cnum = n - c0 < kBigLds ? n - c0 : kBigLds;
                __syncthreads();
                for (int i = tid; i < cnum; i += kBigThreads) sK[i] = fix_key(keys, T, rd[a + c0 + i], ocs, ocn);
                __syncthreads();
                for (int j = 0; j < cnum; ++j) {
                    const uint64_t kj = sK[j];
#pragma unroll
                    for (int m = 0; m < kBigPer; ++m) rk[m] += kj < mk[m] ? 1 : 0;
                }
            }
#pragma unroll
            for (int m = 0; m < kBigPer; ++m)
                if (t0 + tid + m * kBigThreads < n) put(a + rk[m], mv[m]);
        }
    }
}

__global__ void k_occupied(const int32_t *__restrict__ cell_off, int ncl, int cpc, int *__restrict__ out)
{
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t m = __ballot(b < ncl && cell_off[(int64_t)b * cpc] != cell_off[(int64_t)(b + 1) * cpc]);
    if ((threadIdx.x & 63) == 0 && m) atomicAdd(out, __popcll(m));
}

// Slot j of the current order, stored with cluster layout `from`, moved to
// its slot under layout `to` (layout_slot); the cluster of the particle
// comes from its key, cpc = cells per cluster.
__global__ void k_relayout(const uint32_t *__restrict__ keys, int64_t n, const int32_t *__restrict__ cell_off,
                           const int32_t *__restrict__ src, int32_t *__restrict__ dst, int cpc, int from, int to)
{
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const int32_t v = src[j];
    const uint32_t cb = (keys[v] & kKeyMask) & ~(uint32_t)(cpc - 1);
    const int s = cell_off[cb], m = cell_off[cb + cpc] - s;
    const int p = layout_rank(from, (int)(j - s), m);
    dst[s + layout_slot(to, p, m)] = v;
}

// Patch and cell key of loaded particles; all get direction 13 ("stay") so
// that the canonical order of a cell is the input order.
template <int ND>
__global__ void k_bin_initial(Geom g, PartPtrs A, int64_t n, uint32_t *__restrict__ keys)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double x[3] = {A.x[i], A.y[i], ND == 3 ? A.z[i] : 0.};
    keys[i] = (13u << 27) | dev::position_key<ND>(g, x);
}

inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

}  // namespace

int64_t sort_bsum_size(int64_t ncells) { return (ncells + kScanTile - 1) / kScanTile + 1; }

void launch_sort(const Geom &g, const SortTask *tasks, int ns, hipStream_t st, bool counted, bool in_cell_order,
                 int layout, bool placed)
{
    if (ns < 1 || ns > kMaxMerged) throw Error(-1, "bad species count of a sort launch");
    placed = placed && counted && !in_cell_order;
    const int64_t nc = g.ncells;
    // the in-cell pass of the step's sort computes the ties of the particles
    // that stayed in their cluster from the clusters' previous ranges
    int stay13 = 1;
    for (int d = 0; d < g.nd; ++d)
        if (g.npatch[d] * g.n[d] <= 4) stay13 = 0;
    const TieGeom G{g.cells_per_cl, (int)(nc / g.cells_per_cl), layout, stay13};
    // cell-major places go straight to perm unless the canonical order inside
    // the cells and the interleaved layout are both asked for: then they are
    // ordered in tmp and laid out into perm
    const int cpc = layout ? g.cells_per_cl : 0;
    SortSet set{};
    int64_t most = 0;
    for (int q = 0; q < ns; ++q) {
        const SortTask &t = tasks[q];
        const SortBufs &sb = *t.sb;
        SortOne &S = set.s[q];
        S.keys = t.keys;
        S.n = t.n;
        S.tie = t.tie;
        S.counts = sb.counts;
        S.cell_off = sb.cell_off;
        S.first = in_cell_order && layout ? sb.tmp : sb.perm;
        S.perm = sb.perm;
        S.tmp = sb.tmp;
        S.big = sb.big;
        S.nbig = in_cell_order ? sb.nbig : nullptr;
        S.bsum = sb.bsum;
        S.clus_old = counted && t.tie && in_cell_order ? sb.clus_old : nullptr;
        S.stay = placed ? sb.stay : nullptr;
        most = t.n > most ? t.n : most;
        if (in_cell_order && !sb.big) throw Error(-1, "a sort in cell order needs its work lists");
        if (t.n > 0 && !counted) {
            hipLaunchKernelGGL(k_hist, dim3(nblk(t.n, 256)), dim3(256), 0, st, t.keys, t.n, sb.counts);
            SMI_LAUNCH_CHECK();
        }
    }
    const int64_t nb = (nc + kScanTile - 1) / kScanTile;
    const int pref = nb <= kMaxPrefCounts && !placed ? kPrefCounts : (nb <= kMaxPrefSums ? kPrefSums : kPrefScanned);
    const dim3 tiles((unsigned)nb, ns);
    if (pref != kPrefCounts) {
        hipLaunchKernelGGL(k_scan_reduce, tiles, dim3(kScanThreads), 0, st, set, nc);
        SMI_LAUNCH_CHECK();
    }
    if (pref == kPrefScanned) {
        hipLaunchKernelGGL(k_scan_bsum, dim3(1, ns), dim3(kScanThreads), 0, st, set, nb);
        SMI_LAUNCH_CHECK();
    }
    hipLaunchKernelGGL(k_scan_apply, tiles, dim3(kScanThreads), 0, st, set, nc, pref, g.cells_per_cl);
    SMI_LAUNCH_CHECK();
    if (most == 0) return;
    hipLaunchKernelGGL(k_scatter, dim3(nblk(most, kScatTile), ns), dim3(kScatThreads), 0, st, set,
                       in_cell_order ? 0 : cpc, layout, placed ? 1 : 0);
    SMI_LAUNCH_CHECK();
    if (!in_cell_order) return;
    const int wc = fix_cells(nc * ns);
    const int rank = fix_most(most, nc, nc * ns / wc);
    hipLaunchKernelGGL(k_bucket_fix, dim3(nblk(nc, 4 * wc), ns), dim3(256), 0, st, set, nc, wc, rank, cpc, layout, G);
    SMI_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_bucket_fix_big, dim3(big_blocks(most), ns), dim3(kBigThreads), 0, st, set, cpc, layout, G);
    SMI_LAUNCH_CHECK();
}

void launch_sort(const Geom &g, const uint32_t *keys, int64_t n, SortBufs &sb, hipStream_t st, bool counted,
                 bool in_cell_order, int layout, const int32_t *tie, bool placed)
{
    const SortTask one{keys, n, &sb, tie};
    launch_sort(g, &one, 1, st, counted, in_cell_order, layout, placed);
}

void launch_occupied(const Geom &g, const int32_t *cell_off, int *out, hipStream_t st)
{
    const int ncl = (int)(g.ncells / g.cells_per_cl);
    launch_fill_i32(out, 1, 0, st);
    hipLaunchKernelGGL(k_occupied, dim3(nblk(ncl, 256)), dim3(256), 0, st, cell_off, ncl, g.cells_per_cl, out);
    SMI_LAUNCH_CHECK();
}

void launch_relayout(const Geom &g, const uint32_t *keys, int64_t n, SortBufs &sb, int from_layout,
                     int to_layout, hipStream_t st)
{
    if (n == 0 || from_layout == to_layout) return;
    hipLaunchKernelGGL(k_relayout, dim3(nblk(n, 256)), dim3(256), 0, st, keys, n, (const int32_t *)sb.cell_off,
                       (const int32_t *)sb.perm, sb.tmp, g.cells_per_cl, from_layout, to_layout);
    SMI_LAUNCH_CHECK();
    SMI_HIP(hipMemcpyAsync(sb.perm, sb.tmp, n * sizeof(int32_t), hipMemcpyDeviceToDevice, st));
}

void launch_bin_initial(const Geom &g, const PartPtrs &A, int64_t n, uint32_t *keys, hipStream_t st)
{
    if (n == 0) return;
    if (g.nd == 3) hipLaunchKernelGGL(k_bin_initial<3>, dim3(nblk(n, 256)), dim3(256), 0, st, g, A, n, keys);
    else hipLaunchKernelGGL(k_bin_initial<2>, dim3(nblk(n, 256)), dim3(256), 0, st, g, A, n, keys);
    SMI_LAUNCH_CHECK();
}

}  // namespace smi
