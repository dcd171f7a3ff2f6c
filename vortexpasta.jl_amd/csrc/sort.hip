// Deterministic binning of points and nodes by cell, spreading tile or slab.
//
// Replaces the reference's atomic linked-list cell build (CellLists/gpu.jl:28-61,
// whose intra-cell order depends on thread timing) and its target counting sort
// (CellLists/gpu.jl:183-219). One call bins up to two lists that run on one stream:
//
//   1. zero the histograms
//   2. key of every element and histogram, remembering each element's arrival rank: runs
//      of equal keys inside a wavefront (neighbours along a filament mostly share a bin)
//      take one atomic
//   3. sums of 2048-bin tiles, then an exclusive scan of each tile on top of the sums
//      before it
//   4. scatter to start[key] + rank
//   5. tiles and slabs: blocks for every large bin (bin_large; found by the scan) put it in order
//
// The order inside a bin is then that of the arrival ranks. The kernels that gather the
// binned data put an element at start + (number of smaller indices in its bin) (bin_place
// in device_util.hpp): order (key, original index), so sums taken in that order are
// reproducible run to run.
//
// Why this and not a radix sort: below a million elements the library's sort is a merge sort
// of 10 to 36 launches (256k nodes: 36 of 6 us, on both streams), and above it needs the keys
// sorted only to find the bins again. Why no sort of each bin's segment: one thread per bin
// took 160-450 us wherever a few bins hold most points. Five launches for both lists; points
// and nodes of 256k nodes, LR stream, 0.21 -> 0.11 ms; cell lists 0.20 -> 0.07 ms. The count of
// smaller indices is quadratic in a bin's population, while the walks over a tile or a slab that come
// after are linear: large tiles and slabs are put in order by step 5 instead. Sort and records on 384³
// cells, all points and nodes in one tile and slab: 100k 3.3 -> 0.15 ms, 1M 219 -> 0.93 ms (the radix sort
// 1.7 and 2.0); on lines along x in one slab: 1M 117 -> 2.3 ms (2.2).
#include "vpbs_internal.hpp"
#include "device_util.hpp"

#include <algorithm>

namespace vpbs {

namespace {

constexpr int SCAN_BS = 256;
constexpr int SCAN_IPT = 8;
constexpr int SCAN_TILE = SCAN_BS * SCAN_IPT;
// Tiles whose sums one block adds up by itself (16M bins); longer scans go by levels.
constexpr int64_t SCAN_FLAT_TILES = 8192;

inline unsigned nblocks(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

__device__ inline int wrap_cell(int i, int n) {
    i %= n;
    return i < 0 ? i + n : i;
}

// Key of element j of a list; cell lists also store the cell (ix, iy, iz, key).
__device__ inline int32_t bin_key(const BinGeom &g, const BinList &l, int64_t j) {
    const double *p = l.pos + j;
    if (l.kind == BIN_CELL) {
        int ix = cell_index(p[0], g.box.L[0], g.Nc[0]);
        int iy = cell_index(p[l.n], g.box.L[1], g.Nc[1]);
        int iz = cell_index(p[2 * l.n], g.box.L[2], g.Nc[2]);
        // Points folded into [0, L) always give indices in [0, N); clamp defensively.
        ix = min(max(ix, 0), g.Nc[0] - 1);
        iy = min(max(iy, 0), g.Nc[1] - 1);
        iz = min(max(iz, 0), g.Nc[2] - 1);
        const int k = (iz * g.Nc[1] + iy) * g.Nc[0] + ix;
        if (l.cell) reinterpret_cast<int4 *>(l.cell)[j] = make_int4(ix, iy, iz, k);
        return k;
    }
    // first stencil cell per direction, as the records store it
    int i0[3];
#pragma unroll
    for (int d = 0; d < 3; d++) i0[d] = wrap_cell((int)floor(p[d * l.n] * g.scale[d]) - g.M + 1, g.G[d]);
    if (l.kind == BIN_SLAB) return (i0[2] / g.hz) * (g.G[1] / SLAB_HY) + i0[1] / SLAB_HY;
    return ((i0[2] / SPREAD_TZ) * (g.G[1] / SPREAD_TY) + i0[1] / SPREAD_TY) * (g.G[0] / SPREAD_TX) + i0[0] / SPREAD_TX;
}

// The list of a block: lists' blocks follow each other.
__device__ inline int list_of(const BinGroup &g, const unsigned (&first)[2]) {
    return g.count > 1 && blockIdx.x >= first[1] ? 1 : 0;
}

__global__ __launch_bounds__(256) void bin_zero(BinGroup g) {
    const int t = list_of(g, g.scan_block);
    const BinList &l = g.l[t];
    if (g.large && blockIdx.x == 0 && threadIdx.x == 0) g.large[0] = 0;
    const int64_t base = (int64_t)(blockIdx.x - g.scan_block[t]) * SCAN_TILE + threadIdx.x;
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) {
        const int64_t b = base + k * SCAN_BS;
        if (b <= l.nbins) l.start[b] = 0;
    }
}

__global__ __launch_bounds__(256) void bin_histogram(BinGroup g) {
    const int t = list_of(g, g.elem_block);
    const BinList &l = g.l[t];
    const int64_t j = (int64_t)(blockIdx.x - g.elem_block[t]) * 256 + threadIdx.x;
    const int lane = threadIdx.x & 63;
    const int32_t key = j < l.n ? bin_key(g.geom, l, j) : -1;
    // runs of equal keys: the first lane of each adds the run's length
    const int32_t prev = __shfl_up(key, 1, 64);
    const unsigned long long heads = __ballot(lane == 0 || key != prev);
    int first = 63 - __clzll(heads & (~0ull >> (63 - lane)));
    const unsigned long long later = heads & ~(~0ull >> (63 - first));  // heads of later runs
    int count = (later ? __ffsll(later) - 1 : 64) - first, place = lane - first;
    // the runs of up to four keys together: elements in no order, few bins (a million atomics on one
    // counter take 3 ms)
    unsigned long long todo = heads;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        if (!todo) break;
        const int lead = __ffsll(todo) - 1;
        const unsigned long long same = __ballot(key == __builtin_amdgcn_readlane(key, lead));
        if (same >> lane & 1) {
            first = lead;
            count = __popcll(same);
            place = __popcll(same & ((1ull << lane) - 1ull));
        }
        todo &= ~same;
    }
    int base = 0;
    if (lane == first && key >= 0) base = atomicAdd(&l.start[key], count);
    base = __shfl(base, first, 64);
    if (j < l.n) {
        l.key[j] = key;
        l.rank[j] = base + place;
    }
}

__device__ inline int32_t block_sum(int32_t v, int32_t *s_tot) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int incl = wave_incl_scan(v);
    if (lane == 63) s_tot[wid] = incl;
    __syncthreads();
    int32_t s = 0;
#pragma unroll
    for (int w = 0; w < SCAN_BS / 64; w++) s += s_tot[w];
    return s;
}

__global__ __launch_bounds__(SCAN_BS) void bin_tile_sums(BinGroup g) {
    __shared__ int32_t s_tot[SCAN_BS / 64];
    const int t = list_of(g, g.scan_block);
    const BinList &l = g.l[t];
    const int64_t tile = blockIdx.x - g.scan_block[t];
    int32_t v = 0;
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) {
        const int64_t b = tile * SCAN_TILE + threadIdx.x + k * SCAN_BS;
        if (b <= l.nbins) v += l.start[b];
    }
    const int32_t s = block_sum(v, s_tot);
    if (threadIdx.x == 0) l.sums[tile] = s;
}

// Exclusive scan of one tile in place, on top of what comes before it: the sums of the tiles
// before it added up here, or (scanned) read from their exclusive scan. Large bins go to `large`.
__device__ inline void scan_tile(int32_t *a, int64_t n, int64_t tile, const int32_t *sums, bool scanned, int32_t *s_tot,
                                 int32_t *s_tot2, int32_t *large = nullptr, int list = 0, int64_t elements = 0) {
    int32_t before = 0;
    if (scanned) {
        before = sums[tile];
    } else {
        int32_t v = 0;
        for (int64_t k = threadIdx.x; k < tile; k += SCAN_BS) v += sums[k];
        before = block_sum(v, s_tot2);
    }
    const int64_t base = tile * SCAN_TILE + (int64_t)threadIdx.x * SCAN_IPT;
    int32_t v[SCAN_IPT], local = 0;
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) {
        v[k] = base + k < n ? a[base + k] : 0;
        local += v[k];
    }
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int incl = wave_incl_scan(local);
    if (lane == 63) s_tot[wid] = incl;
    __syncthreads();
    int32_t run = before + incl - local;
    for (int w = 0; w < wid; w++) run += s_tot[w];
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) {
        if (base + k < n) a[base + k] = run;
        run += v[k];
        if (large && bin_large(elements, v[k])) {
            const int e = atomicAdd(large, 1);
            large[1 + 2 * e] = list;
            large[2 + 2 * e] = (int32_t)(base + k);
        }
    }
}

__global__ __launch_bounds__(SCAN_BS) void bin_scan(BinGroup g, int scanned) {
    __shared__ int32_t s_tot[SCAN_BS / 64], s_tot2[SCAN_BS / 64];
    const int t = list_of(g, g.scan_block);
    const BinList &l = g.l[t];
    scan_tile(l.start, l.nbins + 1, blockIdx.x - g.scan_block[t], l.sums, scanned != 0, s_tot, s_tot2,
              l.order_large ? g.large : nullptr, t, l.n);
}

// Levels of a scan with more than SCAN_FLAT_TILES tiles.
__global__ __launch_bounds__(SCAN_BS) void level_sums(const int32_t *__restrict__ a, int64_t n,
                                                      int32_t *__restrict__ sums) {
    __shared__ int32_t s_tot[SCAN_BS / 64];
    int32_t v = 0;
#pragma unroll
    for (int k = 0; k < SCAN_IPT; k++) {
        const int64_t b = (int64_t)blockIdx.x * SCAN_TILE + threadIdx.x + k * SCAN_BS;
        if (b < n) v += a[b];
    }
    const int32_t s = block_sum(v, s_tot);
    if (threadIdx.x == 0) sums[blockIdx.x] = s;
}

__global__ __launch_bounds__(SCAN_BS) void level_scan(int32_t *__restrict__ a, int64_t n,
                                                      const int32_t *__restrict__ sums, int scanned) {
    __shared__ int32_t s_tot[SCAN_BS / 64], s_tot2[SCAN_BS / 64];
    scan_tile(a, n, blockIdx.x, sums, scanned != 0, s_tot, s_tot2);
}

// In-place exclusive scan of n tile sums; tmp follows them.
void scan_levels(int32_t *a, int64_t n, int32_t *tmp, hipStream_t s) {
    const int64_t nt = (n + SCAN_TILE - 1) / SCAN_TILE;
    level_sums<<<(unsigned)nt, SCAN_BS, 0, s>>>(a, n, tmp);
    const bool deep = nt > SCAN_FLAT_TILES;
    if (deep) scan_levels(tmp, nt, tmp + nt, s);
    level_scan<<<(unsigned)nt, SCAN_BS, 0, s>>>(a, n, tmp, deep);
}

__global__ __launch_bounds__(256) void bin_scatter(BinGroup g) {
    const int t = list_of(g, g.elem_block);
    const BinList &l = g.l[t];
    const int64_t j = (int64_t)(blockIdx.x - g.elem_block[t]) * 256 + threadIdx.x;
    if (j < l.n) l.perm[l.start[l.key[j]] + l.rank[j]] = (int32_t)j;
}

// Large bins: a block per bin and window of indices marks the bin's elements in the window as bits in LDS
// and writes the set bits, in order, behind the bin's smaller elements (into the ranks, which are done
// with). Bound by the latency of the loads; the blocks are small enough to start beside the other
// stream's kernels, since usually there is nothing to do (blocks of 1024 threads with 33 KB made a call of
// 1.14 ms 3 % slower).
constexpr int ORDER_NT = 256, ORDER_WORDS = 16 * ORDER_NT, ORDER_WINDOW = 32 * ORDER_WORDS;
constexpr int64_t ORDER_BLOCKS = 1024;
__global__ __launch_bounds__(ORDER_NT) void bin_order(BinGroup g, int windows) {
    __shared__ uint32_t bits[ORDER_WORDS];
    __shared__ int32_t s_tot[ORDER_NT / 64], s_before[ORDER_NT / 64];
    constexpr int PER = ORDER_WORDS / ORDER_NT;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int64_t items = (int64_t)g.large[0] * windows;
    for (int64_t item = blockIdx.x; item < items; item += gridDim.x) {
        const int e = (int)(item / windows);
        const int64_t first = (item - (int64_t)e * windows) * ORDER_WINDOW;
        const BinList &l = g.l[g.large[1 + 2 * e]];
        if (first >= l.n) continue;
        const int32_t bin = g.large[2 + 2 * e], s0 = l.start[bin], s1 = l.start[bin + 1];
        const int32_t v0 = (s0 + 3) & ~3, v1 = s1 & ~3;  // whole 16-byte vectors (population > BIN_LARGE: v0 < v1)
#pragma unroll
        for (int q = 0; q < PER; q++) bits[threadIdx.x + q * ORDER_NT] = 0;
        __syncthreads();
        int before = 0;
        auto set = [&](int32_t j) {
            const uint32_t i = (uint32_t)j - (uint32_t)first;
            if (i < (uint32_t)ORDER_WINDOW) atomicOr(&bits[i >> 5], 1u << (i & 31));
            before += j < (int32_t)first ? 1 : 0;
        };
#pragma unroll 4
        for (int32_t k = v0 + 4 * (int32_t)threadIdx.x; k < v1; k += 4 * ORDER_NT) {
            const int4 v = *reinterpret_cast<const int4 *>(l.perm + k);
            set(v.x), set(v.y), set(v.z), set(v.w);
        }
        if (s0 + (int32_t)threadIdx.x < v0) set(l.perm[s0 + threadIdx.x]);
        if (v1 + (int32_t)threadIdx.x < s1) set(l.perm[v1 + threadIdx.x]);
        const int smaller = wave_incl_scan(before);
        if (lane == 63) s_before[wid] = smaller;
        __syncthreads();
        uint32_t b[PER];
        int n = 0;
#pragma unroll
        for (int q = 0; q < PER; q++) {
            b[q] = bits[PER * threadIdx.x + q];
            n += __popc(b[q]);
        }
        const int incl = wave_incl_scan(n);
        if (lane == 63) s_tot[wid] = incl;
        __syncthreads();
        int32_t to = s0 + incl - n;
#pragma unroll
        for (int w = 0; w < ORDER_NT / 64; w++) to += s_before[w] + (w < wid ? s_tot[w] : 0);
#pragma unroll
        for (int q = 0; q < PER; q++)
            for (uint32_t m = b[q]; m; m &= m - 1)
                l.rank[to++] = (int32_t)first + 32 * (PER * (int32_t)threadIdx.x + q) + __ffs(m) - 1;
        __syncthreads();  // bits and sums are read
    }
}

// Storage of the tile sums of n values and of every level above them.
int64_t sums_size(int64_t n) {
    int64_t tot = 1;
    do {
        n = (n + SCAN_TILE - 1) / SCAN_TILE;
        tot += n;
    } while (n > 1);
    return tot;
}

}  // namespace

int bin_lists(vpbs_ctx *c, SortBuffers &sb, BinList *lists, int count, hipStream_t s) {
    BinGroup g{};
    g.count = count;
    g.geom.box = c->box;
    g.geom.M = c->p.nufft_m;
    g.geom.hz = slab_hz(c->p.precision == VPBS_F32 ? 4 : 8, c->G[0]);
    for (int d = 0; d < 3; d++) {
        g.geom.Nc[d] = c->Nc[d];
        g.geom.G[d] = c->G[d];
        g.geom.scale[d] = (double)c->G[d] / c->p.Ls[d];
    }
    int64_t n = 0, nsum = 0, nlarge = 0, nmax = 0;  // nlarge: at most
    for (int t = 0; t < count; t++) {
        n += lists[t].n;
        nsum += sums_size(lists[t].nbins + 1);
        if (lists[t].order_large && bin_large(lists[t].n, lists[t].n)) nlarge += lists[t].n / (BIN_LARGE + 1);
        nmax = std::max(nmax, lists[t].n);
    }
    VPBS_TRY(grow(c, &sb.rank, &sb.cap_n, n));
    VPBS_TRY(grow(c, &sb.sums, &sb.cap_sums, nsum));
    if (nlarge) {
        VPBS_TRY(grow(c, &sb.large, &sb.cap_large, 1 + 2 * nlarge));
        g.large = sb.large;
    }
    unsigned eb = 0, tb = 0;
    int32_t *rank = sb.rank, *sums = sb.sums;
    bool deep = false;
    for (int t = 0; t < count; t++) {
        BinList &l = lists[t];
        l.rank = rank;
        l.sums = sums;
        rank += l.n;
        sums += sums_size(l.nbins + 1);
        g.l[t] = l;
        g.elem_block[t] = eb;
        g.scan_block[t] = tb;
        eb += nblocks(l.n, 256);
        const unsigned nt = nblocks(l.nbins + 1, SCAN_TILE);
        deep |= nt > SCAN_FLAT_TILES;
        tb += nt;
    }
    bin_zero<<<tb, 256, 0, s>>>(g);
    bin_histogram<<<eb, 256, 0, s>>>(g);
    bin_tile_sums<<<tb, SCAN_BS, 0, s>>>(g);
    if (deep)
        for (int t = 0; t < count; t++) {
            const int64_t nt = nblocks(g.l[t].nbins + 1, SCAN_TILE);
            scan_levels(g.l[t].sums, nt, g.l[t].sums + nt, s);
        }
    bin_scan<<<tb, SCAN_BS, 0, s>>>(g, deep);
    bin_scatter<<<eb, 256, 0, s>>>(g);
    if (nlarge) {
        const int64_t windows = (nmax + ORDER_WINDOW - 1) / ORDER_WINDOW;
        bin_order<<<(unsigned)std::min(nlarge * windows, ORDER_BLOCKS), ORDER_NT, 0, s>>>(g, (int)windows);
    }
    VPBS_HIP(c, hipGetLastError());
    return VPBS_OK;
}

}  // namespace vpbs
