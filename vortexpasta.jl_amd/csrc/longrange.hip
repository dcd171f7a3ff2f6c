// Long-range part of the Ewald-split Biot–Savart sum on gfx950: a NUFFT with an
// "exponential of semicircle" (ES) kernel, rocFFT, and one fused Fourier-space
// kernel.
//
//   ω̂(k) = (Γ/V) Σ_j q_j e^{-ik·s_j}         type 1 (longrange.jl:488-495,
//                                           nonuniformffts.jl:173-192)
//   v̂ = i k × ω̂ / k²,  ψ̂ = ω̂ / k²          (longrange.jl:102-142)
//   × exp(-k²/4α²)                          Ewald Gaussian (cache_common.jl:64-76)
//   u(x_i) = Σ_k û(k) e^{ik·x_i}             type 2 (nonuniformffts.jl:195-212)
//
// restricted to the modes kept by _ensure_hermitian_symmetry!
// (longrange.jl:556-583), optionally to |k| ≤ kmax (truncate_spherical).
//
// Kernels:
//   bin_lists       points by the tile, nodes by the slab of their first stencil cell on
//                   the σ-oversampled grid (sort.hip); gather_records their records
//   spread_tiles_kernel  one wavefront per grid tile (16×8×8 cells) takes the points
//                   whose stencils reach it (they start in the tile or in the one or
//                   two tiles before it along each axis) and accumulates their
//                   outer products x-weights ⊗ (y-weight · z-weight · charge) on the
//                   matrix cores, the tile in accumulator registers: every grid value
//                   written exactly once, no atomics, no zero-fill pass,
//                   deterministic order
//   FFT             batched contiguous 1D c2c transforms on rocFFT along x, y and
//                   z, with pencil transposes of our own between them:
//                   x: the real grid holds pairs of y-rows as one complex row, so
//                      one c2c transforms two real rows;
//                   pair_split_to_ypencils: separates the pair, A = (Z_k + conj Z_-k)/2,
//                      B = (Z_k - conj Z_-k)/2i, keeps the retained kx and makes
//                      y contiguous; ypencils_to_zpencils keeps the retained ky and
//                      makes z contiguous. The inverse mirrors this and rebuilds
//                      the Hermitian half kx < 0 and the zero modes.
//   fourier_kernel  deconvolution (twice: type 1 and type 2), Γ/V, Green function,
//                   curl, Ewald Gaussian, zeroing of dropped modes — one pass over
//                   the z-pencils of retained (kx, ky), in place
//   interp_kernel_wave  W³ ES-weighted gather, one wavefront per node
// Everything is templated on the grid type (double for the FP64 path, float
// for the FP32-bulk path).
#include "vpbs_internal.hpp"
#include "device_util.hpp"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <type_traits>
#include <vector>

// Scratch of the allocation-free energy spectrum (vpbs_energy_spectrum_noalloc): the
// per-block partial spectra followed by the summed spectrum. Each GPU the library runs on
// holds its own copy until the process ends; host code reaches it only through the
// per-device address taken with hipGetSymbolAddress at context creation.
constexpr int SPEC_NA_BLOCKS = 256;
constexpr int SPEC_NA_MAXBINS = 1024;
static __device__ __align__(256) double scratch[(size_t)SPEC_NA_BLOCKS * SPEC_NA_MAXBINS + SPEC_NA_MAXBINS];

namespace vpbs {

namespace {

constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
double *g_scratch_ptr[MAX_DEVICES] = {};  // device address of `scratch` on each GPU (null: not taken yet)

// Spreading tile: 16 × 8 × 8 cells: 16 x-cells are the columns and 16 rows (8 in y,
// 2 in z) the rows of a 16×16 matrix-core tile, 4 of them and 3 components in 48
// (FP32) or 96 (FP64) accumulator registers.
constexpr int TX = SPREAD_TX, TY = SPREAD_TY, TZ = SPREAD_TZ;

inline unsigned nblocks(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

template <typename T>
__device__ inline T es_kernel(T z, T beta) {
    T s = (T)1 - z * z;
    return s < (T)0 ? (T)0 : exp(beta * (sqrt(s) - (T)1));
}

__device__ inline int wrapi(int i, int n) {
    i %= n;
    return i < 0 ? i + n : i;
}

// i in (-n, 2n) -> i mod n without an integer division
__device__ inline int wrap1(int i, int n) {
    i += (i < 0) ? n : 0;
    i -= (i >= n) ? n : 0;
    return i;
}

struct LRGeom {
    int G[3];
    double scale[3];  // G/L
    int ntile[3];
    int M;
    int64_t cstride;  // real grid values per component
};

// Per tile-sorted point, the record read by spreading: the 2m kernel weights
// along x, y and z, then the 3 charge components, padded to 16 bytes.
constexpr int rec_len(int W) { return (3 * W + 3 + 3) & ~3; }

template <typename CT>
struct alignas(2 * sizeof(CT)) Cx {
    CT re, im;
};

// ----------------------------------------------------------------------------

// Tile-sorted copy of the points: per point and direction d the first stencil
// index i0_d = ⌊u_d⌋ - m + 1 (wrapped into [0, G_d), component-major for the
// overlap tests) and one record (rec_len(2m) values) holding the 2m kernel
// weights φ((i0_d + k - u_d)/m) per direction and the charge, computed once
// here instead of once per tile in the spreading kernel.
// Records are rec_len(W) values (a multiple of 16 bytes) moved with 16-byte vector
// accesses: one thread writes a whole record.
template <typename CT, int N>
__device__ __forceinline__ void store_rec(CT *__restrict__ p, const CT (&r)[N]) {
    static_assert((N * sizeof(CT)) % 16 == 0, "records are whole 16-byte vectors");
    if constexpr (sizeof(CT) == 4) {
#pragma unroll
        for (int k = 0; k < N; k += 4) reinterpret_cast<float4 *>(p)[k / 4] = float4{r[k], r[k + 1], r[k + 2], r[k + 3]};
    } else {
#pragma unroll
        for (int k = 0; k < N; k += 2) reinterpret_cast<double2 *>(p)[k / 2] = double2{r[k], r[k + 1]};
    }
}

// First stencil cells and record (kernel weights, then the charge if chg) of the element at
// place t of its bins' lists, stored at its place in the order (bin, original index), which is
// returned with the element in j.
template <typename CT, int W, int REC>
__device__ inline int64_t gather_record(int64_t t, int64_t n, const int32_t *key, const int32_t *start,
                                        const int32_t *perm, const int32_t *ordered, const double *pos, const double *chg, const LRGeom &g,
                                        CT beta, int32_t *si0, CT *rec, int32_t &j) {
    constexpr int M = W / 2;
    j = perm[t];
    const int32_t b = key[j], s0 = start[b], s1 = start[b + 1];
    int64_t s = t;
    if (bin_large(n, s1 - s0))
        j = ordered[t];
    else
        s = bin_place(perm, s0, s1, j);
    CT r[REC];
#pragma unroll
    for (int k = 3 * W; k < REC; k++) r[k] = (CT)0;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const double u = pos[d * n + j] * g.scale[d];
        const int i0 = (int)floor(u) - M + 1;
        si0[d * n + s] = wrapi(i0, g.G[d]);
#pragma unroll
        for (int k = 0; k < W; k++) r[d * W + k] = es_kernel<CT>((CT)(((double)(i0 + k) - u) / (double)M), beta);
        if (chg) r[3 * W + d] = (CT)chg[d * n + j];
    }
    store_rec(rec + s * REC, r);
    return s;
}

template <typename CT>
struct GatherArgs {
    LRGeom g;
    CT beta;
    int64_t Nq, Np;
    unsigned point_blocks;  // blocks of 256 points, followed by blocks of 256 nodes
    const int32_t *pkey, *pstart, *pperm, *pordered, *nkey, *nstart, *nperm, *nordered;
    const double *pts, *chg, *nodes;
    int32_t *pi0, *ni0, *nnode;  // nnode: node of each slab-sorted place
    CT *prec, *nrec;
};

// Records of the tile-sorted points (spreading) and of the slab-sorted nodes (interpolation
// fused with the inverse x transform: their W weights per direction, padded with zeros).
template <typename CT, int W>
__global__ __launch_bounds__(256) void gather_records(GatherArgs<CT> a) {
    int32_t j;
    if (blockIdx.x < a.point_blocks) {
        const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
        if (t >= a.Nq) return;
        gather_record<CT, W, rec_len(W)>(t, a.Nq, a.pkey, a.pstart, a.pperm, a.pordered, a.pts, a.chg, a.g, a.beta, a.pi0, a.prec, j);
    } else {
        const int64_t t = (int64_t)(blockIdx.x - a.point_blocks) * 256 + threadIdx.x;
        if (t >= a.Np) return;
        const int64_t s = gather_record<CT, W, slab_rec_len(W, (int)sizeof(CT))>(
            t, a.Np, a.nkey, a.nstart, a.nperm, a.nordered, a.nodes, nullptr, a.g, a.beta, a.ni0, a.nrec, j);
        a.nnode[s] = j;
    }
}

template <typename CT>
void launch_gather(const GatherArgs<CT> &a, unsigned nb, hipStream_t s) {
    switch (a.g.M) {
        case 2: gather_records<CT, 4><<<nb, 256, 0, s>>>(a); break;
        case 3: gather_records<CT, 6><<<nb, 256, 0, s>>>(a); break;
        case 4: gather_records<CT, 8><<<nb, 256, 0, s>>>(a); break;
        case 5: gather_records<CT, 10><<<nb, 256, 0, s>>>(a); break;
        case 6: gather_records<CT, 12><<<nb, 256, 0, s>>>(a); break;
        case 7: gather_records<CT, 14><<<nb, 256, 0, s>>>(a); break;
        default: gather_records<CT, 16><<<nb, 256, 0, s>>>(a); break;
    }
}

// ----------------------------------------------------------------------------
// Spreading (type 1), gather form.

// Block b of the launch handles tile xcd_tile(b): blocks are dealt to the 8 XCDs
// round-robin, so consecutive blocks of one XCD get consecutive tiles and the
// point data shared by neighbouring tiles stays in that XCD's L2.
__device__ inline int64_t xcd_tile(int64_t b, int64_t ntiles) {
    const int64_t per = (ntiles + 7) / 8;
    return (b % 8) * per + b / 8;
}

// f(std::integral_constant<int, I>) for I = B .. E-1: register arrays indexed
// through it keep compile-time indices and stay in registers.
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}

// Matrix-core tile D (16×16) += A (16×4)·B (4×16): lane l holds A[l % 16][l / 16],
// B[l / 16][l % 16] and four values of column l % 16 of D, rows 4·(l / 16) + v in FP32
// and l / 16 + 4·v in FP64. (g, v) of row i of A below is the (l / 16, v) that holds row i of D.
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
template <typename CT>
using acc4 = std::conditional_t<sizeof(CT) == 4, f32x4, f64x4>;
__device__ __forceinline__ f32x4 mfma_16x16x4(float a, float b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f64x4 mfma_16x16x4(double a, double b, f64x4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Tiles along an axis in which the stencils reaching a tile of T cells start.
constexpr int start_tiles(int W, int T) { return 1 + (W - 1 + T - 1) / T; }
// Points staged in LDS at a time: 8 KB of records at W = 8, 4 (FP32) or 3 (FP64) wavefronts per SIMD.
template <typename CT>
constexpr int spread_batch() {
    return sizeof(CT) == 4 ? 64 : 32;
}

// Spreading (type 1): one wavefront per 16×8×8 tile. A point adds w_x[x]·(w_y[y] w_z[z] q_c)
// to cell (x, y, z) of component c: over four points this is the product of a 16×4 matrix
// (rows (y, z), columns the points) and a 4×16 one (the points, x), which the matrix cores
// add to the accumulators of 16 rows: lane = (x, four rows).
//  1) the point ranges of the tiles in which stencils reaching this one start;
//  2) their points are tested 64 at a time, the kept ones queued in order in LDS and, a
//     batch at a time, their records (weights, charge) copied to LDS by all lanes;
//  3) four points per step: each lane takes the x-weight of its column, the y- and z-weights
//     of its row (the record's zero padding outside the stencil) and the charge of its
//     point; the row blocks that none of the four points reaches are skipped.
// Summation order is fixed (range, then sorted order): results are deterministic. The tile is
// written once, from the accumulators: two rows of a pair row per store.
//
// What bounds it: a point reaches 5.05 tiles on average (W = 8). One lane per row cost 80 VALU
// instructions per point and tile, 48 of them FMAs of which 90% multiplied zeros; here it is
// about 15, and 8 matrix instructions per four points. The write of the tile is the floor:
// 3.0M points on 768³, alone, 2.55 -> 1.65 ms in FP32 (5.4 GB written: 3.3 TB/s) and 5.2 -> 2.5 ms
// in FP64 (10.9 GB: 4.4 TB/s); 187k points at W = 12 on 288³, FP64, 0.80 -> 0.29 ms.
template <typename CT, int W>
__global__ __launch_bounds__(64) void spread_tiles_kernel(LRGeom g, int64_t Nq, const int32_t *__restrict__ tstart,
                                                          const int32_t *__restrict__ si0,
                                                          const CT *__restrict__ rec, CT *__restrict__ grid) {
    constexpr int REC = rec_len(W), NB = spread_batch<CT>();
    constexpr int VL = 16 / sizeof(CT), NV = REC / VL;  // record in 16-byte vectors
    constexpr int NX = start_tiles(W, TX), NY = start_tiles(W, TY), NZ = start_tiles(W, TZ), NN = NX * NY * NZ;
    static_assert(REC > 3 * W + 3 && NN <= 64, "the record ends in a zero; one lane per range");
    constexpr int ZERO = REC - 1;
    constexpr int ITEMS = NB * NV / 64;  // vectors of a batch per lane
    static_assert(ITEMS * 64 == NB * NV, "whole vectors per lane");
    typedef CT V16 __attribute__((ext_vector_type(VL)));
    __shared__ V16 s_vec[NB * NV];
    __shared__ int2 s_meta[NB + 64];  // queue: sorted index, stencil start relative to the tile (+64, 8 bits each)
    const CT *s_rec = reinterpret_cast<const CT *>(s_vec);

    const int lane = threadIdx.x;
    const int64_t ntl = (int64_t)g.ntile[0] * g.ntile[1] * g.ntile[2];
    const int64_t tile = xcd_tile(blockIdx.x, ntl);
    if (tile >= ntl) return;  // the whole (one-wavefront) block
    const int tix = (int)(tile % g.ntile[0]);
    const int tiy = (int)((tile / g.ntile[0]) % g.ntile[1]);
    const int tiz = (int)(tile / ((int64_t)g.ntile[0] * g.ntile[1]));
    const int t0x = tix * TX, t0y = tiy * TY, t0z = tiz * TZ;
    const int col = lane & 15, grp = lane >> 4;
    // row (y, z) = (4·(g % 2) + v, g / 2) of a block for row `col` of A
    const int ag = sizeof(CT) == 4 ? col >> 2 : col & 3, av = sizeof(CT) == 4 ? col & 3 : col >> 2;
    const int ay = 4 * (ag & 1) + av, az = ag >> 1;

    acc4<CT> acc[TZ / 2][3];
    static_for<0, TZ / 2>([&](auto R) {
        constexpr int r = decltype(R)::value;
#pragma unroll
        for (int c = 0; c < 3; c++) acc[r][c] = acc4<CT>{(CT)0, (CT)0, (CT)0, (CT)0};
    });

    // 1) point ranges (lane q < NN)
    int s0 = 0, len = 0;
    if (lane < NN) {
        const int tx = wrap1(tix - lane % NX, g.ntile[0]), ty = wrap1(tiy - (lane / NX) % NY, g.ntile[1]),
                  tz = wrap1(tiz - lane / (NX * NY), g.ntile[2]);
        const int64_t tl = ((int64_t)tz * g.ntile[1] + ty) * g.ntile[0] + tx;
        s0 = tstart[tl];
        len = tstart[tl + 1] - s0;
    }
    const int incl = wave_incl_scan(len);
    const int ncand = __builtin_amdgcn_readlane(incl, NN - 1);

    if (ncand > 0) {
        // candidate cnd of range q is point off[q] + cnd (cnd ≥ pre[q])
        const int excl = incl - len, offv = s0 - excl;
        int pre[NN];
#pragma unroll
        for (int q = 0; q < NN; q++) pre[q] = __builtin_amdgcn_readlane(excl, q);

        int nq = 0;  // queued points
        for (int base = 0; base < ncand;) {
            // 2) overlap test and queue
            const int cnd = base + lane;
            int q = 0;
#pragma unroll
            for (int t = 1; t < NN; t++) q += cnd >= pre[t] ? 1 : 0;
            const int sidx = cnd + __shfl(offv, q, 64);
            bool keep = false;
            int meta = 0;
            if (cnd < ncand) {
                // stencil start relative to the tile, in (-G, T): it reaches the tile above -W
                int sx = wrap1(si0[sidx] - t0x, g.G[0]), sy = wrap1(si0[Nq + sidx] - t0y, g.G[1]),
                    sz = wrap1(si0[2 * Nq + sidx] - t0z, g.G[2]);
                sx = sx < TX ? sx : sx - g.G[0];
                sy = sy < TY ? sy : sy - g.G[1];
                sz = sz < TZ ? sz : sz - g.G[2];
                keep = sx > -W && sy > -W && sz > -W;
                meta = (sx + 64) | ((sy + 64) << 8) | ((sz + 64) << 16);
            }
            const unsigned long long mask = __ballot(keep);
            if (keep) s_meta[nq + __popcll(mask & ((1ull << lane) - 1ull))] = make_int2(sidx, meta);
            nq += __popcll(mask);
            base += 64;
            // 3) whole batches, and what is left after the last candidates
            while (nq >= NB || (base >= ncand && nq > 0)) {
                const int n = nq < NB ? nq : NB, n4 = (n + 3) & ~3;
                // up to three points past the end: stencils outside the tile (all weights zero)
                if (lane < n4 - n) s_meta[n + lane] = make_int2(s_meta[0].x, 0);
                __syncthreads();
                V16 t[ITEMS];
#pragma unroll
                for (int i = 0; i < ITEMS; i++) {
                    const int e = lane + 64 * i, p = e / NV, pc = p < n4 ? p : 0;
                    t[i] = reinterpret_cast<const V16 *>(rec)[(int64_t)s_meta[pc].x * NV + (e - p * NV)];
                }
#pragma unroll
                for (int i = 0; i < ITEMS; i++) s_vec[lane + 64 * i] = t[i];
                __syncthreads();
#pragma unroll 1
                for (int p0 = 0; p0 < n4; p0 += 4) {
                    const int p = p0 + grp;
                    const unsigned m = (unsigned)s_meta[p].y;
                    const int kx = col + 64 - (int)(m & 255u), ky = ay + 64 - (int)((m >> 8) & 255u),
                              kz = az + 64 - (int)(m >> 16);
                    const CT *rp = s_rec + p * REC;
                    const CT wx = rp[(unsigned)kx < (unsigned)W ? kx : ZERO];
                    const CT wy = rp[(unsigned)ky < (unsigned)W ? W + ky : ZERO];
                    const CT q0 = wy * rp[3 * W], q1 = wy * rp[3 * W + 1], q2 = wy * rp[3 * W + 2];
                    CT wz[TZ / 2];
                    bool on[TZ / 2];
#pragma unroll
                    for (int r = 0; r < TZ / 2; r++) {
                        on[r] = (unsigned)(kz + 2 * r) < (unsigned)W;
                        wz[r] = rp[on[r] ? 2 * W + kz + 2 * r : ZERO];
                    }
                    static_for<0, TZ / 2>([&](auto R) {
                        constexpr int r = decltype(R)::value;
                        if (__ballot(on[r])) {
                            acc[r][0] = mfma_16x16x4(wz[r] * q0, wx, acc[r][0]);
                            acc[r][1] = mfma_16x16x4(wz[r] * q1, wx, acc[r][1]);
                            acc[r][2] = mfma_16x16x4(wz[r] * q2, wx, acc[r][2]);
                        }
                    });
                }
                // ≤ 64 entries stay: one per lane moves to the front
                const int left = nq - n;
                const int2 mv = s_meta[NB + (lane < left ? lane : 0)];
                __syncthreads();
                if (lane < left) s_meta[lane] = mv;
                __syncthreads();
                nq = left;
            }
        }
    }

    // write: values v, v + 1 of a lane are the rows y, y + 1 of one pair row at its x: one
    // 8- or 16-byte store each, 16 lanes along x; 32-bit offsets from the tile origin
    using C2 = Cx<CT>;
    C2 *const tile0 =
        reinterpret_cast<C2 *>(grid) + ((int64_t)t0z * (g.G[1] >> 1) + (t0y >> 1)) * g.G[0] + t0x;
    const int rstride = g.G[0], zstride = (g.G[1] >> 1) * rstride;
    const int o0 = (grp >> 1) * zstride + 2 * (grp & 1) * rstride + col;
    static_for<0, 3>([&](auto C) {
        constexpr int c = decltype(C)::value;
        C2 *const dst = tile0 + c * (g.cstride >> 1) + o0;
        static_for<0, TZ / 2>([&](auto R) {
            constexpr int r = decltype(R)::value;
            dst[2 * r * zstride] = C2{acc[r][c][0], acc[r][c][1]};
            dst[2 * r * zstride + rstride] = C2{acc[r][c][2], acc[r][c][3]};
        });
    });
}

template <typename CT>
void launch_spread(const LRGeom &g, int64_t ntiles, int64_t Nq, const int32_t *tstart, const int32_t *si0,
                   const CT *rec, CT *grid, hipStream_t s) {
    const unsigned n = (unsigned)(((ntiles + 7) / 8) * 8);  // xcd_tile() maps 8·⌈n/8⌉ blocks onto the tiles
    switch (g.M) {
        case 2: spread_tiles_kernel<CT, 4><<<n, 64, 0, s>>>(g, Nq, tstart, si0, rec, grid); break;
        case 3: spread_tiles_kernel<CT, 6><<<n, 64, 0, s>>>(g, Nq, tstart, si0, rec, grid); break;
        case 4: spread_tiles_kernel<CT, 8><<<n, 64, 0, s>>>(g, Nq, tstart, si0, rec, grid); break;
        case 5: spread_tiles_kernel<CT, 10><<<n, 64, 0, s>>>(g, Nq, tstart, si0, rec, grid); break;
        case 6: spread_tiles_kernel<CT, 12><<<n, 64, 0, s>>>(g, Nq, tstart, si0, rec, grid); break;
        case 7: spread_tiles_kernel<CT, 14><<<n, 64, 0, s>>>(g, Nq, tstart, si0, rec, grid); break;
        default: spread_tiles_kernel<CT, 16><<<n, 64, 0, s>>>(g, Nq, tstart, si0, rec, grid); break;
    }
}

// ----------------------------------------------------------------------------
// Pencil transposes between the 1D transforms. All four move 32×32 (or
// 32×16-pair) tiles through LDS so that both the loads and the stores run
// along contiguous rows.

// Forward, after the x-pass: Z = FFT_x(row 2p + i·row 2p+1) for every pair p.
// Writes ypen[c][kx][z][y] (y contiguous) for the retained kx ∈ [0, nkx):
// A_k = (Z_k + conj Z_{-k})/2 for y = 2p, B_k = (Z_k - conj Z_{-k})/(2i) for y = 2p+1.
// Grid: (⌈nkx/32⌉, G1/32, 3·G2), 256 threads.
template <typename CT>
__global__ __launch_bounds__(256) void pair_split_to_ypencils(const Cx<CT> *__restrict__ zrow,
                                                              Cx<CT> *__restrict__ ypen, int G0, int G1, int G2,
                                                              int nkx) {
    __shared__ Cx<CT> sk[16][33], sm[16][33];
    const int kx0 = blockIdx.x * 32, p0 = blockIdx.y * 16;
    const int cz = blockIdx.z, c = cz / G2, z = cz - c * G2;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const Cx<CT> *rows = zrow + (int64_t)cz * (G1 >> 1) * G0;
    const int kx = kx0 + tx;
    if (kx < nkx) {
        const int km = kx == 0 ? 0 : G0 - kx;
        for (int pp = ty; pp < 16; pp += 8) {
            const Cx<CT> *r = rows + (int64_t)(p0 + pp) * G0;
            sk[pp][tx] = r[kx];
            sm[pp][tx] = r[km];
        }
    }
    __syncthreads();
    const int pp = tx >> 1, par = tx & 1;
    for (int kk = ty; kk < 32 && kx0 + kk < nkx; kk += 8) {
        const Cx<CT> a = sk[pp][kk], b = sm[pp][kk];
        Cx<CT> o;
        if (par == 0) {
            o.re = (a.re + b.re) * (CT)0.5;
            o.im = (a.im - b.im) * (CT)0.5;
        } else {
            o.re = (a.im + b.im) * (CT)0.5;
            o.im = (b.re - a.re) * (CT)0.5;
        }
        ypen[(((int64_t)c * nkx + kx0 + kk) * G2 + z) * G1 + 2 * p0 + tx] = o;
    }
}

// Forward, after the y-pass: ypen[plane][z][iy] -> zpen[plane][j][z] for the
// retained ky = j (j ≤ K1) or j - nky (j > K1), plane = c·nkx + kx.
// Grid: (G2/32, ⌈nky/32⌉, 3·nkx).
template <typename CT>
__global__ __launch_bounds__(256) void ypencils_to_zpencils(const Cx<CT> *__restrict__ ypen,
                                                            Cx<CT> *__restrict__ zpen, int G1, int G2, int nky,
                                                            int K1) {
    __shared__ Cx<CT> s[32][33];
    const int z0 = blockIdx.x * 32, j0 = blockIdx.y * 32;
    const int64_t plane = blockIdx.z;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const Cx<CT> *src = ypen + plane * G2 * G1;
    Cx<CT> *dst = zpen + plane * nky * G2;
    const int j = j0 + tx;
    if (j < nky) {
        const int iy = j <= K1 ? j : G1 + j - nky;
        for (int zz = ty; zz < 32; zz += 8) s[zz][tx] = src[(int64_t)(z0 + zz) * G1 + iy];
    }
    __syncthreads();
    for (int jj = ty; jj < 32 && j0 + jj < nky; jj += 8) dst[(int64_t)(j0 + jj) * G2 + z0 + tx] = s[tx][jj];
}

// Inverse, after the z-pass: zpen[plane][j][z] -> ypen[plane][z][iy] for every
// iy, zero where ky is not retained. Grid: (G2/32, G1/32, 3·nkx).
template <typename CT>
__global__ __launch_bounds__(256) void zpencils_to_ypencils(const Cx<CT> *__restrict__ zpen,
                                                            Cx<CT> *__restrict__ ypen, int G1, int G2, int nky,
                                                            int K1) {
    __shared__ Cx<CT> s[32][33];
    const int z0 = blockIdx.x * 32, iy0 = blockIdx.y * 32;
    const int64_t plane = blockIdx.z;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    const Cx<CT> *src = zpen + plane * nky * G2;
    Cx<CT> *dst = ypen + plane * G2 * G1;
    for (int jj = ty; jj < 32; jj += 8) {
        const int iy = iy0 + jj;
        const int ky = iy <= (G1 >> 1) ? iy : iy - G1;
        Cx<CT> v{(CT)0, (CT)0};
        if (ky >= -K1 && ky <= K1) v = src[(int64_t)(ky >= 0 ? ky : ky + nky) * G2 + z0 + tx];
        s[jj][tx] = v;
    }
    __syncthreads();
    for (int zz = ty; zz < 32; zz += 8) dst[(int64_t)(z0 + zz) * G1 + iy0 + tx] = s[tx][zz];
}

// Inverse, after the y-pass: rebuild each pair row Z_k = A_k + i·B_k for every
// k ∈ [0, G0): A, B from ypen for k < nkx, their conjugates at G0 - k for
// k > G0 - nkx (Hermitian symmetry of real rows), zero otherwise; the DC term
// keeps only its real part (what a c2r transform uses).
// Grid: (G0/32, G1/32, 3·G2).
template <typename CT>
__global__ __launch_bounds__(256) void ypencils_to_pair_rows(const Cx<CT> *__restrict__ ypen,
                                                             Cx<CT> *__restrict__ zrow, int G0, int G1, int G2,
                                                             int nkx) {
    __shared__ Cx<CT> s[32][33];
    const int k0 = blockIdx.x * 32, p0 = blockIdx.y * 16;
    const int cz = blockIdx.z, c = cz / G2, z = cz - c * G2;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int kk = ty; kk < 32; kk += 8) {
        const int k = k0 + kk;
        int kx = -1;
        bool cj = false;
        if (k < nkx) {
            kx = k;
        } else if (k > G0 - nkx) {
            kx = G0 - k;
            cj = true;
        }
        Cx<CT> v{(CT)0, (CT)0};
        if (kx >= 0) {
            v = ypen[(((int64_t)c * nkx + kx) * G2 + z) * G1 + 2 * p0 + tx];
            if (cj) v.im = -v.im;
            if (k == 0) v.im = (CT)0;
        }
        s[kk][tx] = v;
    }
    __syncthreads();
    Cx<CT> *rows = zrow + (int64_t)cz * (G1 >> 1) * G0;
    for (int pp = ty; pp < 16; pp += 8) {
        const Cx<CT> A = s[tx][2 * pp], B = s[tx][2 * pp + 1];
        rows[(int64_t)(p0 + pp) * G0 + k0 + tx] = Cx<CT>{A.re - B.im, A.im + B.re};
    }
}

// ----------------------------------------------------------------------------
// Fused Fourier-space kernel, in place on the z-pencils [3][nkx][nky][G2].

template <typename CT>
struct FourierArgs {
    int G[3];
    int nkx, nky;
    int64_t cstride;  // complex values per component
    int kmax[3];      // retained: kx ∈ [0, kmax0], |ky| ≤ kmax1, |kz| ≤ kmax2
    const double *dx, *dy, *dz;  // 1/ψ̂ per retained mode (dy, dz offset by kmax)
    double kscale[3];            // 2π/L
    double pref;                 // Γ/V
    double inv4a2;               // 1/(4α²)
    double kmax2_trunc;          // < 0: no spherical truncation
    int do_vel, do_psi;
    // unsmoothed field kept for the Fourier-space consumers (velocity if do_vel, else streamfunction):
    // uhat[3][nky][nkz][nkx], kz index jz ≤ kmax2 → kz = jz, else jz - nkz
    CT *uhat;
    int keep_uhat, nkz;
    int64_t ucstride;
};

template <typename CT>
__global__ void fourier_kernel(FourierArgs<CT> a, CT *__restrict__ spec, CT *__restrict__ spec2) {
    int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= a.cstride) return;
    const int iz = (int)(idx % a.G[2]);
    const int j = (int)((idx / a.G[2]) % a.nky);
    const int kx = (int)(idx / ((int64_t)a.G[2] * a.nky));
    const int ky = j <= a.kmax[1] ? j : j - a.nky;
    const int kz = iz <= a.G[2] / 2 ? iz : iz - a.G[2];
    bool keep = kz >= -a.kmax[2] && kz <= a.kmax[2];
    const double KX = a.kscale[0] * kx, KY = a.kscale[1] * ky, KZ = a.kscale[2] * kz;
    const double k2 = KX * KX + KY * KY + KZ * KZ;
    if (a.kmax2_trunc >= 0 && k2 > a.kmax2_trunc) keep = false;
    CT *c1 = spec + 2 * idx;   // complex (re, im) of component 0
    CT *c2 = spec2 + 2 * idx;
    const int64_t cs = 2 * a.cstride;
    // slot of this mode in the kept field (the retained kz only)
    CT *cu = nullptr;
    if (a.keep_uhat && kz >= -a.kmax[2] && kz <= a.kmax[2]) {
        const int jz = kz >= 0 ? kz : kz + a.nkz;
        cu = a.uhat + 2 * (((int64_t)j * a.nkz + jz) * a.nkx + kx);
    }
    if (!keep || k2 == 0) {
        if (cu) {
#pragma unroll
            for (int d = 0; d < 3; d++) cu[2 * d * a.ucstride] = cu[2 * d * a.ucstride + 1] = (CT)0;
        }
#pragma unroll
        for (int d = 0; d < 3; d++) {
            if (a.do_vel) {
                c1[d * cs] = (CT)0;
                c1[d * cs + 1] = (CT)0;
            }
            if (a.do_psi) {
                c2[d * cs] = (CT)0;
                c2[d * cs + 1] = (CT)0;
            }
        }
        // streamfunction-only: the vorticity buffer is not an output, leave it
        return;
    }
    const double D = a.dx[kx] * a.dy[ky + a.kmax[1]] * a.dz[kz + a.kmax[2]];
    // ω̂ = Γ/V · B̂ / ψ̂ ; output = op(ω̂) · e^{-k²/4α²} / ψ̂
    const double s = a.pref * D * D * exp(-k2 * a.inv4a2) / k2;
    double wr[3], wi[3];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        wr[d] = (double)c1[d * cs] * s;
        wi[d] = (double)c1[d * cs + 1] * s;
    }
    if (cu) {
        // unsmoothed field: ω̂/k² (one deconvolution, no Ewald factor), then i k × for the velocity
        const double su = a.pref * D / k2;
        double ur[3], ui[3];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            ur[d] = (double)c1[d * cs] * su;
            ui[d] = (double)c1[d * cs + 1] * su;
        }
        if (a.do_vel) {
            const double ax = KY * ur[2] - KZ * ur[1], bx = KY * ui[2] - KZ * ui[1];
            const double ay = KZ * ur[0] - KX * ur[2], by = KZ * ui[0] - KX * ui[2];
            const double az = KX * ur[1] - KY * ur[0], bz = KX * ui[1] - KY * ui[0];
            ur[0] = -bx, ui[0] = ax, ur[1] = -by, ui[1] = ay, ur[2] = -bz, ui[2] = az;
        }
        const int64_t us = 2 * a.ucstride;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            cu[d * us] = (CT)ur[d];
            cu[d * us + 1] = (CT)ui[d];
        }
    }
    if (a.do_psi) {
#pragma unroll
        for (int d = 0; d < 3; d++) {
            c2[d * cs] = (CT)wr[d];
            c2[d * cs + 1] = (CT)wi[d];
        }
    }
    if (a.do_vel) {
        // i k × w: (i k × w)_x = i (KY w_z - KZ w_y), i (a + ib) = -b + ia
        const double ax = KY * wr[2] - KZ * wr[1], bx = KY * wi[2] - KZ * wi[1];
        const double ay = KZ * wr[0] - KX * wr[2], by = KZ * wi[0] - KX * wi[2];
        const double az = KX * wr[1] - KY * wr[0], bz = KX * wi[1] - KY * wi[0];
        c1[0] = (CT)(-bx);
        c1[1] = (CT)ax;
        c1[cs] = (CT)(-by);
        c1[cs + 1] = (CT)ay;
        c1[2 * cs] = (CT)(-bz);
        c1[2 * cs + 1] = (CT)az;
    }
}

// ----------------------------------------------------------------------------
// Consumers of the kept Fourier field.

// z-pencils of the band-filtered field, ready for the inverse transforms: the
// kept û on kmin² ≤ k² ≤ kmax² times the type-2 deconvolution, zero elsewhere.
template <typename CT>
__global__ void band_to_zpencils(FourierArgs<CT> a, double kmin2, double kmax2, double cf, double cc,
                                 CT *__restrict__ zp) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= a.cstride) return;
    const int iz = (int)(idx % a.G[2]);
    const int j = (int)((idx / a.G[2]) % a.nky);
    const int kx = (int)(idx / ((int64_t)a.G[2] * a.nky));
    const int ky = j <= a.kmax[1] ? j : j - a.nky;
    const int kz = iz <= a.G[2] / 2 ? iz : iz - a.G[2];
    const double KX = a.kscale[0] * kx, KY = a.kscale[1] * ky, KZ = a.kscale[2] * kz;
    const double k2 = KX * KX + KY * KY + KZ * KZ;
    const bool in = kz >= -a.kmax[2] && kz <= a.kmax[2] && k2 >= kmin2 && k2 <= kmax2;
    const int64_t cs = 2 * a.cstride, us = 2 * a.ucstride;
    CT *o = zp + 2 * idx;
    if (!in) {
#pragma unroll
        for (int d = 0; d < 3; d++) o[d * cs] = o[d * cs + 1] = (CT)0;
        return;
    }
    double D = a.dx[kx] * a.dy[ky + a.kmax[1]] * a.dz[kz + a.kmax[2]];
    if (cf > 0) D *= exp(-cf * k2) - exp(-cc * k2);  // difference of two Ewald Gaussians
    const int jz = kz >= 0 ? kz : kz + a.nkz;
    const CT *u = a.uhat + 2 * (((int64_t)j * a.nkz + jz) * a.nkx + kx);
#pragma unroll
    for (int d = 0; d < 3; d++) {
        o[d * cs] = (CT)((double)u[d * us] * D);
        o[d * cs + 1] = (CT)((double)u[d * us + 1] * D);
    }
}

// Energy spectrum of the kept field (Diagnostics/spectra.jl:89-196): mode k goes
// to bin n = trunc(|k|/Δk + 1/2) with weight f·|û|²/Δk (f = 1/2 on the kx = 0
// plane, 1 elsewhere; from the streamfunction |k × ψ̂|² = k²|ψ̂|²). One partial
// spectrum per block (LDS bins), summed over blocks in a fixed order.
template <typename CT>
__global__ void spectrum_partial(const CT *__restrict__ uhat, int64_t ucs, int nkx, int nkz, int K1, int K2,
                                 double kx_scale, double ky_scale, double kz_scale, double dk_inv, int nk,
                                 int from_psi, double *__restrict__ partial) {
    extern __shared__ double bins[];
    for (int b = threadIdx.x; b < nk; b += blockDim.x) bins[b] = 0.0;
    __syncthreads();
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < ucs;
         idx += (int64_t)gridDim.x * blockDim.x) {
        const int kx = (int)(idx % nkx);
        const int jz = (int)((idx / nkx) % nkz);
        const int j = (int)(idx / ((int64_t)nkx * nkz));
        const int ky = j <= K1 ? j : j - (2 * K1 + 1);
        const int kz = jz <= K2 ? jz : jz - nkz;
        const double KX = kx_scale * kx, KY = ky_scale * ky, KZ = kz_scale * kz;
        const double k2 = KX * KX + KY * KY + KZ * KZ;
        const int n = (int)(sqrt(k2) * dk_inv + 0.5);
        if (n >= nk) continue;
        double u2 = 0.0;
#pragma unroll
        for (int d = 0; d < 3; d++) {
            const double re = uhat[2 * (d * ucs + idx)], im = uhat[2 * (d * ucs + idx) + 1];
            u2 += re * re + im * im;
        }
        if (from_psi) u2 *= k2;
        atomicAdd(&bins[n], (kx == 0 ? 0.5 : 1.0) * u2 * dk_inv);
    }
    __syncthreads();
    for (int b = threadIdx.x; b < nk; b += blockDim.x) partial[(int64_t)blockIdx.x * nk + b] = bins[b];
}

// Sum of the partial spectra: a block takes SPEC_RB bins, SPEC_RT threads per bin add every SPEC_RT-th
// partial, then a fixed tree over them. Bound by load latency: one thread per bin that walks all 1024
// partials took 231 µs at 96 bins, this 6.
constexpr int SPEC_RB = 16, SPEC_RT = 64;
__global__ __launch_bounds__(SPEC_RB * SPEC_RT) void spectrum_reduce(const double *__restrict__ partial, int nblocks,
                                                                     int nk, double *__restrict__ Ek) {
    __shared__ double red[SPEC_RT][SPEC_RB];
    const int i = threadIdx.x % SPEC_RB, t = threadIdx.x / SPEC_RB, b = blockIdx.x * SPEC_RB + i;
    double s = 0.0;
    if (b < nk) {
#pragma unroll 8
        for (int k = t; k < nblocks; k += SPEC_RT) s += partial[(int64_t)k * nk + b];
    }
    red[t][i] = s;
    __syncthreads();
    for (int w = SPEC_RT / 2; w > 0; w >>= 1) {
        if (t < w) red[t][i] += red[t + w][i];
        __syncthreads();
    }
    if (t == 0 && b < nk) Ek[b] = red[0][i];
}

// ----------------------------------------------------------------------------
// Interpolation (type 2).

// Type-2 interpolation with a W³ stencil (W = 2m): one wavefront (block) per node.
// Lanes 0..3W-1 evaluate the node's 3·W kernel weights once and share them through
// LDS (exact copies); lane (a, b) = (lane % W, lane / W) then owns stencil column
// x = i0x + a and rows y = i0y + b + R·pass (R = ⌊64/W⌋ rows per pass) and walks the
// W z-planes, so a load instruction touches R rows of W consecutive values; the
// partial sums are combined by DPP steps in a fixed order (total in lane 63).
template <typename CT, int W>
__global__ __launch_bounds__(64) void interp_kernel_wave(LRGeom g, int64_t Np, const double *__restrict__ nodes,
                                                         CT beta, const CT *__restrict__ grid,
                                                         double *__restrict__ out) {
    constexpr int M = W / 2;
    constexpr int R = 64 / W;                  // y rows per pass
    constexpr int PASSES = (W + R - 1) / R;
    __shared__ CT s_w[3][W];
    const int lane = threadIdx.x;
    const int a = lane % W, b = lane / W;
    const bool lane_on = b < R;                // lanes beyond R·W idle
    // Blocks are dealt to the 8 XCDs round-robin; remap so that each XCD works
    // on a contiguous range of nodes (consecutive nodes share stencil rows,
    // which then stay in that XCD's L2).
    const int64_t per = ((int64_t)gridDim.x + 7) / 8;
    const int64_t i = (int64_t)(blockIdx.x % 8) * per + blockIdx.x / 8;
    if (i >= Np) return;  // the whole (one-wavefront) block
    const double ux = nodes[i] * g.scale[0];
    const double uy = nodes[Np + i] * g.scale[1];
    const double uz = nodes[2 * Np + i] * g.scale[2];
    const int i0x = (int)floor(ux) - M + 1, i0y = (int)floor(uy) - M + 1, i0z = (int)floor(uz) - M + 1;
    if (lane < 3 * W) {
        const int t = lane / W, c = lane - t * W;
        const double u = t == 0 ? ux : t == 1 ? uy : uz;
        const int i0 = t == 0 ? i0x : t == 1 ? i0y : i0z;
        s_w[t][c] = es_kernel<CT>((CT)(((double)(i0 + c) - u) / (double)M), beta);
    }
    __syncthreads();
    const CT wx = s_w[0][a];
    CT wz[W];
    int64_t gzo[W];
    const int64_t plane = (int64_t)g.G[0] * g.G[1];  // values per z-plane
#pragma unroll
    for (int c = 0; c < W; c++) {
        wz[c] = s_w[2][c];
        gzo[c] = (int64_t)wrapi(i0z + c, g.G[2]) * plane;
    }
    const int64_t gx = 2 * (int64_t)wrapi(i0x + a, g.G[0]);
    CT acc0 = 0, acc1 = 0, acc2 = 0;
#pragma unroll
    for (int pass = 0; pass < PASSES; pass++) {
        const int bb = b + R * pass;
        if (lane_on && bb < W) {
            const CT wy = s_w[1][bb];
            const int iy = wrapi(i0y + bb, g.G[1]);
            const int64_t gy = (int64_t)(iy >> 1) * 2 * g.G[0] + (iy & 1);
            const CT wxy = wx * wy;
#pragma unroll
            for (int c = 0; c < W; c++) {
                const int64_t off = gzo[c] + gy + gx;
                const CT w = wxy * wz[c];
                acc0 += w * grid[off];
                acc1 += w * grid[g.cstride + off];
                acc2 += w * grid[2 * g.cstride + off];
            }
        }
    }
    acc0 = wave_sum_last(acc0);
    acc1 = wave_sum_last(acc1);
    acc2 = wave_sum_last(acc2);
    if (lane == 63) {
        out[i] = (double)acc0;
        out[Np + i] = (double)acc1;
        out[2 * Np + i] = (double)acc2;
    }
}

template <typename CT>
void launch_interp(const LRGeom &g, int64_t Np, const double *nodes, CT beta, const CT *grid, double *out,
                   hipStream_t s) {
    const unsigned nb = (unsigned)(8 * ((Np + 7) / 8));  // one wavefront per node and block
    switch (g.M) {
        case 2: interp_kernel_wave<CT, 4><<<nb, 64, 0, s>>>(g, Np, nodes, beta, grid, out); break;
        case 3: interp_kernel_wave<CT, 6><<<nb, 64, 0, s>>>(g, Np, nodes, beta, grid, out); break;
        case 4: interp_kernel_wave<CT, 8><<<nb, 64, 0, s>>>(g, Np, nodes, beta, grid, out); break;
        case 5: interp_kernel_wave<CT, 10><<<nb, 64, 0, s>>>(g, Np, nodes, beta, grid, out); break;
        case 6: interp_kernel_wave<CT, 12><<<nb, 64, 0, s>>>(g, Np, nodes, beta, grid, out); break;
        case 7: interp_kernel_wave<CT, 14><<<nb, 64, 0, s>>>(g, Np, nodes, beta, grid, out); break;
        default: interp_kernel_wave<CT, 16><<<nb, 64, 0, s>>>(g, Np, nodes, beta, grid, out); break;
    }
}

__global__ void add3(int64_t n, const double *__restrict__ a, const double *__restrict__ b, double *__restrict__ o) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) o[i] = a[i] + b[i];
}

// ----------------------------------------------------------------------------
// Host helpers

// Gauss–Legendre nodes/weights on [0, 1] by Newton iteration on P_n.
void gauss_legendre01(int n, std::vector<double> &x, std::vector<double> &w) {
    x.resize(n);
    w.resize(n);
    for (int i = 0; i < n; i++) {
        double z = std::cos(M_PI * (i + 0.75) / (n + 0.5));
        double pp = 0;
        for (int it = 0; it < 100; it++) {
            double p1 = 1, p2 = 0;
            for (int j = 1; j <= n; j++) {
                double p3 = p2;
                p2 = p1;
                p1 = ((2.0 * j - 1.0) * z * p2 - (j - 1.0) * p3) / j;
            }
            pp = n * (z * p1 - p2) / (z * z - 1.0);
            double dz = p1 / pp;
            z -= dz;
            if (std::fabs(dz) < 1e-16) break;
        }
        x[i] = (1.0 - z) / 2.0;  // map to [0, 1]
        w[i] = 1.0 / ((1.0 - z * z) * pp * pp);  // = (2/((1-z²)P'²))/2
    }
}

// ψ̂(k) = 2m ∫_0^1 φ(z) cos(2πkmz/G) dz
double es_fourier(int k, int G, int m, double beta, const std::vector<double> &x, const std::vector<double> &w) {
    double s = 0;
    for (size_t q = 0; q < x.size(); q++) {
        double z = x[q];
        double phi = std::exp(beta * (std::sqrt(1 - z * z) - 1));
        s += w[q] * phi * std::cos(2 * M_PI * k * m * z / G);
    }
    return 2 * m * s;
}

template <typename CT>
FourierArgs<CT> fourier_args(const vpbs_ctx *c) {
    FourierArgs<CT> fa;
    for (int d = 0; d < 3; d++) {
        fa.G[d] = c->G[d];
        fa.kmax[d] = c->kmax_mode[d];
        fa.kscale[d] = 2 * M_PI / c->p.Ls[d];
    }
    fa.nkx = c->nkx;
    fa.nky = c->nky;
    fa.cstride = c->zpen_stride;
    fa.dx = c->deconv;
    fa.dy = c->deconv + (c->kmax_mode[0] + 1);
    fa.dz = fa.dy + (2 * c->kmax_mode[1] + 1);
    fa.pref = c->p.Gamma / (c->p.Ls[0] * c->p.Ls[1] * c->p.Ls[2]);
    fa.inv4a2 = 1.0 / (4 * c->p.alpha * c->p.alpha);
    fa.kmax2_trunc = -1;
    if (c->p.truncate_spherical) {
        double km = 1e300;
        for (int d = 0; d < 3; d++) km = std::fmin(km, 2 * M_PI * ((c->p.Ns[d] - 1) / 2) / c->p.Ls[d]);
        fa.kmax2_trunc = km * km;  // params.jl:161-166
    }
    fa.do_vel = fa.do_psi = 0;
    fa.uhat = (CT *)c->uhat;
    fa.keep_uhat = 0;
    fa.nkz = c->nkz;
    fa.ucstride = c->uhat_stride;
    return fa;
}

LRGeom lr_geom(const vpbs_ctx *c) {
    LRGeom g;
    for (int d = 0; d < 3; d++) {
        g.G[d] = c->G[d];
        g.scale[d] = (double)c->G[d] / c->p.Ls[d];
        g.ntile[d] = c->ntile[d];
    }
    g.M = c->p.nufft_m;
    g.cstride = c->comp_stride;
    return g;
}

// Inverse transforms of z-pencils zp into the real grid (z, y, x passes with the
// pencil transposes between them).
template <typename CT>
int inverse_to_grid(vpbs_ctx *c, Cx<CT> *zp) {
    if (c->fft_fused) return spectral_inverse(c, zp);
    hipStream_t s = c->s_lr;
    const int G0 = c->G[0], G1 = c->G[1], G2 = c->G[2];
    const int nkx = c->nkx, nky = c->nky, K1 = c->kmax_mode[1];
    Cx<CT> *rows = (Cx<CT> *)c->grid;
    Cx<CT> *ypen = (Cx<CT> *)c->ypen;
    auto fft = [&](int dim, void *buf) -> int {
        void *io[1] = {buf};
        if (rocfft_execute(c->plan[dim][1], io, nullptr, c->fft_info) != rocfft_status_success)
            return fail(c, VPBS_ERR_FFT, "rocfft_execute failed (dimension %d, inverse)", dim);
        return VPBS_OK;
    };
    VPBS_TRY(fft(2, zp));
    zpencils_to_ypencils<CT><<<dim3(G2 / 32, G1 / 32, 3 * nkx), 256, 0, s>>>(zp, ypen, G1, G2, nky, K1);
    VPBS_TRY(fft(1, ypen));
    ypencils_to_pair_rows<CT><<<dim3(G0 / 32, G1 / 32, 3 * G2), 256, 0, s>>>(ypen, rows, G0, G1, G2, nkx);
    VPBS_TRY(fft(0, rows));
    VPBS_HIP(c, hipGetLastError());
    return VPBS_OK;
}

// Node buffers of the slab interpolation, grown with Np (its partial sums alone take up to 1.9 KB a node).
// fit = false: the GPU has no memory for them, and the interpolation goes through the real grid, which
// needs none.
int slab_node_buffers(vpbs_ctx *c, bool &fit) {
    const int64_t Np = c->Np;
    fit = true;
    if (Np <= c->cap_nd) return VPBS_OK;
    c->cap_nd = 0;  // until all of them are there
    const size_t es = c->p.precision == VPBS_F32 ? sizeof(float) : sizeof(double), i4 = sizeof(int32_t);
    const struct {
        void **p;
        size_t bytes;  // per node
    } bufs[] = {{(void **)&c->nd_key, i4},
                {(void **)&c->nd_perm, i4},
                {(void **)&c->nd_i0, 3 * i4},
                {(void **)&c->nd_node, i4},
                {&c->nd_rec, es * (size_t)slab_rec_len(2 * c->p.nufft_m, (int)es)},
                {&c->slab_part, es * 3 * (size_t)spectral_slab_slots(c)}};
    auto drop = [&]() -> int {
        for (const auto &b : bufs)
            if (*b.p) {
                VPBS_HIP(c, hipFree(*b.p));
                *b.p = nullptr;
            }
        return VPBS_OK;
    };
    VPBS_TRY(drop());
    for (const auto &b : bufs) {
        const hipError_t e = hipMalloc(b.p, b.bytes * (size_t)Np);
        if (e == hipErrorOutOfMemory) {
            (void)hipGetLastError();  // handled here
            *b.p = nullptr;
            fit = false;
            return drop();
        }
        VPBS_HIP(c, e);
    }
    c->cap_nd = Np;
    return VPBS_OK;
}

template <typename CT>
int launch_lr(vpbs_ctx *c, uint32_t flags) {
    hipStream_t s = c->s_lr;
    const int64_t Np = c->Np, Nq = c->Nq;
    const bool vel = flags & VPBS_VELOCITY, psi = flags & VPBS_STREAMFUNCTION;
    const LRGeom g = lr_geom(c);
    const CT beta = (CT)c->es_beta;

    stage_begin(c, ST_LRSORT, s);
    bool slab = c->slab_interp;
    if (slab) VPBS_TRY(slab_node_buffers(c, slab));
    BinList lists[2] = {
        {BIN_TILE, Nq, c->ntiles, c->points, c->lr_key, c->lr_start, c->lr_perm, nullptr, true},
        {BIN_SLAB, Np, c->nslabs, c->nodes, c->nd_key, c->nd_start, c->nd_perm, nullptr, true},
    };
    VPBS_TRY(bin_lists(c, c->sort_lr, lists, slab ? 2 : 1, s));
    GatherArgs<CT> ga{g, beta, Nq, Np, nblocks(Nq, 256), c->lr_key, c->lr_start, c->lr_perm, lists[0].rank, c->nd_key,
                      c->nd_start, c->nd_perm, lists[1].rank, c->points, c->charges, c->nodes, c->lr_i0, c->nd_i0,
                      c->nd_node, (CT *)c->lr_w, (CT *)c->nd_rec};
    launch_gather<CT>(ga, ga.point_blocks + (slab ? nblocks(Np, 256) : 0), s);
    stage_end(c, ST_LRSORT, s);

    CT *grid = (CT *)c->grid;
    stage_begin(c, ST_SPREAD, s);
    launch_spread<CT>(g, c->ntiles, Nq, c->lr_start, c->lr_i0, (const CT *)c->lr_w, grid, s);
    stage_end(c, ST_SPREAD, s);
    VPBS_HIP(c, hipGetLastError());

    if (c->fft_fused) {
        stage_begin(c, ST_FFTF, s);
        VPBS_TRY(spectral_forward(c));
        stage_end(c, ST_FFTF, s);
        stage_begin(c, ST_FOURIER, s);
        VPBS_TRY(spectral_fourier(c, flags));
        stage_end(c, ST_FOURIER, s);
        // inverse transforms to the nodes: with slab interpolation the inverse x transform
        // runs inside the interpolation kernel (the real grid is not written)
        stage_begin(c, ST_FFTB, s);
        if (vel) VPBS_TRY(slab ? spectral_y_inverse(c, c->zpen) : spectral_inverse(c, c->zpen));
        stage_end(c, ST_FFTB, s);
        stage_begin(c, ST_INTERP, s);
        if (vel) {
            if (slab)
                VPBS_TRY(spectral_x_inverse_interp(c, c->v_lr));
            else
                launch_interp<CT>(g, Np, c->nodes, beta, grid, c->v_lr, s);
        }
        if (psi) {
            if (slab) {
                VPBS_TRY(spectral_y_inverse(c, c->zpen2));
                VPBS_TRY(spectral_x_inverse_interp(c, c->psi_lr));
            } else {
                VPBS_TRY(spectral_inverse(c, c->zpen2));
                launch_interp<CT>(g, Np, c->nodes, beta, grid, c->psi_lr, s);
            }
        }
        stage_end(c, ST_INTERP, s);
        VPBS_HIP(c, hipGetLastError());
        return VPBS_OK;
    }

    const int G0 = c->G[0], G1 = c->G[1], G2 = c->G[2];
    const int nkx = c->nkx, nky = c->nky, K1 = c->kmax_mode[1];
    Cx<CT> *rows = (Cx<CT> *)c->grid;
    Cx<CT> *ypen = (Cx<CT> *)c->ypen;
    auto fft = [&](int dim, int dir, void *buf) -> int {
        void *io[1] = {buf};
        if (rocfft_execute(c->plan[dim][dir], io, nullptr, c->fft_info) != rocfft_status_success)
            return fail(c, VPBS_ERR_FFT, "rocfft_execute failed (dimension %d, %s)", dim,
                        dir ? "inverse" : "forward");
        return VPBS_OK;
    };
    auto inverse = [&](Cx<CT> *zp) -> int { return inverse_to_grid<CT>(c, zp); };

    stage_begin(c, ST_FFTF, s);
    Cx<CT> *zpen = (Cx<CT> *)c->zpen;
    VPBS_TRY(fft(0, 0, rows));
    pair_split_to_ypencils<CT><<<dim3((nkx + 31) / 32, G1 / 32, 3 * G2), 256, 0, s>>>(rows, ypen, G0, G1, G2, nkx);
    VPBS_TRY(fft(1, 0, ypen));
    ypencils_to_zpencils<CT><<<dim3(G2 / 32, (nky + 31) / 32, 3 * nkx), 256, 0, s>>>(ypen, zpen, G1, G2, nky, K1);
    VPBS_TRY(fft(2, 0, zpen));
    stage_end(c, ST_FFTF, s);
    VPBS_HIP(c, hipGetLastError());

    FourierArgs<CT> fa = fourier_args<CT>(c);
    fa.do_vel = vel;
    fa.do_psi = psi;
    fa.keep_uhat = (flags & VPBS_KEEP_UHAT) ? 1 : 0;
    Cx<CT> *zpen2 = psi ? (Cx<CT> *)c->zpen2 : zpen;
    stage_begin(c, ST_FOURIER, s);
    fourier_kernel<CT><<<nblocks(fa.cstride, 256), 256, 0, s>>>(fa, (CT *)zpen, (CT *)zpen2);
    stage_end(c, ST_FOURIER, s);
    VPBS_HIP(c, hipGetLastError());

    // velocity: z-pencils -> real grid -> nodes; then the streamfunction reuses the grid
    stage_begin(c, ST_FFTB, s);
    if (vel) VPBS_TRY(inverse(zpen));
    stage_end(c, ST_FFTB, s);
    stage_begin(c, ST_INTERP, s);
    if (vel) launch_interp<CT>(g, Np, c->nodes, beta, grid, c->v_lr, s);
    if (psi) {
        VPBS_TRY(inverse(zpen2));
        launch_interp<CT>(g, Np, c->nodes, beta, grid, c->psi_lr, s);
    }
    stage_end(c, ST_INTERP, s);
    VPBS_HIP(c, hipGetLastError());
    return VPBS_OK;
}

bool rocfft_ok(rocfft_status st) { return st == rocfft_status_success; }

}  // namespace

double es_beta(int m, double sigma) { return 0.98 * M_PI * m * (2.0 - 1.0 / sigma); }

int oversampled_size(int N, double sigma) {
    // smallest multiple of 32 with no prime factor above 5, ≥ ⌈σN⌉
    int n = (int)std::ceil(sigma * N - 1e-9);
    for (;; n++) {
        if (n % 32) continue;
        int r = n;
        for (int p : {2, 3, 5})
            while (r % p == 0) r /= p;
        if (r == 1) return n;
    }
}

// Device address of `scratch` on the context's GPU (current here), taken once per device.
int scratch_address(vpbs_ctx *c) {
    if (c->device < 0 || c->device >= MAX_DEVICES)
        return fail(c, VPBS_ERR_INVALID, "device %d: at most %d devices", c->device, MAX_DEVICES);
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_ptr[c->device]) {
        void *ptr = nullptr;
        VPBS_HIP(c, hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
        g_scratch_ptr[c->device] = (double *)ptr;
    }
    c->spec_scratch = g_scratch_ptr[c->device];
    return VPBS_OK;
}

int longrange_setup(vpbs_ctx *c) {
    const int m = c->p.nufft_m;
    VPBS_TRY(scratch_address(c));
    for (int d = 0; d < 3; d++) {
        c->G[d] = oversampled_size(c->p.Ns[d], c->p.nufft_sigma);
        if (c->G[d] < 4 * m) c->G[d] = ((4 * m + 31) / 32) * 32;
        c->ntile[d] = c->G[d] / (d == 0 ? TX : (d == 1 ? TY : TZ));
    }
    c->ntiles = (int64_t)c->ntile[0] * c->ntile[1] * c->ntile[2];
    c->nslabs = (int64_t)(c->G[1] / SLAB_HY) * (c->G[2] / slab_hz(c->p.precision == VPBS_F32 ? 4 : 8, c->G[0]));
    c->comp_stride = (int64_t)c->G[0] * c->G[1] * c->G[2];
    c->es_beta = es_beta(m, c->p.nufft_sigma);
    // retained modes (longrange.jl:556-583)
    c->kmax_mode[0] = c->p.Ns[0] / 2 - 1;
    for (int d = 1; d < 3; d++)
        c->kmax_mode[d] = (c->p.Ns[d] % 2 == 0) ? c->p.Ns[d] / 2 - 1 : (c->p.Ns[d] - 1) / 2;
    c->nkx = c->kmax_mode[0] + 1;
    c->nky = 2 * c->kmax_mode[1] + 1;
    c->ypen_stride = (int64_t)c->nkx * c->G[2] * c->G[1];
    c->zpen_stride = (int64_t)c->nkx * c->nky * c->G[2];
    c->nkz = 2 * c->kmax_mode[2] + 1;
    c->uhat_stride = (int64_t)c->nkx * c->nky * c->nkz;

    // deconvolution tables 1/ψ̂(k)
    std::vector<double> gx, gw;
    gauss_legendre01(128, gx, gw);
    std::vector<double> tab;
    for (int k = 0; k <= c->kmax_mode[0]; k++) tab.push_back(1.0 / es_fourier(k, c->G[0], m, c->es_beta, gx, gw));
    for (int d = 1; d < 3; d++)
        for (int k = -c->kmax_mode[d]; k <= c->kmax_mode[d]; k++)
            tab.push_back(1.0 / es_fourier(k, c->G[d], m, c->es_beta, gx, gw));
    VPBS_HIP(c, hipMalloc((void **)&c->deconv, sizeof(double) * tab.size()));
    VPBS_HIP(c, hipMemcpy(c->deconv, tab.data(), sizeof(double) * tab.size(), hipMemcpyHostToDevice));

    const size_t es = c->p.precision == VPBS_F32 ? sizeof(float) : sizeof(double);
    VPBS_HIP(c, hipMalloc(&c->grid, es * 3 * (size_t)c->comp_stride));
    VPBS_HIP(c, hipMalloc(&c->ypen, 2 * es * 3 * (size_t)c->ypen_stride));
    VPBS_HIP(c, hipMalloc(&c->zpen, 2 * es * 3 * (size_t)c->zpen_stride));

    c->fft_fused = (c->p.fft == VPBS_FFT_FUSED || c->p.fft == VPBS_FFT_SEPARATE) && spectral_supported(c);
    c->slab_interp = false;
    if (c->fft_fused) {
        VPBS_TRY(spectral_setup(c));
        c->slab_interp = spectral_slab_supported(c);
        c->plans_ready = true;
        return VPBS_OK;
    }

    // rocFFT: in-place batched contiguous c2c along each direction
    const rocfft_precision prec = c->p.precision == VPBS_F32 ? rocfft_precision_single : rocfft_precision_double;
    const size_t len[3] = {(size_t)c->G[0], (size_t)c->G[1], (size_t)c->G[2]};
    const size_t batch[3] = {3 * (size_t)c->G[2] * (c->G[1] / 2), 3 * (size_t)c->nkx * c->G[2],
                             3 * (size_t)c->nkx * c->nky};
    c->fft_work_size = 0;
    for (int d = 0; d < 3; d++) {
        for (int dir = 0; dir < 2; dir++) {
            rocfft_plan_description desc = nullptr;
            if (!rocfft_ok(rocfft_plan_description_create(&desc)))
                return fail(c, VPBS_ERR_FFT, "rocfft_plan_description_create failed");
            const size_t stride[1] = {1};
            const bool ok =
                rocfft_ok(rocfft_plan_description_set_data_layout(
                    desc, rocfft_array_type_complex_interleaved, rocfft_array_type_complex_interleaved, nullptr,
                    nullptr, 1, stride, len[d], 1, stride, len[d])) &&
                rocfft_ok(rocfft_plan_create(&c->plan[d][dir], rocfft_placement_inplace,
                                             dir ? rocfft_transform_type_complex_inverse
                                                 : rocfft_transform_type_complex_forward,
                                             prec, 1, &len[d], batch[d], desc));
            rocfft_plan_description_destroy(desc);
            if (!ok) return fail(c, VPBS_ERR_FFT, "rocfft_plan_create failed (length %zu, batch %zu)", len[d], batch[d]);
            size_t w = 0;
            rocfft_plan_get_work_buffer_size(c->plan[d][dir], &w);
            c->fft_work_size = std::max(c->fft_work_size, w);
        }
    }
    if (c->fft_work_size) VPBS_HIP(c, hipMalloc(&c->fft_work, c->fft_work_size));
    if (!rocfft_ok(rocfft_execution_info_create(&c->fft_info)))
        return fail(c, VPBS_ERR_FFT, "rocfft_execution_info_create failed");
    rocfft_execution_info_set_stream(c->fft_info, c->s_lr);
    if (c->fft_work_size) rocfft_execution_info_set_work_buffer(c->fft_info, c->fft_work, c->fft_work_size);
    c->plans_ready = true;
    return VPBS_OK;
}

int longrange_compute(vpbs_ctx *c, uint32_t flags) {
    const bool psi = flags & VPBS_STREAMFUNCTION;
    const size_t es = c->p.precision == VPBS_F32 ? sizeof(float) : sizeof(double);
    if (psi && !c->zpen2) VPBS_HIP(c, hipMalloc(&c->zpen2, 2 * es * 3 * (size_t)c->zpen_stride));
    const bool keep = flags & VPBS_KEEP_UHAT;
    if (keep && !c->uhat) VPBS_HIP(c, hipMalloc(&c->uhat, 2 * es * 3 * (size_t)c->uhat_stride));
    c->uhat_quantity = 0;
    const int rc = c->p.precision == VPBS_F32 ? launch_lr<float>(c, flags) : launch_lr<double>(c, flags);
    if (rc == VPBS_OK && keep) {
        c->uhat_quantity = (flags & VPBS_VELOCITY) ? VPBS_UHAT_VELOCITY : VPBS_UHAT_STREAMFUNCTION;
        c->uhat_version = c->points_version;
    }
    return rc;
}

namespace {

// Kept field on kmin² ≤ k² ≤ kmax² (weighted by e^{−cf·k²} − e^{−cc·k²} when cf > 0) on the
// real grid.
template <typename CT>
int band_grid(vpbs_ctx *c, double kmin2, double kmax2, double cf, double cc) {
    hipStream_t s = c->s_lr;
    if (c->fft_fused) {
        VPBS_TRY(spectral_band(c, kmin2, kmax2, cf, cc));
    } else {
        FourierArgs<CT> fa = fourier_args<CT>(c);
        band_to_zpencils<CT><<<nblocks(fa.cstride, 256), 256, 0, s>>>(fa, kmin2, kmax2, cf, cc, (CT *)c->zpen);
        VPBS_HIP(c, hipGetLastError());
        VPBS_TRY(inverse_to_grid<CT>(c, (Cx<CT> *)c->zpen));
    }
    return VPBS_OK;
}

template <typename CT>
int band_impl(vpbs_ctx *c, double kmin, double kmax, double *v_out) {
    hipStream_t s = c->s_lr;
    VPBS_TRY(band_grid<CT>(c, kmin * kmin, kmax * kmax, 0.0, 0.0));
    launch_interp<CT>(lr_geom(c), c->Np, c->nodes, (CT)c->es_beta, (const CT *)c->grid, c->v_lr, s);
    VPBS_HIP(c, hipGetLastError());
    VPBS_HIP(c, hipMemcpyAsync(v_out, c->v_lr, sizeof(double) * 3 * (size_t)c->Np, hipMemcpyDeviceToHost, s));
    VPBS_HIP(c, hipStreamSynchronize(s));
    return VPBS_OK;
}

// Partial spectra of nb blocks into partial [nb][nk], their sum into out [nk].
template <typename CT>
void launch_spectrum(vpbs_ctx *c, int nk, double dk, int nb, double *partial, double *out, hipStream_t s) {
    spectrum_partial<CT><<<nb, 256, sizeof(double) * nk, s>>>(
        (const CT *)c->uhat, c->uhat_stride, c->nkx, c->nkz, c->kmax_mode[1], c->kmax_mode[2], 2 * M_PI / c->p.Ls[0],
        2 * M_PI / c->p.Ls[1], 2 * M_PI / c->p.Ls[2], 1.0 / dk, nk, c->uhat_quantity == VPBS_UHAT_STREAMFUNCTION,
        partial);
    spectrum_reduce<<<nblocks(nk, SPEC_RB), SPEC_RB * SPEC_RT, 0, s>>>(partial, nb, nk, out);
}

template <typename CT>
int spectrum_impl(vpbs_ctx *c, int nk, double dk, double *Ek) {
    hipStream_t s = c->s_lr;
    const int nb = 1024;
    const int64_t need = (int64_t)nb * nk + nk;
    if (need > c->cap_spec) {
        if (c->spec_part) VPBS_HIP(c, hipFree(c->spec_part));
        c->spec_part = nullptr;
        c->cap_spec = 0;
        VPBS_HIP(c, hipMalloc((void **)&c->spec_part, sizeof(double) * (size_t)need));
        c->cap_spec = need;
    }
    double *partial = c->spec_part, *out = partial + (size_t)nb * nk;
    launch_spectrum<CT>(c, nk, dk, nb, partial, out, s);
    VPBS_HIP(c, hipGetLastError());
    VPBS_HIP(c, hipMemcpyAsync(Ek, out, sizeof(double) * nk, hipMemcpyDeviceToHost, s));
    VPBS_HIP(c, hipStreamSynchronize(s));
    return VPBS_OK;
}

// The same with the partial spectra and the sum in the GPU's `scratch` array (nk ≤
// SPEC_NA_MAXBINS): no allocation. Every partial bin and every output bin is written by the
// kernels before it is read, so nothing left by an earlier call is used.
template <typename CT>
int spectrum_noalloc_impl(vpbs_ctx *c, int nk, double dk, double *Ek) {
    hipStream_t s = c->s_lr;
    double *partial = c->spec_scratch, *out = partial + (size_t)SPEC_NA_BLOCKS * nk;
    launch_spectrum<CT>(c, nk, dk, SPEC_NA_BLOCKS, partial, out, s);
    VPBS_HIP(c, hipGetLastError());
    VPBS_HIP(c, hipMemcpyAsync(Ek, out, sizeof(double) * nk, hipMemcpyDefault, s));
    VPBS_HIP(c, hipStreamSynchronize(s));
    return VPBS_OK;
}

template <typename CT>
int get_uhat_impl(vpbs_ctx *c, double *out) {
    const int64_t n = 3 * c->uhat_stride;
    std::vector<CT> h(2 * (size_t)n);
    VPBS_HIP(c, hipMemcpy(h.data(), c->uhat, sizeof(CT) * 2 * (size_t)n, hipMemcpyDeviceToHost));
    const int64_t Nkx = c->p.Ns[0] / 2 + 1, N1 = c->p.Ns[1], N2 = c->p.Ns[2];
    const int64_t K = Nkx * N1 * N2;
    std::fill(out, out + 2 * 3 * K, 0.0);
    const int K1 = c->kmax_mode[1], K2 = c->kmax_mode[2];
    for (int d = 0; d < 3; d++)
        for (int kx = 0; kx < c->nkx; kx++)
            for (int j = 0; j < c->nky; j++) {
                const int ky = j <= K1 ? j : j - c->nky;
                const int64_t iy = ky >= 0 ? ky : ky + N1;
                for (int jz = 0; jz < c->nkz; jz++) {
                    const int kz = jz <= K2 ? jz : jz - c->nkz;
                    const int64_t iz = kz >= 0 ? kz : kz + N2;
                    const int64_t src = d * c->uhat_stride + ((int64_t)j * c->nkz + jz) * c->nkx + kx;
                    const int64_t dst = d * K + (iz * N1 + iy) * Nkx + kx;
                    out[2 * dst] = (double)h[2 * src];
                    out[2 * dst + 1] = (double)h[2 * src + 1];
                }
            }
    return VPBS_OK;
}

}  // namespace

int longrange_get_uhat(vpbs_ctx *c, int32_t *quantity, int64_t *dims3, double *out) {
    if (quantity) *quantity = c->uhat_quantity;
    if (dims3) {
        dims3[0] = c->p.Ns[0] / 2 + 1;
        dims3[1] = c->p.Ns[1];
        dims3[2] = c->p.Ns[2];
    }
    if (!out) return VPBS_OK;
    if (!c->uhat_quantity)
        return fail(c, VPBS_ERR_STATE, "no Fourier field kept: run vpbs_compute with VPBS_KEEP_UHAT (and the long range)");
    return c->p.precision == VPBS_F32 ? get_uhat_impl<float>(c, out) : get_uhat_impl<double>(c, out);
}

int longrange_spectrum(vpbs_ctx *c, int64_t nk, double dk, double *Ek) {
    if (c->uhat_quantity != VPBS_UHAT_VELOCITY && c->uhat_quantity != VPBS_UHAT_STREAMFUNCTION)
        return fail(c, VPBS_ERR_STATE, "no Fourier field kept: run vpbs_compute with VPBS_KEEP_UHAT (and the long range)");
    if (nk < 1 || nk > 8192) return fail(c, VPBS_ERR_INVALID, "spectrum length must be in [1, 8192] (got %lld)", (long long)nk);
    if (!(dk > 0) || !std::isfinite(dk)) return fail(c, VPBS_ERR_INVALID, "wavenumber step must be positive");
    if (!Ek) return fail(c, VPBS_ERR_INVALID, "null output");
    return c->p.precision == VPBS_F32 ? spectrum_impl<float>(c, (int)nk, dk, Ek) : spectrum_impl<double>(c, (int)nk, dk, Ek);
}

int longrange_spectrum_noalloc(vpbs_ctx *c, int64_t nk, double dk, double *Ek) {
    if (c->uhat_quantity != VPBS_UHAT_VELOCITY && c->uhat_quantity != VPBS_UHAT_STREAMFUNCTION)
        return fail(c, VPBS_ERR_STATE, "no Fourier field kept: run vpbs_compute with VPBS_KEEP_UHAT (and the long range)");
    if (nk < 1 || nk > SPEC_NA_MAXBINS)
        return fail(c, VPBS_ERR_INVALID, "spectrum length must be in [1, %d] without allocation (got %lld)",
                    SPEC_NA_MAXBINS, (long long)nk);
    if (!(dk > 0) || !std::isfinite(dk)) return fail(c, VPBS_ERR_INVALID, "wavenumber step must be positive");
    if (!Ek) return fail(c, VPBS_ERR_INVALID, "null output");
    if (!c->spec_scratch) return fail(c, VPBS_ERR_STATE, "scratch address of this GPU not taken");
    return c->p.precision == VPBS_F32 ? spectrum_noalloc_impl<float>(c, (int)nk, dk, Ek)
                                      : spectrum_noalloc_impl<double>(c, (int)nk, dk, Ek);
}

int longrange_band(vpbs_ctx *c, double kmin, double kmax, double *v_out) {
    if (!c->uhat_quantity)
        return fail(c, VPBS_ERR_STATE, "no Fourier field kept: run vpbs_compute with VPBS_KEEP_UHAT (and the long range)");
    if (!(kmin >= 0) || !(kmax >= kmin)) return fail(c, VPBS_ERR_INVALID, "expected 0 <= kmin <= kmax");
    if (!v_out) return fail(c, VPBS_ERR_INVALID, "null output");
    return c->p.precision == VPBS_F32 ? band_impl<float>(c, kmin, kmax, v_out) : band_impl<double>(c, kmin, kmax, v_out);
}

int longrange_filtered_grid(vpbs_ctx *c, double cf, double cc) {
    if (!c->uhat_quantity)
        return fail(c, VPBS_ERR_STATE, "no Fourier field kept: run vpbs_compute with VPBS_KEEP_UHAT (and the long range)");
    const double inf = HUGE_VAL;
    return c->p.precision == VPBS_F32 ? band_grid<float>(c, 0.0, inf, cf, cc) : band_grid<double>(c, 0.0, inf, cf, cc);
}

int longrange_interp_at(vpbs_ctx *c, int64_t n, const double *pos, double *out) {
    if (n <= 0) return VPBS_OK;
    if (c->p.precision == VPBS_F32)
        launch_interp<float>(lr_geom(c), n, pos, (float)c->es_beta, (const float *)c->grid, out, c->s_lr);
    else
        launch_interp<double>(lr_geom(c), n, pos, c->es_beta, (const double *)c->grid, out, c->s_lr);
    VPBS_HIP(c, hipGetLastError());
    return VPBS_OK;
}

void longrange_release(vpbs_ctx *c) {
    spectral_release(c);
    for (auto &pd : c->plan)
        for (auto &p : pd) {
            if (p) rocfft_plan_destroy(p);
            p = nullptr;
        }
    if (c->fft_info) rocfft_execution_info_destroy(c->fft_info);
    c->fft_info = nullptr;
    void *bufs[] = {c->fft_work, c->grid, c->ypen, c->zpen, c->zpen2, c->deconv, c->uhat};
    for (void *b : bufs)
        if (b) (void)hipFree(b);
    c->fft_work = c->grid = c->ypen = c->zpen = c->zpen2 = c->uhat = nullptr;
    c->deconv = nullptr;
}

int merge_outputs(vpbs_ctx *c, const double *a, const double *b, double *o, int64_t n, hipStream_t s) {
    add3<<<nblocks(n, 256), 256, 0, s>>>(n, a, b, o);
    VPBS_HIP(c, hipGetLastError());
    return VPBS_OK;
}

}  // namespace vpbs
