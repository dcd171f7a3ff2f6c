// Inverse x transform fused with the interpolation (type 2); instantiated per compute type by
// spectral_slab_f32.hip and spectral_slab_f64.hip.
//
// Slab = SLAB_HY y-rows × HZ z-rows × all G0 x-cells of the 3 components: 6 HZ complex columns
// b = (c·HZ + zz)·SLAB_HP + pp (pair row pp of z-row zz, component c). Each column
// is rebuilt from x1 (Z_k = A_k + i B_k, its Hermitian half, DC real) into the registers of L/E
// threads of one wavefront, transformed there (fft_reg.hpp) with exchanges through the column's
// own part of the LDS, which then takes the grid values (real part: even y, imaginary part: odd
// y): no barrier before the whole slab is there. Every node whose W³ stencil reaches the slab has
// its first stencil cell in one of NYH × NZH home slabs (nodes come sorted by home slab); one
// lane per pair row and node sums the W cells of its two rows with the x-weights and scales by
// the rows' y- and z-weights, and the sum over a node's lanes is the part of its stencil sum that
// lies in this slab. It goes to slot q of the node, q = the home-slab
// range it was found in (one slab per slot); slab_reduce adds the slots in a fixed order. No grid
// written, no atomics: deterministic.
//
// What bounds it: vector and LDS instructions of the transforms and the stencil sums in equal parts
// (FP32, 1M nodes, 768 cells: each about 70 % of the time), memory far less. Against transforms of
// the whole slab in LDS passes with barriers, and eight lanes per node, alone: 1M nodes, 768 cells
// FP32 1.88 -> 1.85 ms, FP64 4.21 -> 3.67 ms; 256k nodes, 384 cells FP32 0.37 -> 0.32 ms, FP64
// 0.75 -> 0.50 ms.
#pragma once

#include "fft_reg.hpp"

namespace vpbs {

struct SlabLaunch {
    const void *kernel = nullptr;
    int threads = 0;
    size_t lds = 0;
};

// Kernel of stencil width W on L x-cells; instantiated for W ≤ 8 and for wider stencils in files of
// their own (two of four that compile side by side).
template <typename CT, int W>
SlabLaunch slab_launch_w(int L);

namespace {

constexpr int SLAB_HP = SLAB_HY / 2;
constexpr int SLAB_LDS_MAX = 160 * 1024;
template <typename CT>
constexpr int slab_bw(int L) {
    return 3 * slab_hz((int)sizeof(CT), L) * SLAB_HP;
}
static_assert(SLAB_HP == 2, "pair row = lowest bit of a node's lane");

// Home slabs along y (z) of the nodes whose W-cell stencil reaches a slab.
constexpr int slab_nyh(int W) { return 1 + (W - 1 + SLAB_HY - 1) / SLAB_HY; }
template <typename CT>
constexpr int slab_nzh(int W, int L) {
    const int hz = slab_hz((int)sizeof(CT), L);
    return 1 + (W - 1 + hz - 1) / hz;
}

// Columns per wavefront (of at most 64 threads; longer ones follow each other), threads per block.
constexpr int slab_cols(int L) { return 64 / reg_plan(L).T; }
template <typename CT>
constexpr int slab_threads(int L) {
    const int T = reg_plan(L).T, bw = slab_bw<CT>(L);
    return T > 64 ? T * bw : 64 * ((bw + slab_cols(L) - 1) / slab_cols(L));
}
// Values between columns: room for the exchanges, and for the cells and the first W - 1 of them
// again (stencils across the periodic end read consecutive values). An odd number: columns start
// on different LDS banks.
template <typename CT, int W, int L>
constexpr int slab_pitch() {
    constexpr int a = L + W - 1, b = ColumnExchange<CT, L>::ROOM;
    return (a > b ? a : b) | 1;
}
template <typename CT, int W, int L>
constexpr size_t slab_lds() {  // columns and twiddles
    return sizeof(C2<CT>) * ((size_t)slab_bw<CT>(L) * slab_pitch<CT, W, L>() + (ColumnExchange<CT, L>::HALF ? L / 2 : L));
}
// Wavefronts per SIMD: what the LDS leaves room for, at most 6 in FP32 (80 registers), 4 or (E > 12)
// 3 in FP64 (128, 168).
template <typename CT, int W, int L>
constexpr int slab_waves() {
    const int blocks = (int)(SLAB_LDS_MAX / slab_lds<CT, W, L>());
    const int w = (blocks < 1 ? 1 : blocks) * (slab_threads<CT>(L) / 64) / 4;
    const int most = sizeof(CT) == 4 ? 6 : reg_plan(L).E > 12 ? 3 : 4;
    return w < 1 ? 1 : w > most ? most : w;
}

// Lane-to-lane move by a DPP control (every lane has a source), FP32 and FP64.
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// Sum over each group of N = 2 or 4 consecutive lanes, in every lane of the group.
template <int N, typename CT>
__device__ __forceinline__ CT sum_lanes(CT v) {
    static_assert(N == 2 || N == 4, "quad permutations");
    v += dpp_move<0xB1>(v);                      // quad_perm [1, 0, 3, 2]
    if constexpr (N == 4) v += dpp_move<0x4E>(v);  // quad_perm [2, 3, 0, 1]
    return v;
}

// i in (-n, 2n) -> i mod n
__device__ __forceinline__ int wrap1(int i, int n) {
    i += (i < 0) ? n : 0;
    i -= (i >= n) ? n : 0;
    return i;
}

struct SlabArgs {
    int G[3];
    int nkx;
    int64_t Np;
    const int32_t *start;  // start[sz·nsy + sy]: first node of home slab (sy, sz); start[nsy·nsz] = Np
    const int32_t *si0;    // [3][Np] first stencil cell per direction of the slab-sorted nodes, in [0, G_d)
    const void *rec;       // [Np][slab_rec(W)] node records (compute type)
    void *part;            // [NYH·NZH][3][Np] stencil sums per slot (compute type)
};

template <typename CT, int W, int L>
__global__ __launch_bounds__((slab_threads<CT>(L)), (slab_waves<CT, W, L>())) void x_inverse_interp(
    SlabArgs a, const C2<CT> *__restrict__ x1, const C2<CT> *__restrict__ tw) {
    constexpr int REC = slab_rec_len(W, (int)sizeof(CT));
    constexpr int NYH = slab_nyh(W), NZH = slab_nzh<CT>(W, L), NRG = NYH * NZH;
    constexpr int RB = (NRG + 63) / 64, RG = (NRG + RB - 1) / RB;  // batches of home slabs, one lane each
    constexpr int E = reg_plan(L).E, T = reg_plan(L).T, NT = slab_threads<CT>(L), PX = slab_pitch<CT, W, L>();
    constexpr int HZ = slab_hz((int)sizeof(CT), L), BW = slab_bw<CT>(L), LN = HZ * SLAB_HP;  // LN: lanes per node
    constexpr int TW = BW * PX;  // offset of the twiddles
    const int G1 = a.G[1], G2 = a.G[2];
    const int nsy = G1 / SLAB_HY, nsz = G2 / HZ;
    const int64_t nslab = (int64_t)nsy * nsz;
    const int64_t sl = xcd_remap(nslab);
    if (sl >= nslab) return;
    // slabs go in 8×8 blocks (ty fastest): the slabs in flight on one XCD share x1 rows and nodes
    const int blk = (int)(sl >> 6), in = (int)(sl & 63), nby = nsy >> 3;
    const int ty = ((blk % nby) << 3) + (in & 7), tz = ((blk / nby) << 3) + (in >> 3);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;

    // nodes: the home-slab ranges, concatenated in RB batches of at most 64 (lane r of batch h:
    // range h·RG + r)
    int s0[RB], incl[RB], len[RB], any = 0;
#pragma unroll
    for (int h = 0; h < RB; h++) {
        s0[h] = len[h] = 0;
        const int q = h * RG + lane;
        if (lane < RG && q < NRG) {
            const int sy = wrap1(ty - (NYH - 1) + q % NYH, nsy);
            const int sz = wrap1(tz - (NZH - 1) + q / NYH, nsz);
            const int key = sz * nsy + sy;
            s0[h] = a.start[key];
            len[h] = a.start[key + 1] - s0[h];
        }
        incl[h] = wave_incl_scan(len[h]);
        any |= __builtin_amdgcn_readlane(incl[h], RG - 1);  // the same in every wavefront
    }
    if (any == 0) return;

    C2<CT> *Sm = lds<CT>(0);
    constexpr int NTW = ColumnExchange<CT, L>::HALF ? L / 2 : L;
    for (int n = threadIdx.x; n < NTW; n += NT) Sm[TW + n] = tw[n];
    __syncthreads();
    constexpr int CW = slab_cols(L);
    const int sub = T > 64 ? (int)threadIdx.x : lane;
    const int col = T > 64 ? sub / T : wave * CW + sub / T;
    if (T > 64 || (sub / T < CW && col < BW)) {
        const int j = sub % T, nkx = a.nkx;
        const int c = col / LN, zz = (col % LN) >> 1, pp = col & 1;
        const C2<CT> *src = x1 + (((int64_t)c * G2 + tz * HZ + zz) * G1 + ty * SLAB_HY + 2 * pp) * nkx;
        // Z_k for kx < nkx, its mirror image for L - k < nkx; modes between are not retained. Every
        // load is in flight before the first is used (clamped index, zeroed after); the middle
        // third of the rows holds no retained mode at oversampling factors from 1.5
        C2<CT> v[E], A[E], B[E];
        auto middle = [](int n) { return 3 * n >= E && 3 * (n + 1) <= 2 * E; };
#pragma unroll
        for (int n = 0; n < E; n++)
            if (!middle(n)) {
                const int k = j + T * n, kk = min(2 * n >= E ? L - k : k, nkx - 1);
                A[n] = src[kk];
                B[n] = src[kk + nkx];
            }
        auto value = [&](int n) {
            const int k = j + T * n, kk = 2 * n >= E ? L - k : k;
            if (kk == 0) A[n].im = B[n].im = (CT)0;
            C2<CT> z = 2 * n >= E ? C2<CT>{A[n].re + B[n].im, B[n].re - A[n].im}
                                  : C2<CT>{A[n].re - B[n].im, A[n].im + B[n].re};
            if (kk >= nkx) z = C2<CT>{(CT)0, (CT)0};
            return z;
        };
#pragma unroll
        for (int n = 0; n < E; n++) {
            v[n] = C2<CT>{(CT)0, (CT)0};
            if (!middle(n)) v[n] = value(n);
        }
        if (3 * nkx > L) {
#pragma unroll
            for (int n = 0; n < E; n++)
                if (middle(n)) {
                    const int k = j + T * n, kk = min(2 * n >= E ? L - k : k, nkx - 1);
                    A[n] = src[kk];
                    B[n] = src[kk + nkx];
                    v[n] = value(n);
                }
        }
        const ColumnExchange<CT, L> x{col * PX, TW};
        reg_fft<CT, L, 1>(v, j, x);
        x.sync();
#pragma unroll
        for (int n = 0; n < E; n++) {
            Sm[col * PX + j + T * n] = v[n];
            if (T * n < W - 1 && j + T * n < W - 1) Sm[col * PX + L + j + T * n] = v[n];
        }
    }
    __syncthreads();

    // stencil sums: lane (j, r) = node j of the group, pair row pp of z-row zz, r = 2·zz + pp
    constexpr int NG = 64 / LN;  // nodes per group
    const int j = lane / LN, r = lane % LN;
    const int y = ty * SLAB_HY + 2 * (r & 1), z = tz * HZ + (r >> 1);
    const int64_t Np = a.Np;
    const int32_t *si0 = a.si0;
    const CT *rec = static_cast<const CT *>(a.rec);
    CT *part = static_cast<CT *>(a.part);
#pragma unroll
    for (int h = 0; h < RB; h++) {
        // candidate cnd of range q of the batch is node off[q] + cnd (cnd ≥ pre[q]); wavefront-uniform
        const int ncand = __builtin_amdgcn_readlane(incl[h], RG - 1);
        const int excl = incl[h] - len[h];
        const int offv = s0[h] - excl;  // lane q: node of candidate 0 of range q
        int pre[RG];
#pragma unroll
        for (int q = 0; q < RG; q++) pre[q] = __builtin_amdgcn_readlane(excl, q);
        for (int g = wave; g * NG < ncand; g += NT / 64) {
            const int cnd = g * NG + j;
            // range of the candidate: the number of later ranges starting at or before it (the
            // starts never decrease); its offset from lane q, with every lane active
            int q = 0;
#pragma unroll
            for (int t = 1; t < RG; t++) q += cnd >= pre[t] ? 1 : 0;
            const int o = __shfl(offv, q, 64);
            int sidx = 0;
            CT v[3] = {(CT)0, (CT)0, (CT)0};
            if (cnd < ncand) {
                sidx = cnd + o;
                const int ix = si0[sidx], iy = si0[Np + sidx], iz = si0[2 * Np + sidx];
                // the record's x weights (whole vectors), and its y and z weights of these rows
                constexpr int VL = 16 / sizeof(CT), NXV = (W + VL - 1) / VL;
                static_assert(NXV * VL <= REC, "x-weight vectors inside the record");
                CT wx[NXV * VL];
                const CT *rp = rec + (int64_t)sidx * REC;
                if constexpr (sizeof(CT) == 4) {
#pragma unroll
                    for (int k = 0; k < NXV; k++) {
                        const float4 u = reinterpret_cast<const float4 *>(rp)[k];
                        wx[4 * k] = u.x, wx[4 * k + 1] = u.y, wx[4 * k + 2] = u.z, wx[4 * k + 3] = u.w;
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < NXV; k++) {
                        const double2 u = reinterpret_cast<const double2 *>(rp)[k];
                        wx[2 * k] = u.x, wx[2 * k + 1] = u.y;
                    }
                }
                const int ky0 = wrap1(y - iy, G1), ky1 = ky0 + 1 == G1 ? 0 : ky0 + 1, kz = wrap1(z - iz, G2);
                if ((ky0 < W || ky1 < W) && kz < W) {
                    const CT wz = rp[2 * W + kz];
                    const CT w0 = ky0 < W ? rp[W + ky0] * wz : (CT)0, w1 = ky1 < W ? rp[W + ky1] * wz : (CT)0;
                    const C2<CT> *p = Sm + r * PX + ix;  // cells ix .. ix+W-1, the first ones again past L-1
#pragma unroll
                    for (int d = 0; d < 3; d++) {
                        CT e = (CT)0, u = (CT)0;
#pragma unroll
                        for (int k = 0; k < W; k++) {
                            const C2<CT> gv = p[LN * d * PX + k];
                            e += wx[k] * gv.re;
                            u += wx[k] * gv.im;
                        }
                        v[d] = w0 * e + w1 * u;
                    }
                }
            }
#pragma unroll
            for (int d = 0; d < 3; d++) v[d] = sum_lanes<LN>(v[d]);
            if (cnd < ncand && r == 0) {
                CT *dst = part + (int64_t)(h * RG + q) * 3 * Np + sidx;
                dst[0] = v[0];
                dst[Np] = v[1];
                dst[2 * Np] = v[2];
            }
        }
    }
}

// out[c][perm[s]] = Σ_q part[q][c][s] over the nslot slots, in slot order. One thread per value (c in
// grid.y) with twelve loads in flight: a thread that walked all slots of all components waited for
// each load (64 nodes: 17.5 -> 4.6 µs; 1M nodes FP32 80 -> 54 µs).
template <typename CT>
__global__ void slab_reduce(int64_t Np, int nslot, const CT *__restrict__ part, const int32_t *__restrict__ perm,
                            double *__restrict__ out) {
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= Np) return;
    const int c = blockIdx.y;
    const CT *p = part + c * Np + s;
    const int64_t i = perm[s];
    constexpr int U = 12;
    double acc = 0;
    for (int q = 0; q < nslot; q += U) {
        CT v[U];
#pragma unroll
        for (int k = 0; k < U; k++) v[k] = p[(int64_t)min(q + k, nslot - 1) * 3 * Np];
#pragma unroll
        for (int k = 0; k < U; k++) acc += q + k < nslot ? (double)v[k] : 0.0;
    }
    out[c * Np + i] = acc;
}

// The compiled lengths: every grid length (32·2^a·3^b·5^c) up to 768 that reg_plan covers, 1024 and 1536
// (800, 864, 1152 and 1280 cells interpolate from the real grid).
#define SLAB_LENGTHS(F)                                                                             \
    F(32) F(64) F(96) F(128) F(160) F(192) F(256) F(288) F(320) F(384) F(512) F(576) F(640) F(768) \
    F(1024) F(1536)

template <typename CT, int W, int L>
SlabLaunch slab_launch_wl() {
    if constexpr (slab_lds<CT, W, L>() <= (size_t)SLAB_LDS_MAX && slab_threads<CT>(L) <= 1024)
        return {(const void *)x_inverse_interp<CT, W, L>, slab_threads<CT>(L), slab_lds<CT, W, L>()};
    else
        return {};
}

}  // namespace

template <typename CT, int W>
SlabLaunch slab_launch_w(int L) {
    switch (L) {
#define SLAB_CASE(len) \
    case len: return slab_launch_wl<CT, W, len>();
        SLAB_LENGTHS(SLAB_CASE)
#undef SLAB_CASE
        default: return {};
    }
}

namespace {

template <typename CT>
SlabLaunch slab_launch(int W, int L) {
    switch (W) {
        case 4: return slab_launch_w<CT, 4>(L);
        case 6: return slab_launch_w<CT, 6>(L);
        case 8: return slab_launch_w<CT, 8>(L);
        case 10: return slab_launch_w<CT, 10>(L);
        case 12: return slab_launch_w<CT, 12>(L);
        case 14: return slab_launch_w<CT, 14>(L);
        case 16: return slab_launch_w<CT, 16>(L);
        default: return {};
    }
}

}  // namespace

template <typename CT>
size_t SlabKernels<CT>::lds_bytes(int W, int L) {
    return slab_launch<CT>(W, L).lds;
}

template <typename CT>
int SlabKernels<CT>::slots(int W, int L) {
    return slab_nyh(W) * slab_nzh<CT>(W, L);
}

template <typename CT>
bool SlabKernels<CT>::fits(int W, int L, int G1, int G2) {
    // whole 8×8 blocks of slabs, and no home slab counted twice
    const int hz = slab_hz((int)sizeof(CT), L);
    return G1 % (8 * SLAB_HY) == 0 && G2 % (8 * hz) == 0 && G1 / SLAB_HY >= slab_nyh(W) && G2 / hz >= slab_nzh<CT>(W, L);
}

template <typename CT>
hipError_t SlabKernels<CT>::setup(int W, int L) {
    const SlabLaunch k = slab_launch<CT>(W, L);
    return hipFuncSetAttribute(k.kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)k.lds);
}

template <typename CT>
hipError_t SlabKernels<CT>::run(vpbs_ctx *c, double *out) {
    const int W = 2 * c->p.nufft_m, L = c->G[0];
    SlabArgs a{};
    for (int d = 0; d < 3; d++) a.G[d] = c->G[d];
    a.nkx = c->nkx;
    a.Np = c->Np;
    a.start = c->nd_start;
    a.si0 = c->nd_i0;
    a.rec = c->nd_rec;
    a.part = c->slab_part;
    const C2<CT> *x1 = (const C2<CT> *)c->ypen;
    const C2<CT> *tw = twiddles<CT>(c, 0);
    void *args[] = {(void *)&a, (void *)&x1, (void *)&tw};
    const SlabLaunch k = slab_launch<CT>(W, L);
    const hipError_t e = hipLaunchKernel(k.kernel, dim3(grid8(c->nslabs)), dim3(k.threads), args, k.lds, c->s_lr);
    if (e != hipSuccess) return e;
    slab_reduce<CT><<<dim3((unsigned)((c->Np + 255) / 256), 3), 256, 0, c->s_lr>>>(
        c->Np, slots(W, L), (const CT *)c->slab_part, c->nd_node, out);
    return hipGetLastError();
}

}  // namespace vpbs
