// Device-side point data: the work of add_point_charges!
// (src/BiotSavart/pointdata_impl.jl:121-188) on the GPU, from the filaments'
// periodic quintic splines (src/Filaments/spline/spline.jl:116-319).
//
// Inputs (uploaded by vpbs_set_filaments): node positions X, knots t_i
// (t = 0 at each filament's first node), knot periods T, end-to-end offsets
// Xoff and the B-spline coefficients c of the periodised curve
// Y(t) = X(t) - (t/T)·Xoff (spline.jl:163-193). The derivative coefficients
//   d_j = 5(c_j - c_{j-1})/(t_{j+5} - t_j),  e_j = 4(d_j - d_{j-1})/(t_{j+4} - t_j)
// (spline_derivative!, src/Filaments/spline/spline.jl:298-319) give S′ and S″
// as order-5 and order-4 splines. One thread per node then
// writes the folded node, idx_prev, s′, s″, δ± (Gauss–Legendre integral of |S′|
// over the LIA fraction of the two adjacent segments, pointdata_impl.jl:133-143)
// and the nquad quadrature points (folded) and charges w·Δt·S′(ζ) of its right
// segment (pointdata_impl.jl:173-183), in the layout of vpbs_set_points.
#include "vpbs_internal.hpp"

#include <cmath>
#include <cstring>
#include <vector>

namespace vpbs {

// No FMA contraction in this file: the point data comes out bit-identical to a
// plain IEEE evaluation of the same formulas (numpy's). This matters beyond
// rounding: a quadrature point lying exactly on a NUFFT grid plane (a ring in
// the plane z = L/2, say) selects its 2m-point ES stencil by floor(x·G/L), and
// a 1-ulp change there moves a weight φ(±1) = e^{-β} (≈ 1e-7 at m = 4) from one
// end of the stencil to the other.
#pragma clang fp contract(off)

namespace {

inline unsigned nblocks(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

struct Fil {
    const int32_t *fid;    // [Np] filament of each node
    const int64_t *off;    // [Nf] first node
    const int32_t *N;      // [Nf] nodes per filament
    const double *T;       // [Nf] knot period
    const double *Xoff;    // [3*Nf] end-to-end offset
    const double *ts;      // [Np] knots
    int64_t Np, Nf;
};

__device__ inline double knot(const Fil &f, int64_t off, int N, double T, int j) {
    int q = j / N, r = j - q * N;
    if (r < 0) {
        r += N;
        q -= 1;
    }
    return f.ts[off + r] + q * T;
}

// Non-zero order-K B-splines at t ∈ [t_i, t_{i+1}): B[r] = B_{i-K+1+r,K}(t).
template <int K>
__device__ inline void basis(const Fil &f, int64_t off, int N, double T, int i, double t, double *B) {
    double left[K], right[K];
    B[0] = 1.0;
#pragma unroll
    for (int j = 1; j < K; j++) {
        left[j] = t - knot(f, off, N, T, i + 1 - j);
        right[j] = knot(f, off, N, T, i + j) - t;
        double saved = 0.0;
#pragma unroll
        for (int r = 0; r < j; r++) {
            const double temp = B[r] / (right[r + 1] + left[j - r]);
            B[r] = saved + right[r + 1] * temp;
            saved = left[j - r] * temp;
        }
        B[j] = saved;
    }
}

// S^(deriv)(t) on segment `seg` at local coordinate ζ, coefficient array `co`
// (c for deriv 0, d for 1, e for 2), with the periodisation undone.
template <int DERIV>
__device__ inline void eval_spline(const Fil &f, int fi, int seg, double zeta, const double *co, double *out) {
    constexpr int K = 6 - DERIV;
    const int64_t off = f.off[fi];
    const int N = f.N[fi];
    const double T = f.T[fi];
    const double ti = knot(f, off, N, T, seg), ti1 = knot(f, off, N, T, seg + 1);
    const double t = (1 - zeta) * ti + zeta * ti1;
    double B[K];
    basis<K>(f, off, N, T, seg, t, B);
    double s[3] = {0, 0, 0};
#pragma unroll
    for (int r = 0; r < K; r++) {
        int j = seg - K + 1 + r;
        j %= N;
        j += (j < 0) ? N : 0;
        const int64_t idx = off + j;
#pragma unroll
        for (int d = 0; d < 3; d++) s[d] += B[r] * co[d * f.Np + idx];
    }
#pragma unroll
    for (int d = 0; d < 3; d++) {
        const double xo = f.Xoff[d * f.Nf + fi];
        if (DERIV == 0) s[d] += (t / T) * xo;
        if (DERIV == 1) s[d] += xo / T;
        out[d] = s[d];
    }
}

// fold_coordinates_periodic (min_distance.jl:5-20): the x < 0 loop first, so
// that a tiny negative value ends at 0, never at L. Values more than 64
// periods away are first reduced by the exact fmod (the loops alone would not
// end for |x| ≫ L); non-finite values become NaN, which the folded-range check
// after the build reports as an error.
__device__ inline double fold(double x, double L) {
    if (!isfinite(x)) return __builtin_nan("");
    if (fabs(x) > 64.0 * L) x = fmod(x, L);
    while (x < 0) x += L;
    while (x >= L) x -= L;
    return x;
}

// Spline coefficients of the first derivative (order 5) of node l of a filament.
__device__ inline void derivative_coef(const Fil &f, const double *__restrict__ c, int64_t off, int N, double T, int l,
                                       double (&out)[3]) {
    const int64_t i = off + l, ip = off + (l == 0 ? N - 1 : l - 1);
    const double den = knot(f, off, N, T, l + 5) - knot(f, off, N, T, l);
#pragma unroll
    for (int d = 0; d < 3; d++) out[d] = 5.0 * (c[d * f.Np + i] - c[d * f.Np + ip]) / den;
}

// Coefficients of both derivatives, and for filaments that were just uploaded the filament of each
// node (the last one whose first node is ≤ i). The second derivative needs the first one's
// coefficient of the previous node: computed again, with the same operations, instead of a kernel of
// its own that reads it back: one launch for three (64 nodes: 25 µs of point data kernels -> 20).
template <bool UPLOADED>
__global__ void derivative_coefs(Fil f, const double *__restrict__ c, int32_t *__restrict__ fid,
                                 double *__restrict__ dco, double *__restrict__ eco) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= f.Np) return;
    int fi;
    if constexpr (UPLOADED) {
        int64_t lo = 0, hi = f.Nf - 1;  // off[0] = 0 ≤ i
        while (lo < hi) {
            const int64_t mid = (lo + hi + 1) / 2;
            if (f.off[mid] <= i)
                lo = mid;
            else
                hi = mid - 1;
        }
        fid[i] = fi = (int)lo;
    } else {
        fi = fid[i];
    }
    const int64_t off = f.off[fi];
    const int N = f.N[fi];
    const double T = f.T[fi];
    const int l = (int)(i - off);
    double v[3], vp[3];
    derivative_coef(f, c, off, N, T, l, v);
    derivative_coef(f, c, off, N, T, l == 0 ? N - 1 : l - 1, vp);
    const double den = knot(f, off, N, T, l + 4) - knot(f, off, N, T, l);
#pragma unroll
    for (int d = 0; d < 3; d++) {
        dco[d * f.Np + i] = v[d];
        eco[d * f.Np + i] = 4.0 * (v[d] - vp[d]) / den;
    }
}

struct Quad {
    int n;                      // quadrature points per segment (1 for straight segments)
    bool straight;              // NoQuadrature: midpoint of straight segments (pointdata_impl.jl:190-219)
    double gamma;               // lia_segment_fraction (1 if unset) for straight segments
    double z[16], w[16];        // rule on [0, 1]
    double lim_m[2], lim_p[2];  // integration limits of δ⁻ (segment i-1) and δ⁺ (segment i)
};

// A flag in pinned host memory, read after the stream has been waited for.
__device__ inline void set_flag(unsigned int *flag) {
    __hip_atomic_store(flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Bound by FP64 arithmetic (spline evaluations). Blocks of 128 threads may use 210 registers; without
// the bound the compiler kept to 128, for blocks of 1024, and 56 values per thread went to scratch
// memory (256k nodes 71 -> 48 µs, 17k 27.6 -> 16.5).
__global__ __launch_bounds__(128) void point_data_kernel(
    Fil f, Quad qd, Box box, const double *__restrict__ X, const double *__restrict__ c,
    const double *__restrict__ dco, const double *__restrict__ eco, double *__restrict__ nodes,
    int32_t *__restrict__ idx_prev, double *__restrict__ sp, double *__restrict__ spp, double *__restrict__ dlm,
    double *__restrict__ dlp, double *__restrict__ pts, double *__restrict__ chg, unsigned int *__restrict__ invalid) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t Np = f.Np;
    if (i >= Np) return;
    const int fi = f.fid[i];
    const int64_t off = f.off[fi];
    const int N = f.N[fi];
    const double T = f.T[fi];
    const int l = (int)(i - off);
    const int64_t ip = l == 0 ? off + N - 1 : i - 1;
    bool ok = true;  // everything written is folded into [0, L) (false for NaN); idx_prev is by construction
    auto folded = [&](double x, int d) {
        const double y = fold(x, box.L[d]);
        ok = ok && y >= 0.0 && y < box.L[d];
        return y;
    };
    for (int d = 0; d < 3; d++) nodes[d * Np + i] = folded(X[d * Np + i], d);
    idx_prev[i] = (int32_t)ip;
    double v[3];
    eval_spline<1>(f, fi, l, 0.0, dco, v);
    for (int d = 0; d < 3; d++) sp[d * Np + i] = v[d];
    eval_spline<2>(f, fi, l, 0.0, eco, v);
    for (int d = 0; d < 3; d++) spp[d * Np + i] = v[d];
    if (qd.straight) {
        // f[i-1], f[i+1] of the periodically extended filament
        const int64_t in = l == N - 1 ? off : i + 1;
        double xi[3], xp[3], xn[3];
        for (int d = 0; d < 3; d++) {
            const double xo = f.Xoff[d * f.Nf + fi];
            xi[d] = X[d * Np + i];
            xp[d] = X[d * Np + ip] - (l == 0 ? xo : 0.0);
            xn[d] = X[d * Np + in] + (l == N - 1 ? xo : 0.0);
        }
        double am = 0, ap = 0;
        for (int d = 0; d < 3; d++) {
            am += (xi[d] - xp[d]) * (xi[d] - xp[d]);
            ap += (xn[d] - xi[d]) * (xn[d] - xi[d]);
        }
        dlm[i] = qd.gamma * sqrt(am);
        dlp[i] = qd.gamma * sqrt(ap);
        for (int d = 0; d < 3; d++) {
            pts[d * Np + i] = folded((xi[d] + xn[d]) / 2, d);
            chg[d * Np + i] = xn[d] - xi[d];
        }
        if (!ok) set_flag(invalid);
        return;
    }
    // δ⁻, δ⁺ (integrate.jl:40-61 with Quadratures.integrate over (a, b))
    for (int side = 0; side < 2; side++) {
        const int seg = side == 0 ? (l == 0 ? N - 1 : l - 1) : l;
        const double a = side == 0 ? qd.lim_m[0] : qd.lim_p[0];
        const double b = side == 0 ? qd.lim_m[1] : qd.lim_p[1];
        const double delta = b - a;
        const double dt = knot(f, off, N, T, seg + 1) - knot(f, off, N, T, seg);
        double acc = 0.0;
        for (int q = 0; q < qd.n; q++) {
            eval_spline<1>(f, fi, seg, a + delta * qd.z[q], dco, v);
            acc = acc + qd.w[q] * sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
        }
        (side == 0 ? dlm : dlp)[i] = dt * (delta * acc);
    }
    // quadrature points and charges of segment l
    const double dt = knot(f, off, N, T, l + 1) - knot(f, off, N, T, l);
    const int64_t Nq = (int64_t)qd.n * Np;
    for (int q = 0; q < qd.n; q++) {
        const int64_t j = (int64_t)qd.n * i + q;
        eval_spline<0>(f, fi, l, qd.z[q], c, v);
        for (int d = 0; d < 3; d++) pts[d * Nq + j] = folded(v[d], d);
        eval_spline<1>(f, fi, l, qd.z[q], dco, v);
        const double wq = qd.w[q] * dt;
        for (int d = 0; d < 3; d++) chg[d * Nq + j] = wq * v[d];
    }
    if (!ok) set_flag(invalid);
}

// Near-singular local integrals for lia_segment_fraction = γ
// (add_local_integrals!, local_integrals.jl:209-305): the parts of the two
// segments next to node i not covered by the LIA term, ζ ∈ [0, 1-γ] of segment
// i-1 and ζ ∈ [γ, 1] of segment i, integrated with the full Biot–Savart
// kernel and the near-singularity quadrature rule; FP64, added to the
// short-range outputs (v += Γ/4π Σ q × r/|r|³, ψ += Γ/4π Σ q/|r|).
struct LocalQuad {
    int n;
    double z[16], w[16];
    double lo[2], hi[2];
};

__global__ __launch_bounds__(128) void local_integrals_kernel(Fil f, LocalQuad lq, Box box, const double *__restrict__ c,
                                       const double *__restrict__ dco, const double *__restrict__ nodes, double pref,
                                       double *__restrict__ v, double *__restrict__ psi) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t Np = f.Np;
    if (i >= Np) return;
    const int fi = f.fid[i];
    const int64_t off = f.off[fi];
    const int N = f.N[fi];
    const double T = f.T[fi];
    const int l = (int)(i - off);
    const double x[3] = {nodes[i], nodes[Np + i], nodes[2 * Np + i]};
    double av[3] = {0, 0, 0}, ap[3] = {0, 0, 0};
    for (int side = 0; side < 2; side++) {
        const int seg = side == 0 ? (l == 0 ? N - 1 : l - 1) : l;
        const double lo = lq.lo[side], delta = lq.hi[side] - lq.lo[side];
        const double dt = (knot(f, off, N, T, seg + 1) - knot(f, off, N, T, seg)) * delta;
        for (int q = 0; q < lq.n; q++) {
            const double y = lo + delta * lq.z[q];
            double sv[3], s1[3], r[3];
            eval_spline<0>(f, fi, seg, y, c, sv);
            eval_spline<1>(f, fi, seg, y, dco, s1);
            const double wq = lq.w[q] * dt;
            for (int d = 0; d < 3; d++) {
                const double sd = fold(sv[d], box.L[d]);
                double rd = x[d] - sd;
                if (rd >= box.Lh[d]) rd -= box.L[d];
                if (rd < -box.Lh[d]) rd += box.L[d];
                r[d] = rd;
                s1[d] *= wq;
            }
            const double rinv = 1.0 / sqrt(r[0] * r[0] + r[1] * r[1] + r[2] * r[2]);
            const double rinv3 = rinv * rinv * rinv;
            av[0] += (s1[1] * r[2] - s1[2] * r[1]) * rinv3;
            av[1] += (s1[2] * r[0] - s1[0] * r[2]) * rinv3;
            av[2] += (s1[0] * r[1] - s1[1] * r[0]) * rinv3;
            for (int d = 0; d < 3; d++) ap[d] += s1[d] * rinv;
        }
    }
    for (int d = 0; d < 3; d++) {
        if (v) v[d * Np + i] += pref * av[d];
        if (psi) psi[d * Np + i] += pref * ap[d];
    }
}

// ----------------------------------------------------------------------------
// Time stepping on the device (Timestepping: SSPRK33.jl:17-39, advect.jl:20-72).

// Chordal knots of each filament: t_0 = 0, t_{i+1} = t_i + |X_{i+1} - X_i|, and the
// period T including the closing segment to X_0 + offset. One wavefront per filament: the
// lanes take 64 segments at a time, whose lengths are then added in order (the sum of a plain
// loop, bit for bit). One thread per filament waited for its loads node after node: 0.24 ms
// for 1000 filaments of 256 nodes, now 0.02.
__global__ __launch_bounds__(64) void chordal_knots(Fil f, const double *__restrict__ X, double *__restrict__ ts,
                                                    double *__restrict__ T) {
    const int64_t fi = blockIdx.x;
    const int64_t off = f.off[fi];
    const int N = f.N[fi], lane = threadIdx.x;
    const int64_t Np = f.Np;
    double acc = 0.0;
    if (lane == 0) ts[off] = 0.0;
    for (int i0 = 0; i0 < N; i0 += 64) {
        const int i = i0 + lane;
        double v = 0.0;
        if (i < N) {
            const int64_t a = off + i, b = (i == N - 1) ? off : a + 1;
            double d2 = 0.0;
            for (int d = 0; d < 3; d++) {
                const double xb = X[d * Np + b] + (i == N - 1 ? f.Xoff[d * f.Nf + fi] : 0.0);
                const double dd = xb - X[d * Np + a];
                d2 = d2 + dd * dd;
            }
            v = sqrt(d2);
        }
        const long long bits = __double_as_longlong(v);
        double mine = 0.0;  // sum up to and including this lane's segment
#pragma unroll
        for (int k = 0; k < 64; k++) {  // segments past the end add 0
            const int lo = __builtin_amdgcn_readlane((int)bits, k), hi = __builtin_amdgcn_readlane((int)(bits >> 32), k);
            acc = acc + __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
            mine = lane == k ? acc : mine;
        }
        if (i < N - 1) ts[off + i + 1] = mine;
    }
    if (lane == 0) T[fi] = acc;
}

// Coefficients c of the periodic quintic interpolant of Y(t_i) = X_i - (t_i/T)·offset
// (spline.jl:163-193). Row i of the collocation system holds B_{i-5+r,6}(t_i), r = 0..4,
// at columns (i-5+r) mod N; with unknowns shifted by 3 it is a cyclic 5-band matrix with
// the largest value on the diagonal. The band part is eliminated without pivoting
// (B-spline collocation matrices are totally positive) and the periodic corners are added
// back through the Woodbury identity with U = [e_0, e_1, e_{N-2}, e_{N-1}].
//
// spline_rows writes the rows (band[r] = buf + r·Np, r = 0..4, corners in place) and the
// three components of Y (buf + (5 + d)·Np), one thread per node. spline_solve takes one
// wavefront per filament: the elimination is a chain along the filament that every lane
// follows, with the seven right-hand sides (Y, then the columns of U) in seven lanes; rows
// come and go 64 at a time through LDS, so the chain waits for arithmetic (a division a row
// each way) and not for memory. One thread per filament doing all of it in global memory took
// 4.2 ms for 1000 filaments of 256 nodes; this takes 0.14 ms. The operations on each value are those of that plain
// elimination, in its order: equal bits, which quadrature points on NUFFT grid planes need (above).
__global__ void spline_rows(Fil f, const double *__restrict__ X, double *__restrict__ buf) {
    const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t Np = f.Np;
    if (n >= Np) return;
    const int fi = f.fid[n];
    const int64_t off = f.off[fi];
    const double T = f.T[fi], ti = f.ts[n];
    double B[6];
    basis<6>(f, off, f.N[fi], T, (int)(n - off), ti, B);
#pragma unroll
    for (int r = 0; r < 5; r++) buf[r * Np + n] = B[r];
#pragma unroll
    for (int d = 0; d < 3; d++) buf[(5 + d) * Np + n] = X[d * Np + n] - (ti / T) * f.Xoff[d * f.Nf + fi];
}

// buf: 12 arrays of Np doubles: on entry the rows and Y as above; the factors (pivot and the
// two upper diagonals) replace the first three bands, the solutions the arrays 5 to 11.
__global__ __launch_bounds__(64) void spline_solve(Fil f, double *__restrict__ buf, double *__restrict__ c) {
    constexpr int CH = 64;
    __shared__ double s_a[CH][6];  // rows: 5 band values (forward), 3 factors (backward)
    __shared__ double s_y[CH][9];  // right-hand sides, in lane order
    const int64_t fi = blockIdx.x, off = f.off[fi], Np = f.Np;
    const int N = f.N[fi], lane = threadIdx.x;
    double *const g = buf + off;
    const int col = lane < 7 ? lane : 7;  // lanes past the seventh repeat a dead column
    // periodic corners
    const double c0a = g[0], c0b = g[Np], c1 = g[1], c2 = g[4 * Np + N - 2], c3a = g[3 * Np + N - 1],
                 c3b = g[4 * Np + N - 1];

    // forward elimination (row i: band r at column i - 2 + r)
    double p1 = 1, u11 = 0, u21 = 0, p2 = 1, u12 = 0, u22 = 0;  // rows i-1 and i-2: pivot, upper diagonals
    double y1 = 0, y2 = 0;
    double nb[8];  // next chunk
    auto fetch = [&](int i) {
#pragma unroll
        for (int r = 0; r < 8; r++) nb[r] = i < N ? g[r * Np + i] : 0.0;
    };
    fetch(lane);
    for (int i0 = 0; i0 < N; i0 += CH) {
        const int i = i0 + lane, rows = min(CH, N - i0);
        s_a[lane][0] = i >= 2 ? nb[0] : 0.0;
        s_a[lane][1] = i >= 1 ? nb[1] : 0.0;
        s_a[lane][2] = nb[2];
        s_a[lane][3] = i < N - 1 ? nb[3] : 0.0;
        s_a[lane][4] = i < N - 2 ? nb[4] : 0.0;
#pragma unroll
        for (int d = 0; d < 3; d++) s_y[lane][d] = nb[5 + d];
        s_y[lane][3] = i == 0 ? 1.0 : 0.0;
        s_y[lane][4] = i == 1 ? 1.0 : 0.0;
        s_y[lane][5] = i == N - 2 ? 1.0 : 0.0;
        s_y[lane][6] = i == N - 1 ? 1.0 : 0.0;
        s_y[lane][7] = 0.0;
        __syncthreads();
        if (i0 + CH < N) fetch(i + CH);
#pragma unroll 4
        for (int r = 0; r < rows; r++) {
            const double l2 = s_a[r][0] / p2;
            const double l1 = (s_a[r][1] - l2 * u12) / p1;
            const double piv = (s_a[r][2] - l2 * u22) - l1 * u11;
            const double u1 = s_a[r][3] - l1 * u21, u2 = s_a[r][4];
            const double y = (s_y[r][col] - l2 * y2) - l1 * y1;
            p2 = p1, u12 = u11, u22 = u21, y2 = y1;
            p1 = piv, u11 = u1, u21 = u2, y1 = y;
            if (lane < 8) s_y[r][lane] = y;
            if (lane == 0) {
                s_a[r][0] = piv;
                s_a[r][1] = u1;
            }
        }
        __syncthreads();
        if (lane < rows) {
            g[i] = s_a[lane][0];
            g[Np + i] = s_a[lane][1];
            g[2 * Np + i] = s_a[lane][4];
#pragma unroll
            for (int q = 0; q < 7; q++) g[(5 + q) * Np + i] = s_y[lane][q];
        }
        __syncthreads();
    }
    // back substitution
    double x1 = 0, x2 = 0, xl1 = 0, xl2 = 0;  // rows i+1, i+2; rows N-1, N-2
    const int last = ((N - 1) / CH) * CH;
    auto fetch_back = [&](int i, double (&v)[10]) {
#pragma unroll
        for (int r = 0; r < 3; r++) v[r] = i < N ? g[r * Np + i] : 0.0;
#pragma unroll
        for (int q = 0; q < 7; q++) v[3 + q] = i < N ? g[(5 + q) * Np + i] : 0.0;
    };
    double fb[10];
    fetch_back(last + lane, fb);
    for (int i0 = last; i0 >= 0; i0 -= CH) {
        const int i = i0 + lane, rows = min(CH, N - i0);
#pragma unroll
        for (int r = 0; r < 3; r++) s_a[lane][r] = fb[r];
#pragma unroll
        for (int q = 0; q < 7; q++) s_y[lane][q] = fb[3 + q];
        s_y[lane][7] = 0.0;
        __syncthreads();
        if (i0 > 0) fetch_back(i - CH, fb);
#pragma unroll 4
        for (int r = rows - 1; r >= 0; r--) {
            const double x = ((s_y[r][col] - s_a[r][1] * x1) - s_a[r][2] * x2) / s_a[r][0];
            if (i0 + r == N - 1) xl1 = x;
            if (i0 + r == N - 2) xl2 = x;
            x2 = x1, x1 = x;
            if (lane < 8) s_y[r][lane] = x;
        }
        __syncthreads();
        if (lane < rows) {
#pragma unroll
            for (int q = 0; q < 7; q++) g[(5 + q) * Np + i] = s_y[lane][q];
        }
        __syncthreads();
    }
    // Woodbury: x = z - Z (I + Vᵀ Z)⁻¹ Vᵀ z, Vᵀ rows = the corner entries, on the rows 0, 1
    // (x1, x2), N-2 and N-1 of every column; the 4×4 system in every lane alike
    const double vt[4] = {c0a * xl2 + c0b * xl1, c1 * xl1, c2 * x1, c3a * x1 + c3b * x2};
    double M[4][4], h[4][3];
#pragma unroll
    for (int a = 0; a < 4; a++) {
#pragma unroll
        for (int b = 0; b < 4; b++) M[a][b] = (a == b ? 1.0 : 0.0) + __shfl(vt[a], 3 + b, 64);
#pragma unroll
        for (int d = 0; d < 3; d++) h[a][d] = __shfl(vt[a], d, 64);
    }
    // elimination with partial pivoting, rows exchanged (the same in every lane)
#pragma unroll
    for (int k = 0; k < 4; k++) {
#pragma unroll
        for (int r = k + 1; r < 4; r++)
            if (fabs(M[r][k]) > fabs(M[k][k])) {
#pragma unroll
                for (int b = 0; b < 4; b++) {
                    const double t = M[k][b];
                    M[k][b] = M[r][b], M[r][b] = t;
                }
#pragma unroll
                for (int d = 0; d < 3; d++) {
                    const double t = h[k][d];
                    h[k][d] = h[r][d], h[r][d] = t;
                }
            }
#pragma unroll
        for (int r = k + 1; r < 4; r++) {
            const double l = M[r][k] / M[k][k];
#pragma unroll
            for (int b = 0; b < 4; b++) M[r][b] -= l * M[k][b];
#pragma unroll
            for (int d = 0; d < 3; d++) h[r][d] -= l * h[k][d];
        }
    }
    double w[4][3];
#pragma unroll
    for (int k = 3; k >= 0; k--)
#pragma unroll
        for (int d = 0; d < 3; d++) {
            double v = h[k][d];
#pragma unroll
            for (int b = k + 1; b < 4; b++) v -= M[k][b] * w[b][d];
            w[k][d] = v / M[k][k];
        }
    // unknown m = (j + 3) mod N holds coefficient j
    for (int j = lane; j < N; j += 64) {
        int m = j + 3;
        if (m >= N) m -= N;
        double z[4];
#pragma unroll
        for (int b = 0; b < 4; b++) z[b] = g[(8 + b) * Np + m];
#pragma unroll
        for (int d = 0; d < 3; d++) {
            double v = g[(5 + d) * Np + m];
#pragma unroll
            for (int b = 0; b < 4; b++) v -= z[b] * w[b][d];
            c[d * Np + off + j] = v;
        }
    }
}

// One stage of SSPRK33 (SSPRK33.jl:17-39) on the 3·Np node coordinates x, with the velocity v
// just evaluated: x0 and vs hold the step's first nodes and the velocities combined so far.
//   stage 1: x0 = x, vs = v, x = x0 + dt·v;  stage 2: vs += v, x = x0 + dt/4·vs;
//   stage 3: x = x0 + dt·(vs + 4 v)/6
__global__ void rk_stage(int64_t n, int stage, double dt, const double *__restrict__ v, double *__restrict__ x0,
                         double *__restrict__ vs, double *__restrict__ x) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (stage == 1) {
        const double x00 = x[i], v1 = v[i];
        x0[i] = x00;
        vs[i] = v1;
        x[i] = x00 + dt * v1;
    } else if (stage == 2) {
        const double s = vs[i] + v[i];
        vs[i] = s;
        x[i] = x0[i] + (dt / 4) * s;
    } else {
        x[i] = x0[i] + dt * ((vs[i] + 4.0 * v[i]) / 6.0);
    }
}

}  // namespace

Fil filament_view(const vpbs_ctx *c) {
    Fil f;
    f.fid = c->fil_fid;
    f.off = c->fil_off;
    f.N = c->fil_n;
    f.T = c->fil_T;
    f.Xoff = c->fil_xoff;
    f.ts = c->fil_ts;
    f.Np = c->Np;
    f.Nf = c->pd_nf;
    return f;
}

// Point data from the filament state on the device (nodes, knots, periods,
// offsets, spline coefficients), with the quadrature set by vpbs_set_filaments.
int point_data_from_state(vpbs_ctx *c, bool uploaded) {
    hipStream_t s = c->s_sr;
    const Fil f = filament_view(c);
    const int64_t Np = c->Np;
    Quad qd{};
    qd.n = c->p.nquad;
    qd.straight = c->pd_straight;
    qd.gamma = std::isnan(c->pd_gamma) ? 1.0 : c->pd_gamma;
    for (int q = 0; q < qd.n && !qd.straight; q++) {
        qd.z[q] = c->pd_z[q];
        qd.w[q] = c->pd_w[q];
    }
    if (std::isnan(c->pd_gamma)) {
        qd.lim_m[0] = 0.0;
        qd.lim_m[1] = 1.0;
        qd.lim_p[0] = 0.0;
        qd.lim_p[1] = 1.0;
    } else {  // lia_integration_limits (local_integrals.jl:100-101)
        const double g = c->pd_gamma;
        qd.lim_m[0] = 1.0 - g;
        qd.lim_m[1] = 1.0;
        qd.lim_p[0] = 0.0;
        qd.lim_p[1] = g;
    }
    c->have_points = false;
    stage_break(c, s);
    stage_begin(c, ST_POINTS, s);
    auto *flag = reinterpret_cast<volatile unsigned int *>(c->host_stage);
    unsigned int *dflag = nullptr;
    VPBS_HIP(c, hipHostGetDevicePointer((void **)&dflag, c->host_stage, 0));
    *flag = 0;  // nothing on the device uses it: the call that did has waited
    const auto coefs = uploaded ? derivative_coefs<true> : derivative_coefs<false>;
    coefs<<<nblocks(Np, 256), 256, 0, s>>>(f, c->fil_c, c->fil_fid, c->fil_d, c->fil_e);
    point_data_kernel<<<nblocks(Np, 128), 128, 0, s>>>(f, qd, c->box, c->fil_x, c->fil_c, c->fil_d, c->fil_e,
                                                       c->nodes, c->idx_prev, c->sp, c->spp, c->dlm, c->dlp,
                                                       c->points, c->charges, dflag);
    VPBS_HIP(c, hipGetLastError());
    stage_end(c, ST_POINTS, s);
    VPBS_HIP(c, hipStreamSynchronize(s));
    c->have_filaments = true;  // complete from here on: the filament of each node comes from the first kernel
    if (*flag) VPBS_TRY(device_check(c));  // counts what is wrong
    float ms = 0.f;
    VPBS_HIP(c, hipEventElapsedTime(&ms, c->stage_from[ST_POINTS], c->ev_end[ST_POINTS]));
    c->timings.point_data = ms;
    c->have_points = true;
    c->points_version++;
    c->have_stats = false;
    c->last_vel = c->last_psi = false;
    return VPBS_OK;
}

// Upload the filament description, then derive the point data on the device.
// Argument meaning as in vpbs_set_filaments (include/vpbs.h); the host checks
// done here make every index the kernels form stay inside its array.
int build_point_data(vpbs_ctx *c, int64_t Nf, const int64_t *counts, const double *X, const double *knots,
                     const double *periods, const double *offsets, const double *coefs, const double *quad_nodes,
                     const double *quad_weights, double lia_segment_fraction, int32_t nquad_ns,
                     const double *quad_ns_nodes, const double *quad_ns_weights) {
    if (Nf < 1) return fail(c, VPBS_ERR_INVALID, "need at least one filament (got Nf = %lld)", (long long)Nf);
    if (!counts || !X || !knots || !periods || !offsets || !coefs)
        return fail(c, VPBS_ERR_INVALID, "null input array");
    if ((quad_nodes == nullptr) != (quad_weights == nullptr))
        return fail(c, VPBS_ERR_INVALID, "quad_nodes and quad_weights must both be given or both be NULL");
    const bool straight = quad_nodes == nullptr;
    const int nq = c->p.nquad;
    if (straight && nq != 1)
        return fail(c, VPBS_ERR_INVALID, "straight segments (no quadrature rule) need nquad = 1 (got %d)", nq);
    if (!std::isnan(lia_segment_fraction) && !(lia_segment_fraction > 0.0 && lia_segment_fraction <= 1.0))
        return fail(c, VPBS_ERR_INVALID, "lia_segment_fraction must be in (0, 1] (got %g)", lia_segment_fraction);
    if (nquad_ns < 0 || nquad_ns > 16 || (nquad_ns > 0 && (!quad_ns_nodes || !quad_ns_weights)))
        return fail(c, VPBS_ERR_INVALID, "near-singularity quadrature: 0..16 points with nodes and weights");
    std::vector<int64_t> off((size_t)Nf);
    std::vector<int32_t> nn((size_t)Nf);
    int64_t Np = 0;
    for (int64_t f = 0; f < Nf; f++) {
        if (counts[f] < 5 || counts[f] > INT32_MAX)
            return fail(c, VPBS_ERR_INVALID, "filament %lld has %lld nodes; quintic splines need at least 5",
                        (long long)f, (long long)counts[f]);
        off[(size_t)f] = Np;
        nn[(size_t)f] = (int32_t)counts[f];
        Np += counts[f];
        if (Np > INT32_MAX) return fail(c, VPBS_ERR_INVALID, "too many nodes for 32-bit indices");
        if (!(periods[f] > 0.0) || !std::isfinite(periods[f]))
            return fail(c, VPBS_ERR_INVALID, "period of filament %lld is %g (must be finite and > 0)",
                        (long long)f, periods[f]);
    }
    const int64_t Nq = (int64_t)nq * Np;
    if (Nq > INT32_MAX / 2) return fail(c, VPBS_ERR_INVALID, "too many quadrature points for 32-bit indices");
    VPBS_HIP(c, hipSetDevice(c->device));
    c->have_points = false;
    VPBS_TRY(ensure_capacity(c, Np, Nq));
    c->have_filaments = false;
    if (Np > c->cap_fil_np) {
        c->cap_fil_np = 0;
        double **bufs[] = {&c->fil_d, &c->fil_e};
        for (double **b : bufs) {
            if (*b) VPBS_HIP(c, hipFree(*b));
            *b = nullptr;
            VPBS_HIP(c, hipMalloc((void **)b, sizeof(double) * 3 * (size_t)Np));
        }
        if (c->fil_fid) VPBS_HIP(c, hipFree(c->fil_fid));
        c->fil_fid = nullptr;
        VPBS_HIP(c, hipMalloc((void **)&c->fil_fid, sizeof(int32_t) * (size_t)Np));
        c->cap_fil_np = Np;
    }
    // one block for everything that is uploaded: positions, coefficients, knots, periods, offsets, first
    // nodes and node counts behind each other
    const size_t d3 = sizeof(double) * 3 * (size_t)Np, d1 = sizeof(double) * (size_t)Np;
    const size_t f1 = sizeof(double) * (size_t)Nf;
    const struct {
        void **dst;
        const void *src;
        size_t bytes;
    } part[] = {{(void **)&c->fil_x, X, d3},          {(void **)&c->fil_c, coefs, d3},
                {(void **)&c->fil_ts, knots, d1},     {(void **)&c->fil_T, periods, f1},
                {(void **)&c->fil_xoff, offsets, 3 * f1}, {(void **)&c->fil_off, off.data(), f1},
                {(void **)&c->fil_n, nn.data(), sizeof(int32_t) * (size_t)Nf}};
    size_t total = 0;
    for (const auto &q : part) total += q.bytes;
    if (total > c->cap_fil_block) {
        if (c->fil_block) VPBS_HIP(c, hipFree(c->fil_block));
        c->fil_block = nullptr;
        c->cap_fil_block = 0;
        VPBS_HIP(c, hipMalloc((void **)&c->fil_block, total));
        c->cap_fil_block = total;
    }
    hipStream_t s = c->s_sr;
    StreamDrain drain{c};  // the staging memory and the local arrays outlive the copies on every return
    const bool staged = total <= STAGE_BYTES && host_memory(X) && host_memory(coefs) && host_memory(knots) &&
                        host_memory(offsets);
    size_t at = 0;
    for (const auto &q : part) {
        *q.dst = c->fil_block + at;
        if (staged)
            std::memcpy(c->host_stage + STAGE_OFFSET + at, q.src, q.bytes);
        else
            VPBS_HIP(c, hipMemcpyAsync(c->fil_block + at, q.src, q.bytes, hipMemcpyHostToDevice, s));
        at += q.bytes;
    }
    if (staged) VPBS_HIP(c, hipMemcpyAsync(c->fil_block, c->host_stage + STAGE_OFFSET, total, hipMemcpyHostToDevice, s));

    // quadrature and local-integral configuration, kept for rebuilds from the device state
    c->pd_nf = Nf;
    c->pd_straight = straight;
    c->pd_gamma = lia_segment_fraction;
    for (int q = 0; q < nq && !straight; q++) {
        c->pd_z[q] = quad_nodes[q];
        c->pd_w[q] = quad_weights[q];
    }
    c->local_ns = (!std::isnan(lia_segment_fraction) && nquad_ns > 0) ? nquad_ns : 0;
    c->local_gamma = lia_segment_fraction;
    c->local_nf = Nf;
    for (int q = 0; q < c->local_ns; q++) {
        c->local_z[q] = quad_ns_nodes[q];
        c->local_w[q] = quad_ns_weights[q];
    }
    c->Np = Np;
    c->Nq = Nq;
    return point_data_from_state(c, true);
}

int add_local_integrals(vpbs_ctx *c, uint32_t flags, hipStream_t s) {
    if (!c->local_ns) return VPBS_OK;
    const bool vel = flags & VPBS_VELOCITY, psi = flags & VPBS_STREAMFUNCTION;
    const Fil f = filament_view(c);
    LocalQuad lq{};
    lq.n = c->local_ns;
    for (int q = 0; q < lq.n; q++) {
        lq.z[q] = c->local_z[q];
        lq.w[q] = c->local_w[q];
    }
    lq.lo[0] = 0.0;  // nonlia_integration_limits (local_integrals.jl:103-104)
    lq.hi[0] = 1.0 - c->local_gamma;
    lq.lo[1] = c->local_gamma;
    lq.hi[1] = 1.0;
    const double pref = c->p.Gamma / (4 * M_PI);
    local_integrals_kernel<<<nblocks(c->Np, 128), 128, 0, s>>>(f, lq, c->box, c->fil_c, c->fil_d, c->nodes, pref,
                                                              vel ? c->v_sr : nullptr, psi ? c->psi_sr : nullptr);
    VPBS_HIP(c, hipGetLastError());
    return VPBS_OK;
}

// SSPRK33 steps of the Biot–Savart velocity on the device-resident filaments
// (Timestepping.jl:1038-1076 without forcing, reconnections or adaptivity).
int advance_filaments(vpbs_ctx *c, double dt, int nsteps) {
    const int64_t Np = c->Np, n3 = 3 * Np;
    if (n3 > c->cap_step) {
        c->cap_step = 0;  // until the new buffer is there
        if (c->step_buf) VPBS_HIP(c, hipFree(c->step_buf));
        c->step_buf = nullptr;
        VPBS_HIP(c, hipMalloc((void **)&c->step_buf, sizeof(double) * 2 * (size_t)n3));
        c->cap_step = n3;
    }
    if (12 * Np > c->cap_solve) {
        c->cap_solve = 0;
        if (c->solve_buf) VPBS_HIP(c, hipFree(c->solve_buf));
        c->solve_buf = nullptr;
        VPBS_HIP(c, hipMalloc((void **)&c->solve_buf, sizeof(double) * 12 * (size_t)Np));
        c->cap_solve = 12 * Np;
    }
    double *X0 = c->step_buf, *Vs = X0 + n3;
    hipStream_t s = c->s_sr;
    const Fil f = filament_view(c);
    // node velocities into c->v_out from the current point data: the learned evaluation (cheap
    // splitting, correction, sampled check) when a network is set up, else the plain one
    const bool learned = c->lc_ready && c->lc_net;
    auto velocity = [&]() -> int {
        if (learned) return vpbs_compute_learned(c, nullptr, nullptr);
        return vpbs_compute(c, VPBS_VELOCITY, __builtin_nan(""), nullptr, nullptr);
    };
    // the point data of the filaments on the device is current unless its last build failed
    if (!c->have_points) VPBS_TRY(point_data_from_state(c));
    for (int step = 0; step < nsteps; step++) {
        for (int k = 1; k <= 3; k++) {
            VPBS_TRY(velocity());
            rk_stage<<<nblocks(n3, 256), 256, 0, s>>>(n3, k, dt, c->v_out, X0, Vs, c->fil_x);
            // stages keep the knots; after the step they are recomputed (chordal)
            if (k == 3) chordal_knots<<<(unsigned)c->pd_nf, 64, 0, s>>>(f, c->fil_x, c->fil_ts, c->fil_T);
            spline_rows<<<nblocks(Np, 256), 256, 0, s>>>(f, c->fil_x, c->solve_buf);
            spline_solve<<<(unsigned)c->pd_nf, 64, 0, s>>>(f, c->solve_buf, c->fil_c);
            VPBS_HIP(c, hipGetLastError());
            VPBS_TRY(point_data_from_state(c));
        }
    }
    return VPBS_OK;
}

}  // namespace vpbs
