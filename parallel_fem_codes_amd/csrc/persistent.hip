// Persistent batched mixed-precision GMRES: one workgroup per system runs the whole solve of its
// system in one launch -- the FP64 residual and refinement, the FP32 inner GMRES(m) on the sliced-ELL
// copy of A with the Jacobi-applied parallel ILU(0) factors, fused MGS passes, and the Givens and
// least-squares steps in LDS. Every system has its own Krylov space and Hessenberg matrix, so a
// system's iterates do not depend on the other systems of the launch: at one workgroup size (the order
// of its sums) its answer is bit-identical alone and in any batch. For the small systems of the serving loop, where one launch per kernel
// step would cost more than the step's memory traffic.
//
// Two forms. A system whose vectors fit in the workgroup's LDS runs there, its matrix and factors in
// registers where the rows per thread allow it (a step then touches memory for the FP64 residual only);
// larger ones keep the vectors in global memory. femgpu_gmres_mixed and femgpu_gmres_mixed_batched take
// the first form for small systems, where a chain of launches of 2 to 4 us each was the solve's time.
//
// Synchronisation is workgroup-local only (__syncthreads), every loop is bounded (max_refinements
// outer steps, m - 1 inner steps, the Jacobi iteration count), and every exit decision is taken
// from values that all threads of the workgroup hold identically, so every wave reaches the end.
#include <algorithm>
#include <cstring>

#include "common.h"
#include "device_util.h"

namespace fg {
namespace {

constexpr int kWgMaxBasis = 64;   // inner basis size limit: the Hessenberg matrix lives in LDS

struct WgArgs {
    const int *row_off;          // null: one system of n rows
    int n;
    const int *IA, *JA;          // FP64 CSR (outer residual)
    const double *AA;
    const int *sptr, *scol;      // sliced ELL of A (FP32 SpMV) and of the factors
    const float *sval;
    const int *rinfo;            // row -> strict-lower count | row length << 8
    const float *LU, *Dinv;      // parallel ILU(0) factors in the sliced-ELL layout, 1/diag(U)
    const double *F;
    double *X, *R;
    float *V, *T;                // basis (m + 1 vectors) and three work vectors, ldv apart
    size_t ldv;
    int kin, jac, max_ref;
    double tol, inner_tol;
    femgpu_batch_info *info;
};

__device__ __forceinline__ bool finite_norm(double v) { return v <= 1.7976931348623157e308; }

__device__ __forceinline__ void wg_report(const WgArgs &a, int sys, int refinements, int inner, double rn, double normF)
{
    femgpu_batch_info inf;
    inf.refinements = refinements;
    inf.inner_iterations = inner;
    inf.status = finite_norm(rn) && rn <= a.tol * normF ? 0 : 1;
    inf.pad = 0;
    inf.normF = normF;
    inf.true_rel_residual = normF == 0.0 ? 0.0 : finite_norm(normF) ? rn / normF : normF;
    a.info[sys] = inf;
}

// Sum over the workgroup, the same value (same order) in every thread. Two barriers: red may be
// reused by the next call at once.
template <int BS>
__device__ __forceinline__ double wg_sum(double v, double *red)
{
    v = wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < BS / 64; ++k) t += red[k];
    return t;
}

// Row loops are unrolled so that a thread has several rows' loads in flight, and the entry loop of
// a row is unrolled to the matrix's row-width bound QW with its loads unconditional (positions past
// the row's end are clamped to its first entry and their terms not added): the loads of a row go
// out together instead of one dependent round trip per entry, and the sums are the same for any QW.
template <int QW>
__device__ __forceinline__ float sell_row_dot(const WgArgs &a, const float *vals, int p, int q0, int q1,
                                              const float *x)
{
    float t = 0.0f;
#pragma unroll
    for (int u = 0; u < QW; ++u) {
        const int q = q0 + u;
        const bool in = q < q1;
        const int e = p + ((in ? q : 0) << 6);
        const float v = vals[e] * x[a.scol[e]];
        t = in ? t + v : t;
    }
    return t;
}

// z = (U~ L~)^-1 b approximated by jac Jacobi iterations per triangle (the iteration of the
// multi-kernel path): y_k = b - L y_{k-1} (y_0 = b), then z_k = Dinv (y - U z_{k-1})
// (z_0 = Dinv y, formed first into a free buffer). b is T0; the lower iterates go to T1/T2, the
// upper ones alternate over the two free buffers, and the last one lands in out.
template <int BS, int QW>
__device__ void wg_jacobi(const WgArgs &a, int r0, int r1, float *T0, float *T1, float *T2, float *out)
{
    const float *prev = nullptr;
    for (int k = 0; k < a.jac; ++k) {
        float *dst = (k & 1) ? T2 : T1;
        const float *src = prev ? prev : T0;
#pragma unroll 2
        for (int r = r0 + threadIdx.x; r < r1; r += BS) {
            const int p = a.sptr[r >> 6] + (r & 63), nl = a.rinfo[r] & 0xff;
            dst[r] = T0[r] - sell_row_dot<QW>(a, a.LU, p, 0, nl, src);
        }
        __syncthreads();
        prev = dst;
    }
    const float *y = prev;
    float *fa = T0, *fb = (y == T1) ? T2 : T1;
    // z_0 = Dinv y into fb; the iterates then alternate fa, fb, ..., the last one into out
#pragma unroll 2
    for (int r = r0 + threadIdx.x; r < r1; r += BS) fb[r] = a.Dinv[r] * y[r];
    __syncthreads();
    const float *zin = fb;
    for (int k = 1; k <= a.jac; ++k) {
        float *dst = (k == a.jac) ? out : ((k & 1) ? fa : fb);
#pragma unroll 2
        for (int r = r0 + threadIdx.x; r < r1; r += BS) {
            const int p = a.sptr[r >> 6] + (r & 63), inf = a.rinfo[r];
            const int nl = inf & 0xff, len = inf >> 8;
            dst[r] = a.Dinv[r] * (y[r] - sell_row_dot<QW>(a, a.LU, p, nl + 1, len, zin));
        }
        __syncthreads();
        zin = dst;
    }
}

// ---- systems of at most R rows per thread: the vectors a row gathers from are in LDS, its own values in
// registers. Row r0 + tid + k*BS belongs to thread tid; a Jacobi or product phase gathers from one of two
// LDS vectors and writes the other, one barrier each. Where they fit, the rows' matrix entries, factors
// and columns stay in registers for the whole solve (KEEP), so a phase touches no memory; else they are read
// again (from L2) in every phase. What bounds a step is then its chain of barriers and reductions.
// Against the path that keeps the vectors in global memory, transient systems of 361 / 1 472 / 3 481 rows:
// 84 / 181 / 337 us a solve, 139 / 429 / 734 us before (10, 14 and 12 Arnoldi steps).

__device__ __forceinline__ double lane_value(double v, int lane)   // lane: uniform
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane(static_cast<int>(b), lane), hi = __builtin_amdgcn_readlane(static_cast<int>(b >> 32), lane);
    return __longlong_as_double(static_cast<long long>(static_cast<unsigned>(lo)) | (static_cast<long long>(hi) << 32));
}

// Sum over the workgroup in every thread (as wg_sum) with one barrier: successive calls alternate between
// the two halves of red, and the barrier of a call separates the reads of the call before it from the
// writes of the call after it.
template <int BS>
__device__ __forceinline__ double wg_sum1(double v, double *red, int &half)
{
    constexpr int NW = BS / 64;
    v = wave_sum(v);
    double *rd = red + half * NW;
    half ^= 1;
    if ((threadIdx.x & 63) == 0) rd[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < NW; ++k) t += rd[k];
    return t;
}

template <int R, int QW, bool KEEP>
struct WgRows {
    int p[R], inf[R];              // sliced-ELL position of the row's first entry; strict-lower count | length << 8
    float dinv[R];
    float av[KEEP ? R : 1][QW], lv[KEEP ? R : 1][QW];
    unsigned cc[KEEP ? R : 1][QW / 2];   // columns within the system, two per word
};

// dot[k] = sum over entries q0[k] <= q < q1[k] of the thread's row k of val * x[col], in order (LU: the
// factors, else A).
template <int BS, bool LU, int R, int QW, bool KEEP>
__device__ __forceinline__ void wg_dots(const WgArgs &a, const WgRows<R, QW, KEEP> &w, const int (&q0)[R], const int (&q1)[R],
                                        int r0, int n, const float *x, float (&dot)[R])
{
#pragma unroll
    for (int k = 0; k < R; ++k) dot[k] = 0.0f;
    if constexpr (KEEP) {
        (void)r0, (void)n;
#pragma unroll
        for (int k = 0; k < R; ++k)
#pragma unroll
            for (int q = 0; q < QW; ++q) {
                const unsigned c = w.cc[k][q / 2];
                const float z = (LU ? w.lv[k][q] : w.av[k][q]) * x[q & 1 ? c >> 16 : c & 0xffffu];
                dot[k] = q >= q0[k] && q < q1[k] ? dot[k] + z : dot[k];
            }
    } else {
        const float *vals = LU ? a.LU : a.sval;
#pragma unroll
        for (int k = 0; k < R; ++k) {
            if (static_cast<int>(threadIdx.x) + k * BS >= n) continue;
            for (int q = q0[k]; q < q1[k]; q += 4) {   // four entries' loads in flight
                float v[4];
                int c[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int e = w.p[k] + ((q + u < q1[k] ? q + u : q) << 6);
                    v[u] = vals[e];
                    c[u] = a.scol[e] - r0;
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const float z = v[u] * x[c[u]];
                    dot[k] = q + u < q1[k] ? dot[k] + z : dot[k];
                }
            }
        }
    }
}

// out = (U~ L~)^-1 b by jac Jacobi iterations per triangle, as wg_jacobi: b in registers and in S0. The last
// lower iteration leaves Dinv y, the upper iteration's start, in LDS. Both vectors are free on return.
template <int BS, int R, int QW, bool KEEP>
__device__ __forceinline__ void wg_jacobi_lds(const WgArgs &a, const WgRows<R, QW, KEEP> &w, int r0, int n, const float (&b)[R],
                                              float *S0, float *S1, float (&out)[R])
{
    float y[R], d[R];
    int z[R], nl[R], nu[R], len[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {
        z[k] = 0;
        nl[k] = w.inf[k] & 0xff;
        nu[k] = nl[k] + 1;
        len[k] = w.inf[k] >> 8;
    }
    for (int it = 1; it <= a.jac; ++it) {
        wg_dots<BS, true>(a, w, z, nl, r0, n, S0, d);
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int i = static_cast<int>(threadIdx.x) + k * BS;
            y[k] = b[k] - d[k];
            if (i < n) S1[i] = it == a.jac ? w.dinv[k] * y[k] : y[k];
        }
        __syncthreads();
        float *t = S0;
        S0 = S1;
        S1 = t;
    }
    for (int it = 1; it <= a.jac; ++it) {
        wg_dots<BS, true>(a, w, nu, len, r0, n, S0, d);
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int i = static_cast<int>(threadIdx.x) + k * BS;
            out[k] = i < n ? w.dinv[k] * (y[k] - d[k]) : 0.0f;
            if (it < a.jac && i < n) S1[i] = out[k];
        }
        __syncthreads();
        float *t = S0;
        S0 = S1;
        S1 = t;
    }
}

// Givens update of column i by the first wavefront (pgmres.c:118-159): lane j holds rotation j and entry j
// of the column; the running entry is carried along the rotations.
__device__ __forceinline__ void wg_givens(int i, int ld, double hn, double eps, int last, double *H, double *cs, double *sn,
                                          double *e, int *done)
{
#pragma clang fp contract(off)
    const int lane = threadIdx.x & 63, jl = lane < i ? lane : 0;
    const double c = cs[jl], s = sn[jl], h = H[(lane <= i ? lane : 0) * ld + i], ei = e[i];
    double run = lane_value(h, 0), mine = 0.0;
    for (int j = 0; j < i; ++j) {
        const double cj = lane_value(c, j), sj = lane_value(s, j), hx = lane_value(h, j + 1);
        const double h1 = cj * run + sj * hx, h2 = -sj * run + cj * hx;
        mine = lane == j ? h1 : mine;
        run = h2;
    }
    const double rr = sqrt(run * run + hn * hn), ci = run / rr, si = hn / rr, en = -si * ei;
    if (lane < i) H[lane * ld + i] = mine;
    if (lane == 0) {
        cs[i] = ci;
        sn[i] = si;
        H[i * ld + i] = rr;
        H[(i + 1) * ld + i] = 0.0;
        e[i + 1] = en;
        e[i] = ci * ei;
        *done = !(fabs(en) > eps) || last;
    }
}

// H y = e over steps columns by the first wavefront, a column at a time: lane j holds e_j.
__device__ __forceinline__ void wg_back(int steps, int ld, const double *H, const double *e, double *y)
{
    const int lane = threadIdx.x & 63;
    double r = lane < steps ? e[lane] : 0.0, mine = 0.0;
    for (int k = steps - 1; k >= 0; --k) {
        const double yk = lane_value(r, k) / H[k * ld + k];
        const double hk = lane < k ? H[lane * ld + k] : 0.0;
        mine = lane == k ? yk : mine;
        r = r - hk * yk;
    }
    if (lane < steps) y[lane] = mine;
}

template <int BS, int QW, int R>
__device__ __forceinline__ void wg_solve_lds(const WgArgs &a, double *sm, int *s_done)
{
    constexpr bool KEEP = R * QW <= (BS == 1024 ? 16 : 32);   // what 128 / 256 registers hold
    using Rows = WgRows<R, QW, KEEP>;
    const int ld = a.kin + 1, sys = blockIdx.x, tid = threadIdx.x;
    double *H = sm, *cs = H + ld * ld, *sn = cs + ld, *e = sn + ld, *y = e + ld, *red = y + ld;
    double *XS = red + 2 * (BS / 64);                       // the FP64 iterate, in the space of S0 and S1
    float *S0 = reinterpret_cast<float *>(XS), *S1 = S0 + R * BS;
    const int r0 = a.row_off ? a.row_off[sys] : 0, n = (a.row_off ? a.row_off[sys + 1] : a.n) - r0;
    int half = 0;
    Rows w;
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int i = tid + k * BS, row = r0 + (i < n ? i : 0);   // rows past the system repeat its first, unused
        w.p[k] = n > 0 ? a.sptr[row >> 6] + (row & 63) : 0;
        w.inf[k] = n > 0 ? a.rinfo[row] : 0;
        w.dinv[k] = n > 0 ? a.Dinv[row] : 0.0f;
        if constexpr (KEEP) {
            const int ln = w.inf[k] >> 8;
#pragma unroll
            for (int q = 0; q < QW; ++q) {
                const int at = w.p[k] + ((q < ln ? q : 0) << 6);
                w.av[k][q] = n > 0 ? a.sval[at] : 0.0f;
                w.lv[k][q] = n > 0 ? a.LU[at] : 0.0f;
                const unsigned c = n > 0 ? static_cast<unsigned>(a.scol[at] - r0) : 0u;
                w.cc[k][q / 2] = q & 1 ? w.cc[k][q / 2] | (c << 16) : c;
            }
        }
    }
    int none[R], len[R];
    double acc = 0.0, x[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {
        none[k] = 0;
        len[k] = w.inf[k] >> 8;
        const double f = tid + k * BS < n ? a.F[r0 + tid + k * BS] : 0.0;
        acc += f * f;
        x[k] = 0.0;
    }
    const double normF = sqrt(wg_sum1<BS>(acc, red, half));
    int refinements = 0, inner = 0;
    double rn = normF;
    while (normF > 0.0) {
        // outer FP64 residual r = F - A X (X = 0 on the first pass), entries in row order, X from LDS
        double res[R];
        acc = 0.0;
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int i = tid + k * BS;
            res[k] = 0.0;
            if (i < n) {
                double v = a.F[r0 + i];
                if (refinements > 0) {
                    const int p0 = a.IA[r0 + i];
                    double s = 0.0;
                    for (int q = 0; q < len[k]; q += 4) {
                        double t[4];
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const int at = p0 + (q + u < len[k] ? q + u : q);
                            t[u] = a.AA[at] * XS[a.JA[at] - r0];
                        }
#pragma unroll
                        for (int u = 0; u < 4; ++u) s = q + u < len[k] ? s + t[u] : s;
                    }
                    v = v - s;
                }
                res[k] = v;
                acc += v * v;
            }
        }
        rn = sqrt(wg_sum1<BS>(acc, red, half));
        if (!finite_norm(rn) || rn <= a.tol * normF || refinements >= a.max_ref) break;
        ++refinements;
        // inner FP32 solve of M^-1 A d = M^-1 r / ||r||, started from d = 0
        const double inv_rn = 1.0 / rn;
        float b[R], v[R];
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int i = tid + k * BS;
            b[k] = static_cast<float>(res[k] * inv_rn);
            if (i < n) S0[i] = b[k];
        }
        __syncthreads();
        wg_jacobi_lds<BS>(a, w, r0, n, b, S0, S1, v);
        acc = 0.0;
#pragma unroll
        for (int k = 0; k < R; ++k) acc += static_cast<double>(v[k]) * v[k];
        const double e0 = sqrt(wg_sum1<BS>(acc, red, half));
        if (!(e0 > 0.0)) break;   // preconditioned residual vanished in FP32: nothing left to correct
        const double eps = a.inner_tol * e0;
        double scale = 1.0 / e0;
        if (tid == 0) e[0] = e0;
        int steps = 0;
        for (int i = 0; i < a.kin - 1; ++i) {
            // v_i = w / h into LDS and the basis; b = A v_i; w = M^-1 b
            const float inv = static_cast<float>(scale);
            float *Vi = a.V + i * a.ldv + r0;
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const int r = tid + k * BS;
                v[k] = v[k] * inv;
                if (r < n) {
                    S1[r] = v[k];
                    Vi[r] = v[k];
                }
            }
            __syncthreads();
            wg_dots<BS, false>(a, w, none, len, r0, n, S1, b);
#pragma unroll
            for (int k = 0; k < R; ++k)
                if (tid + k * BS < n) S0[tid + k * BS] = b[k];
            __syncthreads();
            float z[R];
            wg_jacobi_lds<BS>(a, w, r0, n, b, S0, S1, z);
            // MGS on the thread's own rows: h_j = <v_j, w>, then w -= h_j v_j; the next basis vector is
            // loaded while the workgroup sums
            float vj[R];
#pragma unroll
            for (int k = 0; k < R; ++k) vj[k] = tid + k * BS < n ? a.V[r0 + tid + k * BS] : 0.0f;
            for (int j = 0; j <= i; ++j) {
                acc = 0.0;
                float vn[R];
                const float *Vn = a.V + (j < i ? j + 1 : j) * a.ldv + r0;
#pragma unroll
                for (int k = 0; k < R; ++k) {
                    acc += static_cast<double>(vj[k]) * static_cast<double>(z[k]);
                    vn[k] = tid + k * BS < n ? Vn[tid + k * BS] : 0.0f;
                }
                const double h = wg_sum1<BS>(acc, red, half);
                if (tid == 0) H[j * ld + i] = h;
                const float hf = static_cast<float>(h);
#pragma unroll
                for (int k = 0; k < R; ++k) {
                    z[k] = z[k] - hf * vj[k];
                    vj[k] = vn[k];
                }
            }
            acc = 0.0;
#pragma unroll
            for (int k = 0; k < R; ++k) acc += static_cast<double>(z[k]) * static_cast<double>(z[k]);
            const double hn = sqrt(wg_sum1<BS>(acc, red, half));
            if (tid < 64) wg_givens(i, ld, hn, eps, i + 1 >= a.kin - 1, H, cs, sn, e, s_done);
            __syncthreads();
            steps = i + 1;
            if (*s_done) break;
            scale = 1.0 / hn;
#pragma unroll
            for (int k = 0; k < R; ++k) v[k] = z[k];
        }
        inner += steps;
        if (tid < 64) wg_back(steps, ld, H, e, y);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < R; ++k) {   // X += ||r|| * V y
            const int r = tid + k * BS;
            if (r < n) {
                double d = 0.0;
                for (int j = 0; j < steps; ++j) d = d + static_cast<double>(a.V[j * a.ldv + r0 + r]) * y[j];
                x[k] = x[k] + rn * d;
                XS[r] = x[k];
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < R; ++k)
        if (tid + k * BS < n) a.X[r0 + tid + k * BS] = x[k];
    if (tid == 0) wg_report(a, sys, refinements, inner, rn, normF);
}

// Systems of any size: vectors in global memory.
template <int BS, int QW>
__device__ void wg_solve_global(const WgArgs &a, double *sm, int &s_done)
{
    const int ld = a.kin + 1;
    double *H = sm, *cs = H + ld * ld, *sn = cs + ld, *e = sn + ld, *y = e + ld, *red = y + ld;
    const int sys = blockIdx.x, tid = threadIdx.x;
    const int r0 = a.row_off ? a.row_off[sys] : 0, r1 = a.row_off ? a.row_off[sys + 1] : a.n;
    float *T0 = a.T, *T1 = a.T + a.ldv, *T2 = a.T + 2 * a.ldv;

    double acc = 0.0;
    for (int r = r0 + tid; r < r1; r += BS) {
        const double f = a.F[r];
        acc += f * f;
        a.X[r] = 0.0;
    }
    const double normF = sqrt(wg_sum<BS>(acc, red));
    int refinements = 0, inner = 0;
    double rn = normF;
    while (normF > 0.0) {
        // outer FP64 residual r = F - A X (X = 0 on the first pass), CSR entries in row order
        acc = 0.0;
#pragma unroll 2
        for (int r = r0 + tid; r < r1; r += BS) {
            double v = a.F[r];
            if (refinements > 0) {
                const int p0 = a.IA[r], len = a.IA[r + 1] - p0;
                double s = 0.0;
#pragma unroll
                for (int q = 0; q < QW; ++q) {
                    const bool in = q < len;
                    const int p = p0 + (in ? q : 0);
                    const double t = a.AA[p] * a.X[a.JA[p]];
                    s = in ? s + t : s;
                }
                v = v - s;
            }
            a.R[r] = v;
            acc += v * v;
        }
        rn = sqrt(wg_sum<BS>(acc, red));
        if (!finite_norm(rn) || rn <= a.tol * normF || refinements >= a.max_ref) break;
        ++refinements;
        // inner FP32 solve of M^-1 A d = M^-1 r / ||r||, started from d = 0
        const double inv_rn = 1.0 / rn;
#pragma unroll 4
        for (int r = r0 + tid; r < r1; r += BS) T0[r] = static_cast<float>(a.R[r] * inv_rn);
        __syncthreads();
        float *V0 = a.V;
        wg_jacobi<BS, QW>(a, r0, r1, T0, T1, T2, V0);
        acc = 0.0;
#pragma unroll 4
        for (int r = r0 + tid; r < r1; r += BS) acc += static_cast<double>(V0[r]) * V0[r];
        const double e0 = sqrt(wg_sum<BS>(acc, red));
        if (!(e0 > 0.0)) break;   // preconditioned residual vanished in FP32: nothing left to correct
        const double eps = a.inner_tol * e0;
        const float inv0 = static_cast<float>(1.0 / e0);
#pragma unroll 4
        for (int r = r0 + tid; r < r1; r += BS) V0[r] = V0[r] * inv0;
        if (tid == 0) e[0] = e0;
        __syncthreads();
        int steps = 0;
        for (int i = 0; i < a.kin - 1; ++i) {
            const float *Vi = a.V + i * a.ldv;
            float *W = a.V + (i + 1) * a.ldv;
#pragma unroll 2
            for (int r = r0 + tid; r < r1; r += BS) {   // T0 = A v_i (sliced ELL, FP32)
                const int p = a.sptr[r >> 6] + (r & 63), len = a.rinfo[r] >> 8;
                T0[r] = sell_row_dot<QW>(a, a.sval, p, 0, len, Vi);
            }
            __syncthreads();
            wg_jacobi<BS, QW>(a, r0, r1, T0, T1, T2, W);   // W = M^-1 A v_i
            // MGS: pass j subtracts h_{j-1,i} v_{j-1} and accumulates <v_j, w> (j = i + 1: ||w||^2)
            double hprev = 0.0;
            for (int j = 0; j <= i + 1; ++j) {
                const float *Vj = a.V + j * a.ldv, *Vp = a.V + (j > 0 ? j - 1 : 0) * a.ldv;
                const float hp = static_cast<float>(hprev);
                acc = 0.0;
#pragma unroll 4
                for (int r = r0 + tid; r < r1; r += BS) {
                    float wv = W[r];
                    if (j > 0) {
                        wv = wv - hp * Vp[r];
                        W[r] = wv;
                    }
                    const float u = j <= i ? Vj[r] : wv;
                    acc += static_cast<double>(u) * static_cast<double>(wv);
                }
                const double h = wg_sum<BS>(acc, red);
                if (tid == 0 && j > 0) H[(j - 1) * ld + i] = hprev;
                hprev = h;
            }
            const double hn = sqrt(hprev);
            if (tid == 0) {
#pragma clang fp contract(off)
                H[(i + 1) * ld + i] = hn;
                for (int j = 0; j <= i - 1; ++j) {   // pgmres.c:118-159 on this system's column
                    const double h1 = cs[j] * H[j * ld + i] + sn[j] * H[(j + 1) * ld + i];
                    const double h2 = -sn[j] * H[j * ld + i] + cs[j] * H[(j + 1) * ld + i];
                    H[j * ld + i] = h1;
                    H[(j + 1) * ld + i] = h2;
                }
                const double ha = H[i * ld + i], hb = H[(i + 1) * ld + i];
                const double rr = sqrt(ha * ha + hb * hb);
                cs[i] = ha / rr;
                sn[i] = hb / rr;
                H[i * ld + i] = rr;
                H[(i + 1) * ld + i] = 0.0;
                e[i + 1] = -sn[i] * e[i];
                e[i] = cs[i] * e[i];
                s_done = !(fabs(e[i + 1]) > eps) || (i + 1 >= a.kin - 1);
            }
            __syncthreads();
            steps = i + 1;
            if (s_done) break;
            const float invh = static_cast<float>(1.0 / hn);
#pragma unroll 4
            for (int r = r0 + tid; r < r1; r += BS) W[r] = W[r] * invh;
            __syncthreads();
        }
        inner += steps;
        if (tid == 0) {   // back substitution (pgmres.c:159-170)
#pragma clang fp contract(off)
            const int i = steps - 1;
            y[i] = e[i] / H[i * ld + i];
            for (int j = i - 1; j >= 0; --j) {
                double soma = 0.0;
                for (int k = j + 1; k <= i; ++k) soma = soma + H[j * ld + k] * y[k];
                y[j] = (e[j] - soma) / H[j * ld + j];
            }
        }
        __syncthreads();
#pragma unroll 2
        for (int r = r0 + tid; r < r1; r += BS) {   // X += ||r|| * V y
            double d = 0.0;
            for (int j = 0; j < steps; ++j) d = d + static_cast<double>(a.V[j * a.ldv + r]) * y[j];
            a.X[r] = a.X[r] + rn * d;
        }
        __syncthreads();
    }
    if (tid == 0) wg_report(a, sys, refinements, inner, rn, normF);
}

// R rows per thread at most in LDS systems (the size alone decides a system's path, so its answer does not
// depend on the batch); LARGE: systems of more rows are possible.
template <int BS, int QW, int R, bool LARGE>
__global__ __launch_bounds__(BS) void k_gmres_wg(WgArgs a)
{
    extern __shared__ double sm[];
    __shared__ int s_done;
    if constexpr (LARGE) {
        if ((a.row_off ? a.row_off[blockIdx.x + 1] - a.row_off[blockIdx.x] : a.n) > R * BS) {
            wg_solve_global<BS, QW>(a, sm, s_done);
            return;
        }
    }
    wg_solve_lds<BS, QW, R>(a, sm, &s_done);
}

constexpr int kWgLdsRows = 4;   // most rows per thread of an LDS system

template <int BS, int QW>
static void wg_launch(femgpu_ctx *ctx, const WgArgs &a, int nsys, int widest)
{
    const int ld = a.kin + 1, r = (widest + BS - 1) / BS;
    const auto lds = [&](int rows) {
        return sizeof(double) * (static_cast<size_t>(ld) * ld + 4 * ld + 2 * (BS / 64) + static_cast<size_t>(rows) * BS);
    };
    if (r > kWgLdsRows) k_gmres_wg<BS, QW, kWgLdsRows, true><<<nsys, BS, lds(kWgLdsRows), ctx->stream>>>(a);
    else if (r == 4) k_gmres_wg<BS, QW, 4, false><<<nsys, BS, lds(4), ctx->stream>>>(a);
    else if (r == 3) k_gmres_wg<BS, QW, 3, false><<<nsys, BS, lds(3), ctx->stream>>>(a);
    else if (r == 2) k_gmres_wg<BS, QW, 2, false><<<nsys, BS, lds(2), ctx->stream>>>(a);
    else k_gmres_wg<BS, QW, 1, false><<<nsys, BS, lds(1), ctx->stream>>>(a);
}

template <int QW>
static void wg_launch_width(femgpu_ctx *ctx, const WgArgs &a, int nsys, int widest, int threads)
{
    if (threads == 256) wg_launch<256, QW>(ctx, a, nsys, widest);
    else if (threads == 512) wg_launch<512, QW>(ctx, a, nsys, widest);
    else wg_launch<1024, QW>(ctx, a, nsys, widest);
}

}  // namespace

// Workgroup size from the systems' mean size when the caller leaves it to the library: as few wavefronts as
// hold the rows with their matrix in registers (steady systems of 500 / 1 000 / 2 000 rows: 512 threads 137 /
// 477 / 1 427 us, 1 024 threads 194 / 533 / 1 385 us).
int wg_threads_for(long long rows, int nsys)
{
    const long long mean = rows / std::max(1, nsys);
    return mean <= 256 ? 256 : mean <= 1536 ? 512 : 1024;
}

// One launch over nsys systems (row_off: host offsets; null: the whole matrix is one system) after the
// parallel factorisation; info: device-visible memory, valid once the stream has passed the launch.
static int wg_enqueue(femgpu_ctx *ctx, femgpu_csr *A, int nsys, const int *row_off, const femgpu_mixed_opts *opt, double tol,
                      int threads, const double *d_F, double *d_X, femgpu_batch_info *d_info)
{
    const int n = A->n, kin = opt->inner_kmax;
    FG_TRY(launch_parilu32(ctx, A, opt->factor_sweeps));
    A->f32_factored = true;
    const size_t ldv = (static_cast<size_t>(n) + 63) / 64 * 64;
    FG_TRY(ctx->gm_basis32.alloc(ldv * (kin + 1)));
    FG_TRY(ctx->gm_w32.alloc(ldv * 3));
    FG_TRY(ctx->gm_r.alloc(static_cast<size_t>(n) + 64));
    if (row_off) FG_TRY(ctx->bt_rowoff.upload(row_off, static_cast<size_t>(nsys) + 1, ctx->stream));
    int widest = row_off ? 0 : n;
    if (row_off)
        for (int k = 0; k < nsys; ++k) widest = std::max(widest, row_off[k + 1] - row_off[k]);
    WgArgs a;
    a.row_off = row_off ? ctx->bt_rowoff.p : nullptr;
    a.n = n;
    a.IA = A->IA.p;
    a.JA = A->JA.p;
    a.AA = A->AA.p;
    a.sptr = A->sell_ptr.p;
    a.scol = A->sell_col.p;
    a.sval = A->sell_val.p;
    a.rinfo = A->par_rinfo.p;
    a.LU = A->par_a.p;
    a.Dinv = A->Dinv32.p;
    a.F = d_F;
    a.X = d_X;
    a.R = ctx->gm_r.p;
    a.V = ctx->gm_basis32.p;
    a.T = ctx->gm_w32.p;
    a.ldv = ldv;
    a.kin = kin;
    a.jac = opt->sweep_mode;
    a.max_ref = opt->max_refinements;
    a.tol = tol;
    a.inner_tol = opt->inner_tol;
    a.info = d_info;
    // row-width bound of the unrolled entry loops: the sliced-ELL layout holds rows of <= 16 entries
    if (A->par_maxw <= 8) wg_launch_width<8>(ctx, a, nsys, widest, threads);
    else if (A->par_maxw <= 12) wg_launch_width<12>(ctx, a, nsys, widest, threads);
    else wg_launch_width<16>(ctx, a, nsys, widest, threads);
    FG_HIP(hipGetLastError());
    return FEMGPU_OK;
}

// Whether the multi-launch mixed solvers hand a solve to the workgroup solver: the same operator and
// preconditioner, systems small enough for its LDS path (four rows for each of 1 024 threads), one workgroup each. Their own launches cost about
// 3 us each whatever the rows, 6 + i of them in Arnoldi step i (4 with classical Gram-Schmidt). Transient
// systems of 361 / 1 472 / 3 481 rows: 84 / 181 / 337 us against 479 / 669 / 601 us; a steady one of 3 800
// rows 2.42 ms against 3.97 ms; batches of 16 steady systems of 1 000 / 2 000 / 3 000 rows 0.48 / 1.38 /
// 2.06 ms against 2.06 / 2.29 / 2.51 ms for the block-diagonal launches. On either side of the lines: a
// transient system of 4 096 rows 389 us (launches 752), of 4 489, its vectors in global memory, 884 (716), of 8 281
// 1 604 (784); 16 steady systems of 2 500 / 3 300 / 4 200 rows 2.04 / 2.49 / 7.15 ms against 4.86 / 5.15 / 7.44 ms of
// launches with MGS, 2.15 / 2.41 / 3.57 ms with CGS.
bool wg_preferred(const femgpu_ctx *ctx, const femgpu_system *S, const femgpu_mixed_opts *opt, int nsys, int widest)
{
    const femgpu_csr *A = S->csr;
    return opt->multi_launch != 1 && A && S->ilu == A && A->sell_ok && A->par_ok && A->n > 0 && opt->factor_sweeps >= 1 && opt->factor_sweeps <= 16 &&
           opt->sweep_mode >= 1 && opt->sweep_mode <= 16 && opt->inner_kmax >= 2 && opt->inner_kmax <= kWgMaxBasis &&
           opt->max_refinements >= 1 && nsys <= ctx->num_cus && widest <= (nsys == 1 ? 4096 : 3072);
}

// The workgroup of a system reads no other system's rows (its vectors in LDS hold its own only): whether no
// entry of A lies between two systems.
bool uncoupled_systems(const femgpu_csr *A, int nsys, const int *row_off)
{
    for (int s = 0; s <= nsys; ++s)
        if (!A->hsplit[row_off[s]]) return false;
    return true;
}

int wg_solve_one(femgpu_ctx *ctx, femgpu_csr *A, const femgpu_mixed_opts *opt, double tol, const double *d_F, double *d_X,
                 femgpu_batch_info *info)
{
    // the result goes to host-mapped memory past the solvers' status words
    constexpr int kAt = 240;
    static_assert(kAt % 2 == 0 && kAt * sizeof(int) + sizeof(femgpu_batch_info) <= 256 * sizeof(int), "inside the status words");
    const int width = A->par_maxw <= 8 ? 8 : A->par_maxw <= 12 ? 12 : 16;
    const int threads = A->n <= 256 ? 256 : A->n <= 512 * (32 / width) ? 512 : 1024;
    FG_TRY(wg_enqueue(ctx, A, 1, nullptr, opt, tol, threads, d_F, d_X, reinterpret_cast<femgpu_batch_info *>(ctx->d_status + kAt)));
    FG_HIP(hipStreamSynchronize(ctx->stream));
    memcpy(info, const_cast<const int *>(ctx->h_status + kAt), sizeof(*info));
    return FEMGPU_OK;
}

int wg_solve_batch(femgpu_ctx *ctx, femgpu_csr *A, int nsys, const int *row_off, const femgpu_mixed_opts *opt, double tol,
                   int threads, const double *d_F, double *d_X, femgpu_batch_info *info)
{
    FG_TRY(ctx->wg_info.alloc(static_cast<size_t>(nsys)));
    FG_TRY(wg_enqueue(ctx, A, nsys, row_off, opt, tol, threads, d_F, d_X, ctx->wg_info.p));
    FG_HIP(hipMemcpyAsync(info, ctx->wg_info.p, sizeof(femgpu_batch_info) * nsys, hipMemcpyDeviceToHost, ctx->stream));
    FG_HIP(hipStreamSynchronize(ctx->stream));
    return FEMGPU_OK;
}

}  // namespace fg

using namespace fg;

extern "C" int femgpu_gmres_mixed_wg(femgpu_ctx *ctx, const femgpu_system *S, int nsys, const int *row_off,
                                     const femgpu_mixed_opts *opt, double tol, int threads, const double *d_F,
                                     double *d_X, femgpu_batch_info *info)
{
    FG_CHECK(ctx && S && S->csr && S->ilu == S->csr && !S->ebe && opt && d_F && d_X && nsys >= 1 && row_off && info,
             FEMGPU_ERR_ARG, "femgpu_gmres_mixed_wg: needs a CSR operator that is also its ILU(0) matrix");
    femgpu_csr *A = S->csr;
    const int n = A->n;
    FG_CHECK(row_off[0] == 0 && row_off[nsys] == n, FEMGPU_ERR_ARG,
             "femgpu_gmres_mixed_wg: row offsets must run from 0 to n = %d", n);
    for (int s = 0; s < nsys; ++s)
        FG_CHECK(row_off[s + 1] >= row_off[s], FEMGPU_ERR_ARG, "femgpu_gmres_mixed_wg: offsets not monotone");
    FG_CHECK(opt->factor_sweeps >= 1 && opt->factor_sweeps <= 16 && opt->sweep_mode >= 1 && opt->sweep_mode <= 16,
             FEMGPU_ERR_ARG, "femgpu_gmres_mixed_wg: needs the parallel factorisation (factor_sweeps 1..16) "
             "applied by Jacobi iterations (sweep_mode 1..16)");
    FG_CHECK(opt->inner_kmax >= 2 && opt->inner_kmax <= kWgMaxBasis && opt->max_refinements >= 0, FEMGPU_ERR_ARG,
             "femgpu_gmres_mixed_wg: inner basis %d outside [2, %d]", opt->inner_kmax, kWgMaxBasis);
    FG_CHECK(threads == 0 || threads == 256 || threads == 512 || threads == 1024, FEMGPU_ERR_ARG,
             "femgpu_gmres_mixed_wg: threads must be 0 (automatic), 256, 512 or 1024");
    FG_CHECK(A->sell_ok && A->par_ok, FEMGPU_ERR_ARG,
             "femgpu_gmres_mixed_wg: the matrix has no sliced-ELL factor layout (rows wider than 16 entries or "
             "created without the mixed-precision plans)");
    FG_CHECK(uncoupled_systems(A, nsys, row_off), FEMGPU_ERR_ARG,
             "femgpu_gmres_mixed_wg: an entry of the matrix couples two of the systems");
    if (threads == 0) threads = wg_threads_for(n, nsys);
    return wg_solve_batch(ctx, A, nsys, row_off, opt, tol, threads, d_F, d_X, info);
}
