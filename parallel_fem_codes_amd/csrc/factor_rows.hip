// ILU(0) numeric factorisation for rows of at most 32 entries that the streamed kernel does not take
// (the 9x9- and 12x12-block systems): one workgroup walks the lower sweep's level schedule, 16 lanes
// per row, four rows per wavefront, a barrier between levels.
//
// What bounds it is the dependency chain: a level's rows wait for the U parts and inverse pivots of
// earlier levels, and inside a row each multiplier waits for the ones before it. So a row's entries are
// spread over lanes (lane e holds entries e and e + 16): multiplier t is broadcast from its lane to the
// row's 16 lanes by a DPP move (row_newbcast) and every entry is updated at once, 10 short steps for a
// 21-entry row instead of the 110 updates of its list one by one through LDS. The U values a row needs
// do not depend on each other: all are loaded together right after the level's barrier, at addresses
// known before it -- each (entry, L entry t) pair carries the U column of the entry in row j_t as a
// 4-bit code (8 bits for rows with more than 16 L or 15 U entries) -- and everything else of the next
// level's first rows is loaded before the barrier. 81 x 81-node cavity (n = 1.9e4, 711 levels): 2.2 ms,
// against 14.8 ms with one thread per row walking its update list; 513 x 513 (n = 7.9e5, 4 599 levels):
// 60 ms against 179 ms.
//
// Arithmetic (ILUp_precond_setup.c:84-166, p = 0; contraction off): entry e starts from a_e and
// subtracts l_t * u_{j_t, col_e} for the L entries t < e in order, an L entry then becomes
// l_e = v_e * Dinv[j_e]: each entry's sequence of operations in the serial elimination, bit for bit.
#include <algorithm>

#include "common.h"
#include "device_util.h"

namespace fg {

template <int T>
__device__ __forceinline__ int row_bcast(int v)   // lane T of each 16 lanes to all 16
{
    return __builtin_amdgcn_update_dpp(0, v, 0x150 + T, 0xf, 0xf, true);
}
template <int T>
__device__ __forceinline__ double row_bcast(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = row_bcast<T>(static_cast<int>(b)), hi = row_bcast<T>(static_cast<int>(b >> 32));
    return __longlong_as_double(static_cast<long long>(static_cast<unsigned>(lo)) |
                                (static_cast<long long>(hi) << 32));
}

struct RowsArgs {
    int depth;
    const int *lvl_ptr;
    const int4 *info;     // schedule position -> {first entry, length, L count, row}
    const int2 *dep;      // [position][pass][lane t]: {first U entry of row j_t, row j_t}
    const ulonglong2 *code;   // [position][pass][word][lane]: the pairs' U columns
    const double *AA;
    double *LU, *Dinv;
    int *err;
};

// U column of the pair (entry in the low / high half of the row, L entry t of the pass); kNone: absent
template <bool WIDE>
struct Codes;
template <>
struct Codes<false> {   // 16 codes of 4 bits per half
    static constexpr unsigned kNone = 15;
    ulonglong2 w;
    __device__ __forceinline__ void load(const ulonglong2 *c) { w = c[0]; }
    template <int T>
    __device__ __forceinline__ unsigned lo() const { return static_cast<unsigned>(w.x >> (4 * T)) & 15u; }
    template <int T>
    __device__ __forceinline__ unsigned hi() const { return static_cast<unsigned>(w.y >> (4 * T)) & 15u; }
};
template <>
struct Codes<true> {    // 16 codes of 8 bits per half
    static constexpr unsigned kNone = 255;
    ulonglong2 a, b;
    __device__ __forceinline__ void load(const ulonglong2 *c) { a = c[0], b = c[16]; }
    template <int T>
    __device__ __forceinline__ unsigned lo() const
    {
        return static_cast<unsigned>((T < 8 ? a.x : a.y) >> (8 * (T % 8))) & 255u;
    }
    template <int T>
    __device__ __forceinline__ unsigned hi() const
    {
        return static_cast<unsigned>((T < 8 ? b.x : b.y) >> (8 * (T % 8))) & 255u;
    }
};

struct RowStage {
    int4 ri;
    int2 dp;
    double a0, a1;
};

template <bool WIDE>
__device__ __forceinline__ void rows_fetch(RowStage &g, Codes<WIDE> &c, const RowsArgs &A, int q, int lane)
{
    constexpr int NP = WIDE ? 2 : 1, NW = WIDE ? 2 : 1;
    g.ri = A.info[q];
    g.dp = A.dep[static_cast<size_t>(q) * (16 * NP) + lane];
    c.load(A.code + static_cast<size_t>(q) * (16 * NP * NW) + lane);
    g.a0 = A.AA[g.ri.x + (lane < g.ri.y ? lane : 0)];
    g.a1 = A.AA[g.ri.x + (lane + 16 < g.ri.y ? lane + 16 : 0)];
}

// Loads of pair T's U values (an absent pair reads the dependency's first U entry and is dropped).
template <bool WIDE, int T>
__device__ __forceinline__ void rows_load(const Codes<WIDE> &c, const double *LU, int ub, int nmax, double (&u0)[16],
                                          double (&u1)[16])
{
    if constexpr (T < 16) {
        if (T >= nmax) return;
        const int base = row_bcast<T>(ub);
        const unsigned k0 = c.template lo<T>(), k1 = c.template hi<T>();
        u0[T] = LU[base + static_cast<int>(k0 != Codes<WIDE>::kNone ? k0 : 0u)];
        u1[T] = LU[base + static_cast<int>(k1 != Codes<WIDE>::kNone ? k1 : 0u)];
        rows_load<WIDE, T + 1>(c, LU, ub, nmax, u0, u1);
    }
}

// Step T of the chain: multiplier t = 16 * PASS + T from its lane, then the update of every entry.
template <bool WIDE, int PASS, int T>
__device__ __forceinline__ void rows_chain(const Codes<WIDE> &c, int lane, int nL, int nmax, double dj,
                                           const double (&u0)[16], const double (&u1)[16], double &v0, double &v1)
{
#pragma clang fp contract(off)
    if constexpr (T < 16) {
        if (T >= nmax) return;
        double &own = PASS == 0 ? v0 : v1;
        const double m = own * dj;
        const bool mine = lane == T && 16 * PASS + T < nL;
        own = mine ? m : own;
        const double l = row_bcast<T>(m);
        const double x0 = v0 - l * u0[T], x1 = v1 - l * u1[T];
        v0 = c.template lo<T>() != Codes<WIDE>::kNone ? x0 : v0;
        v1 = c.template hi<T>() != Codes<WIDE>::kNone ? x1 : v1;
        rows_chain<WIDE, PASS, T + 1>(c, lane, nL, nmax, dj, u0, u1, v0, v1);
    }
}

__device__ __forceinline__ int rows_max(int v)   // over the wavefront's four rows (uniform)
{
    return max(max(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
               max(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

template <bool WIDE>
__device__ __forceinline__ void rows_factor(const RowsArgs &A, const RowStage &g, const Codes<WIDE> &c, int q, int lane,
                                            bool on)
{
#pragma clang fp contract(off)
    const int nL = on ? g.ri.z : 0, len = on ? g.ri.y : 0;
    double v0 = g.a0, v1 = g.a1;
    {
        const int nmax = min(16, rows_max(nL));
        const double dj = A.Dinv[g.dp.y];
        double u0[16], u1[16];
        rows_load<WIDE, 0>(c, A.LU, g.dp.x, nmax, u0, u1);
        rows_chain<WIDE, 0, 0>(c, lane, nL, nmax, dj, u0, u1, v0, v1);
    }
    if constexpr (WIDE) {
        const int nmax = rows_max(nL) - 16;
        if (nmax > 0) {
            const int2 dp = A.dep[static_cast<size_t>(q) * 32 + 16 + lane];
            Codes<true> c2;
            c2.load(A.code + static_cast<size_t>(q) * 64 + 32 + lane);
            const double dj = A.Dinv[dp.y];
            double u0[16], u1[16];
            rows_load<WIDE, 0>(c2, A.LU, dp.x, nmax, u0, u1);
            rows_chain<WIDE, 1, 0>(c2, lane, nL, nmax, dj, u0, u1, v0, v1);
        }
    }
    if (lane < len) A.LU[g.ri.x + lane] = v0;
    if (lane + 16 < len) A.LU[g.ri.x + lane + 16] = v1;
    const double piv = nL < 16 ? v0 : v1;
    if (on && lane == (nL & 15)) {
        double d = 1.0 / piv;
        if (piv == 0.0) {
            d = 0.0;
            __hip_atomic_store(A.err, 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        A.Dinv[g.ri.w] = d;
    }
}

// THREADS / 16 rows of a level at a time; every lane of a wavefront with rows runs the same loads (a
// row group past the level's end takes its first row again and stores nothing).
template <int THREADS, bool WIDE>
__global__ __launch_bounds__(THREADS) void k_ilu0_factor_rows(RowsArgs A)
{
    constexpr int NR = THREADS / 16;
    const int lane = threadIdx.x & 15, grp = threadIdx.x >> 4;
    const int wfirst = static_cast<int>(threadIdx.x >> 6) * 4;   // the wavefront's first row of a round
    RowStage g;
    Codes<WIDE> c;
    int q0 = 0, q1 = A.lvl_ptr[1], q2 = A.depth > 1 ? A.lvl_ptr[2] : q1;
    if (wfirst < q1) rows_fetch<WIDE>(g, c, A, grp < q1 ? grp : 0, lane);
    for (int l = 0; l < A.depth; ++l) {
        for (int r = q0; r + wfirst < q1; r += NR) {
            const int q = r + grp;
            const bool on = q < q1;
            if (r != q0) rows_fetch<WIDE>(g, c, A, on ? q : q0, lane);
            rows_factor<WIDE>(A, g, c, on ? q : q0, lane, on);
        }
        q0 = q1;
        q1 = q2;
        q2 = l + 3 <= A.depth ? A.lvl_ptr[l + 3] : q2;
        if (q0 + wfirst < q1) rows_fetch<WIDE>(g, c, A, q0 + grp < q1 ? q0 + grp : q0, lane);
        __syncthreads();
    }
}

// Short rows in wide levels: a thread per row, 512 rows of a level at a time. A row first issues all of its loads
// together (its update list, the finished U values and pivots it reads, its own values); its values and
// multipliers then live in LDS while the list is applied one by one. That chain is longer than the 16
// lanes', but a level of several hundred rows takes one round of it, where those take a round per 64 rows.
// Same operations in the same order, contraction off.
constexpr int kListRow = 8, kListUpd = 24, kListThreads = 512;

__global__ __launch_bounds__(kListThreads) void k_ilu0_factor_lists(int depth, const int *__restrict__ lvl_ptr,
                                                                    const int4 *__restrict__ rowinfo,
                                                                    const int2 *__restrict__ upd,
                                                                    const int *__restrict__ JA,
                                                                    const double *__restrict__ AA, double *LU,
                                                                    double *Dinv, int *err)
{
#pragma clang fp contract(off)
    __shared__ double scratch[2 * kListRow * kListThreads];
    double *v = scratch + threadIdx.x;                                 // row value e at v[e * kListThreads]
    double *dj = scratch + kListRow * kListThreads + threadIdx.x;      // pivot inverse of L entry t, likewise
    for (int l = 0; l < depth; ++l) {
        const int q1 = lvl_ptr[l + 1];
        for (int q = lvl_ptr[l] + static_cast<int>(threadIdx.x); q < q1; q += kListThreads) {
            const int4 ri = rowinfo[q];
            const int p0 = ri.x, len = ri.y, nL = ri.z, ub = ri.w;
            const int nu = rowinfo[q + 1].w - ub;   // rowinfo has a sentinel entry after the last row
            const int i = JA[p0 + nL];
            int jr[kListRow];
#pragma unroll
            for (int t = 0; t < kListRow; ++t)
                if (t < nL) jr[t] = JA[p0 + t];
#pragma unroll
            for (int e = 0; e < kListRow; ++e)
                if (e < len) v[e * kListThreads] = AA[p0 + e];
#pragma unroll
            for (int t = 0; t < kListRow; ++t)
                if (t < nL) dj[t * kListThreads] = Dinv[jr[t]];
            int sc = 0;   // L entries [0, sc) already turned into multipliers
            for (int u0 = 0; u0 < nu; u0 += kListUpd) {   // a chunk's list entries and U values loaded together
                int2 U[kListUpd];
                double Uv[kListUpd];
#pragma unroll
                for (int u = 0; u < kListUpd; ++u)
                    if (u0 + u < nu) U[u] = upd[ub + u0 + u];
#pragma unroll
                for (int u = 0; u < kListUpd; ++u)
                    if (u0 + u < nu) Uv[u] = LU[U[u].x];
#pragma unroll
                for (int u = 0; u < kListUpd; ++u) {
                    if (u0 + u < nu) {
                        const int t = U[u].y >> 16, dest = U[u].y & 0xffff;
                        for (; sc <= t; ++sc) v[sc * kListThreads] = v[sc * kListThreads] * dj[sc * kListThreads];
                        v[dest * kListThreads] -= v[t * kListThreads] * Uv[u];
                    }
                }
            }
            for (; sc < nL; ++sc) v[sc * kListThreads] = v[sc * kListThreads] * dj[sc * kListThreads];
#pragma unroll
            for (int e = 0; e < kListRow; ++e)
                if (e < len) LU[p0 + e] = v[e * kListThreads];
            const double piv = v[nL * kListThreads];
            if (piv == 0.0) {
                __hip_atomic_store(err, 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                Dinv[i] = 0.0;
            } else {
                Dinv[i] = 1.0 / piv;
            }
        }
        __syncthreads();
    }
}

// Rows per level, on average, from which rows of at most 8 entries take a thread each. Seven-point matrices,
// a thread per row against 16 lanes: 133 rows 7.4 / 5.5 ms, 167 9.7 / 8.4, 200 12.4 / 13.5, 333 30 / 38 (400 x 400 to
// 1000 x 1000 squares, SYMRCM); in random order 700 rows 0.22 / 0.38 ms (n = 9 801), 24 000 rows 12.3 / 18.4
// (n = 4.9e5).
constexpr int kListLevel = 192;

int build_rows_factor(femgpu_ctx *ctx, femgpu_csr *A)
{
    RowsFactor &F = A->rfac;
    F.ok = false;
    const int n = A->n, *IA = A->hIA.data(), *JA = A->hJA.data();
    if (n == 0) return FEMGPU_OK;
    std::vector<int> diag(n);
    for (int i = 0; i < n; ++i) diag[i] = static_cast<int>(std::lower_bound(JA + IA[i], JA + IA[i + 1], i) - JA);
    int maxrow = 0, maxL = 0, maxU = 0;
    for (int i = 0; i < n; ++i) {
        maxrow = std::max(maxrow, IA[i + 1] - IA[i]);
        maxL = std::max(maxL, diag[i] - IA[i]);
        maxU = std::max(maxU, IA[i + 1] - diag[i] - 1);
    }
    if (maxrow > 32) return FEMGPU_OK;
    F.lists = maxrow <= kListRow && n / std::max(1, A->plo.depth) >= kListLevel;
    if (F.lists) {
        FG_TRY(build_factor_plan(ctx, A, IA, JA, diag.data(), false, F.plan));
        F.ok = true;
        return FEMGPU_OK;
    }
    F.wide = maxL > 16 || maxU > 15;
    const int np = F.wide ? 2 : 1, nw = F.wide ? 2 : 1;
    std::vector<int> row_of(n), slot(n, -1);
    FG_HIP(hipMemcpy(row_of.data(), A->plo.row_of.p, sizeof(int) * n, hipMemcpyDeviceToHost));
    std::vector<int4> info(n);
    std::vector<int2> dep(static_cast<size_t>(n) * 16 * np, make_int2(0, 0));
    std::vector<unsigned long long> code(static_cast<size_t>(n) * 32 * np * nw, ~0ull);
    for (int q = 0; q < n; ++q) {
        const int i = row_of[q], p0 = IA[i], len = IA[i + 1] - p0, nL = diag[i] - p0;
        info[q] = make_int4(p0, len, nL, i);
        for (int e = 0; e < len; ++e) slot[JA[p0 + e]] = e;
        for (int t = 0; t < nL; ++t) {
            const int j = JA[p0 + t], pass = t / 16, tt = t % 16;
            dep[(static_cast<size_t>(q) * np + pass) * 16 + tt] = make_int2(diag[j] + 1, j);
            for (int k = diag[j] + 1; k < IA[j + 1]; ++k) {
                const int e = slot[JA[k]];
                if (e < 0) continue;
                const unsigned long long u = static_cast<unsigned long long>(k - diag[j] - 1);
                const int half = e / 16, lane = e % 16;
                // narrow: word pair {low half, high half}; wide: one pair of words per half
                const size_t pair = ((static_cast<size_t>(q) * np + pass) * nw + (F.wide ? half : 0)) * 16 + lane;
                unsigned long long &w = code[2 * pair + (F.wide ? tt / 8 : half)];
                const int sh = F.wide ? 8 * (tt % 8) : 4 * tt;
                const unsigned long long m = (F.wide ? 255ull : 15ull) << sh;
                w = (w & ~m) | (u << sh);
            }
        }
        for (int e = 0; e < len; ++e) slot[JA[p0 + e]] = -1;
    }
    std::vector<int> lptr(static_cast<size_t>(A->plo.depth) + 1);
    FG_HIP(hipMemcpy(lptr.data(), A->plo.lvl_ptr.p, sizeof(int) * lptr.size(), hipMemcpyDeviceToHost));
    F.maxlevel = 0;
    for (int l = 0; l < A->plo.depth; ++l) F.maxlevel = std::max(F.maxlevel, lptr[l + 1] - lptr[l]);
    FG_TRY(F.info.upload(info.data(), info.size(), ctx->stream));
    FG_TRY(F.dep.upload(dep.data(), dep.size(), ctx->stream));
    FG_TRY(F.code.upload(code.data(), code.size(), ctx->stream));
    FG_HIP(hipStreamSynchronize(ctx->stream));   // the host arrays end here
    F.ok = true;
    return FEMGPU_OK;
}

int launch_rows_factor(femgpu_ctx *ctx, femgpu_csr *A)
{
    const RowsFactor &F = A->rfac;
    if (F.lists) {
        k_ilu0_factor_lists<<<1, kListThreads, 0, ctx->stream>>>(A->plo.depth, A->plo.lvl_ptr.p, F.plan.rowinfo.p,
                                                                 F.plan.upd.p, A->JA.p, A->AA.p, A->LU.p, A->Dinv.p,
                                                                 ctx->err.p);
        FG_HIP(hipGetLastError());
        return FEMGPU_OK;
    }
    RowsArgs a;
    a.depth = A->plo.depth;
    a.lvl_ptr = A->plo.lvl_ptr.p;
    a.info = F.info.p;
    a.dep = F.dep.p;
    a.code = reinterpret_cast<const ulonglong2 *>(F.code.p);
    a.AA = A->AA.p;
    a.LU = A->LU.p;
    a.Dinv = A->Dinv.p;
    a.err = ctx->err.p;
    if (F.wide) k_ilu0_factor_rows<512, true><<<1, 512, 0, ctx->stream>>>(a);
    else if (F.maxlevel <= 32) k_ilu0_factor_rows<512, false><<<1, 512, 0, ctx->stream>>>(a);
    else k_ilu0_factor_rows<1024, false><<<1, 1024, 0, ctx->stream>>>(a);
    FG_HIP(hipGetLastError());
    return FEMGPU_OK;
}

}  // namespace fg
