// Element-by-element operator (ebemv.c:4-64, ebemvNDOF3.c:3-92, ebemvNDOF4.c:4-121): Q = sum_e A_e P|_e
// for s x s element blocks (s = 3 ndof, ndof = 1 transport, 3 Navier-Stokes, 4 Euler).
//
// The product is gathered per node instead of scattered per element. Element row ndof*a + d of
// element e belongs to dof d of its vertex a; a node's rows over all its elements form one group,
// summed by one thread in element order:
//   Q[eq_d] = sum over the node's elements e (ascending) of  sum_b A_e[ndof*a + d][b] * P[lm_e[b]]
// with the row sum left to right and P at the Dirichlet sink read as 0 -- the reference's own
// operations in its own order (its element loop adds the row sums of element e to Q in ascending
// e), so Q is bit-identical to its element loop, and written exactly once: no colouring, atomics or
// read-modify-write. Groups go in slices of 64, one lane each; a slice stores its incidences
// column-major (value (d, b) of incidence row r, lane l at ((r*ndof + d)*s + b)*64 + l), so every
// load of a wavefront is one contiguous run; the element rows of prescribed dofs are not stored.
// Columns are kept as int16 offsets from the node's first unknown when the mesh numbering allows
// (2 bytes per entry), else as int32 unknowns.
#include <climits>
#include <vector>

#include "common.h"
#include "device_util.h"
#include "arnoldi.h"

namespace fg {

constexpr short kSink16 = -32768;   // int16 column of the Dirichlet sink

template <typename CT>
__device__ __forceinline__ int ebe_col(CT c, int key, int NEQ);
template <>
__device__ __forceinline__ int ebe_col<short>(short c, int key, int)
{
    return c == kSink16 ? -1 : key + c;
}
template <>
__device__ __forceinline__ int ebe_col<int>(int c, int, int NEQ)
{
    return c < NEQ ? c : -1;
}

// One thread per node group. The loads of U incidences are issued together (incidences past the
// list re-read the first of the batch and are not added), then summed in list order. No
// contraction into fused multiply-adds: products and sums round as the reference's.
template <typename T, typename CT, int ND, int U>
__global__ __launch_bounds__(256) void k_ebe_gather(int ngroups, int NEQ, const int *__restrict__ iptr,
                                                    const int *__restrict__ len, const int *__restrict__ eq,
                                                    const int *__restrict__ key, const CT *__restrict__ col,
                                                    const T *__restrict__ val, const T *__restrict__ P,
                                                    T *__restrict__ Q, const int *__restrict__ skip)
{
#pragma clang fp contract(off)
    constexpr int S = 3 * ND;
    if (skip && *skip) return;
    const int g = xcd_block() * 256 + static_cast<int>(threadIdx.x);
    if (g >= ngroups) return;
    const int sl = g >> 6, l = g & 63;
    const int r0 = iptr[sl], n = len[g];
    const int kg = key ? key[g] : 0;
    T acc[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) acc[d] = T(0);
    for (int j = 0; j < n; j += U) {
        T a[U][ND][S], p[U][S];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const size_t r = static_cast<size_t>(r0 + (j + u < n ? j + u : j));
#pragma unroll
            for (int b = 0; b < S; ++b) {
                const int idx = ebe_col<CT>(col[(r * S + b) * 64 + l], kg, NEQ);
                const T pv = P[idx >= 0 ? idx : 0];
                p[u][b] = idx >= 0 ? pv : T(0);
            }
#pragma unroll
            for (int d = 0; d < ND; ++d)
#pragma unroll
                for (int b = 0; b < S; ++b) a[u][d][b] = val[((r * ND + d) * S + b) * 64 + l];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (j + u < n) {
#pragma unroll
                for (int d = 0; d < ND; ++d) {
                    T t = a[u][d][0] * p[u][0];
#pragma unroll
                    for (int b = 1; b < S; ++b) t = t + a[u][d][b] * p[u][b];
                    acc[d] = acc[d] + t;
                }
            }
    }
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        const int q = eq[(static_cast<size_t>(sl) * ND + d) * 64 + l];
        if (q < NEQ) Q[q] = acc[d];
    }
}

template <typename T>
__global__ void k_ebe_zero(int n, T *__restrict__ q, const int *__restrict__ skip)
{
    if (skip && *skip) return;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) q[i] = T(0);
}

// The FP32 product, on node block rows: a node's element blocks that share a column node are summed (in
// FP64, in element order, by the fill kernel below) and rounded to FP32 once, so a node of six triangles
// reads 7 blocks of ND x ND values instead of 6 x 3 -- the product streams values, so that is what it costs:
// 801 x 401 nodes, ND = 4, 29 us back to back and 39.6 us from HBM (170 MB; 81 us on the FP32 copy of
// the element rows, 412 MB). The FP64 product keeps the element rows: its sums are the reference's, bit for bit.
// Block row r of lane l: ND values of dof row d at ((r*ND + d)*64 + l)*ND, the ND columns at
// (r*64 + l)*ND. xs, xout: the operand is P * *xs, and that product is stored to xout (the Arnoldi
// normalisation, as k_spmv's).
template <int ND>
struct NodeVec {
    float v[ND];
};

// TAIL: the product inside an Arnoldi step (ArnoldiTail), which waits in its chains of loads where systems have some
// ten thousand unknowns: a wavefront per block, so that the nodes spread over more CUs, and a whole node of six
// triangles in one batch. 20 000 nodes of four dofs: 7.9 us with the end of the step before and the nodal blocks
// (9.6 us with 256 threads and batches of four); as three kernels 8.9 + 4.7 + 3.3. At any size: a whole inner step
// (CGS) of 20 000 / 80 000 / 181 000 / 321 000 nodes of four dofs takes 25.7 / 41.1 / 60.6 / 88.9 us so, 27.2 / 42.3 /
// 60.3 / 90.6 with 256 threads and batches of four, 32.9 / 49.3 / 65.1 / 97.9 with the nodal blocks in a kernel of
// their own; 812 000 nodes of one dof 56.5 / 56.8 / 59.7.
constexpr int kTailThreads = 64, kTailRows = 7;

template <typename CT, int ND, int U, bool TAIL>
__global__ __launch_bounds__(TAIL ? kTailThreads : 256) void k_node_rows(int ngroups, int NEQ, const int *__restrict__ bptr,
                                                   const int *__restrict__ blen, const int *__restrict__ eq,
                                                   const int *__restrict__ key, const CT *__restrict__ col,
                                                   const float *__restrict__ val, const float *__restrict__ P,
                                                   const double *__restrict__ xs_ptr, float *__restrict__ xout,
                                                   float *__restrict__ Q, const int *__restrict__ skip,
                                                   ArnoldiTail T)
{
    constexpr int BS = TAIL ? kTailThreads : 256;
    const int w = xcd_block(), g = w * BS + static_cast<int>(threadIdx.x);
    float xs;
    if constexpr (TAIL) {
        __shared__ double red[4];
        __shared__ int done;   // one read per block: the block that ends the step may set the flag meanwhile
        if (threadIdx.x == 0) done = __hip_atomic_load(skip, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (done) return;
        if (T.nb > 0) {
            const double hn = sqrt(sum_partials<BS>(T.part, T.nb, red)), inv = 1.0 / hn;
            if (w == (ngroups + BS - 1) / BS) {
                if (threadIdx.x == 0) {
                    T.G.hnorm[T.col + 1] = hn;
                    T.G.invh[T.col + 1] = inv;
                }
                givens_column(T.G, T.col, hn);
                return;
            }
            xs = static_cast<float>(inv);
        } else {
            xs = static_cast<float>(*xs_ptr);
        }
    } else {
        if (skip && *skip) return;
        xs = xs_ptr ? static_cast<float>(*xs_ptr) : 1.0f;
    }
    if (g >= ngroups) return;
    const int sl = g >> 6, l = g & 63;
    const int r0 = bptr[sl], n = blen[g];
    const int kg = key ? key[g] : 0;
    double acc[ND];   // FP32 products are exact in FP64: one rounding at the end
#pragma unroll
    for (int d = 0; d < ND; ++d) acc[d] = 0.0;
    for (int j = 0; j < n; j += U) {
        NodeVec<ND> a[U][ND];
        float p[U][ND];
#pragma unroll
        for (int u = 0; u < U; ++u) {   // block rows past the list re-read the batch's first, not added
            const size_t r = static_cast<size_t>(r0 + (j + u < n ? j + u : j));
            CT c[ND];
#pragma unroll
            for (int b = 0; b < ND; ++b) c[b] = col[(r * 64 + l) * ND + b];
#pragma unroll
            for (int d = 0; d < ND; ++d) {
                const float *src = val + ((r * ND + d) * 64 + l) * ND;
                if constexpr (ND == 4) {
                    const float4 w = *reinterpret_cast<const float4 *>(src);
                    a[u][d].v[0] = w.x, a[u][d].v[1] = w.y, a[u][d].v[2] = w.z, a[u][d].v[3] = w.w;
                } else {
#pragma unroll
                    for (int b = 0; b < ND; ++b) a[u][d].v[b] = src[b];
                }
            }
#pragma unroll
            for (int b = 0; b < ND; ++b) {
                const int idx = ebe_col<CT>(c[b], kg, NEQ);
                const float pv = P[idx >= 0 ? idx : 0] * xs;
                p[u][b] = idx >= 0 ? pv : 0.0f;
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (j + u < n) {
#pragma unroll
                for (int d = 0; d < ND; ++d)
#pragma unroll
                    for (int b = 0; b < ND; ++b)
                        acc[d] = fma(static_cast<double>(a[u][d].v[b]), static_cast<double>(p[u][b]), acc[d]);
            }
    }
    int q[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) q[d] = eq[(static_cast<size_t>(sl) * ND + d) * 64 + l];
    float x[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) x[d] = q[d] < NEQ ? static_cast<float>(acc[d]) : 0.0f;
    if constexpr (TAIL) {
        const int v = T.gnode ? T.gnode[g] : -1;
        if (v >= 0) {
#pragma clang fp contract(off)
            const float *m = T.inv + static_cast<size_t>(v) * ND * ND;
            float z[ND];
#pragma unroll
            for (int i = 0; i < ND; ++i) {
                z[i] = m[i * ND] * x[0];
#pragma unroll
                for (int j = 1; j < ND; ++j) z[i] = z[i] + m[i * ND + j] * x[j];
            }
#pragma unroll
            for (int i = 0; i < ND; ++i) x[i] = z[i];
        }
    }
#pragma unroll
    for (int d = 0; d < ND; ++d)
        if (q[d] < NEQ) {
            Q[q[d]] = x[d];
            if (xout) xout[q[d]] = P[q[d]] * xs;
        }
}

// The node of B whose unknowns are the group's, with the counts of groups that have one and that have none.
__global__ __launch_bounds__(256) void k_match_nodes(int ngroups, int ND, int NEQ, const int *__restrict__ eq,
                                                     const int *__restrict__ node_of, const int *__restrict__ id,
                                                     int *__restrict__ gnode, int *__restrict__ found)
{
    const int g = blockIdx.x * 256 + threadIdx.x;
    int v = -1, bad = 0;
    if (g < ngroups) {
        const int *e = eq + static_cast<size_t>(g >> 6) * ND * 64 + (g & 63);
        for (int d = 0; d < ND && v < 0; ++d)
            if (e[d * 64] < NEQ) v = node_of[e[d * 64]];
        for (int d = 0; d < ND; ++d) bad |= v < 0 ? e[d * 64] < NEQ : id[v * ND + d] != min(e[d * 64], NEQ);
        gnode[g] = v;
    }
    const unsigned long long has = __ballot(g < ngroups && v >= 0 && !bad), none = __ballot(g < ngroups && bad);
    if ((threadIdx.x & 63) == 0) {
        if (has) atomicAdd(found, __popcll(has));
        if (none) atomicAdd(found + 1, __popcll(none));
    }
}

// Element matrices (element order, ebe_assembly.c layout) into the gathered FP64 layout and the FP32 node
// block rows. One wavefront per (slice, dof row d): per incidence row it reads the 64 element rows in
// order -- lane l the l-th value of the rows one after the other, so a load covers whole rows instead
// of 64 strided words -- turns them through LDS, writes them column-major, and adds them to the lane's block
// row in LDS, which it rounds and writes at the end. Both sides are streams: 401 x 201
// nodes, ND = 4, 98 us for 410 MB (136 us with a thread per incidence, whose loads and stores were strided, for
// 470 MB). RB incidence rows have their loads in flight together; 2 for ND > 1: one or three are slower at
// 61 x 31 nodes or at 801 x 401 (7.7 / 383 us; 8.6 / 374 and 7.6 / 391). Nodes with more
// than kFillBlocks column nodes (LDS) take k_node_rows_fill for their FP32 rows (ACC = false here).
constexpr int kFillBlocks = 24;

template <int ND, int RB, bool ACC>
__global__ __launch_bounds__(64) void k_ebe_fill(const int *__restrict__ iptr, const int *__restrict__ bptr,
                                                 const int *__restrict__ src, const unsigned *__restrict__ slots,
                                                 const double *__restrict__ Ae, double *__restrict__ val,
                                                 float *__restrict__ val32)
{
    constexpr int S = 3 * ND, LD = S + 1;
    extern __shared__ double fill_lds[];
    double *turn = fill_lds, *acc = fill_lds + RB * 64 * LD;
    const int sl = blockIdx.x / ND, d = blockIdx.x % ND, l = threadIdx.x;
    const int nb = ACC ? bptr[sl + 1] - bptr[sl] : 0;
    if (ACC)
        for (int k = 0; k < nb * ND; ++k) acc[k * 64 + l] = 0.0;
    const int r1 = iptr[sl + 1];
    for (int r = iptr[sl]; r < r1; r += RB) {   // RB incidence rows, their loads issued together
        int base[RB];
        unsigned sc[RB];
        double w[RB][S];
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            const int ri = r + i < r1 ? r + i : r;
            base[i] = src[ri * 64 + l];
            sc[i] = ACC ? slots[ri * 64 + l] : 0u;
        }
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int k = 0; k < S; ++k) {   // value k * 64 + l of the 64 rows
                const int q = k * 64 + l, inc = q / S, b = q - inc * S;
                const int ib = __shfl(base[i], inc, 64);
                w[i][k] = Ae[static_cast<size_t>(ib >= 0 ? ib : 0) + d * S + b];   // padding dropped below
            }
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int k = 0; k < S; ++k) {
                const int q = k * 64 + l, inc = q / S, b = q - inc * S;
                turn[(i * 64 + inc) * LD + b] = w[i][k];
            }
        __syncthreads();   // one wavefront: orders its LDS writes before the reads
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            if (r + i >= r1) break;
            double v[S];
#pragma unroll
            for (int b = 0; b < S; ++b) {
                const double t = turn[(i * 64 + l) * LD + b];
                v[b] = base[i] >= 0 ? t : 0.0;
            }
            double *o = val + (static_cast<size_t>(r + i) * ND + d) * S * 64 + l;
#pragma unroll
            for (int b = 0; b < S; ++b) o[b * 64] = v[b];
            if (ACC && base[i] >= 0) {
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    const unsigned s = (sc[i] >> (8 * a)) & 255u;
                    if (s == 255u) continue;   // a column node without unknowns
#pragma unroll
                    for (int c = 0; c < ND; ++c) acc[(s * ND + c) * 64 + l] += v[ND * a + c];
                }
            }
        }
        __syncthreads();   // the turned rows have been read
    }
    if (ACC)
        for (int j = 0; j < nb; ++j) {
            float *o = val32 + ((static_cast<size_t>(bptr[sl] + j) * ND + d) * 64 + l) * ND;
            if constexpr (ND == 4) {
                *reinterpret_cast<float4 *>(o) = make_float4(
                    static_cast<float>(acc[(j * 4) * 64 + l]), static_cast<float>(acc[(j * 4 + 1) * 64 + l]),
                    static_cast<float>(acc[(j * 4 + 2) * 64 + l]), static_cast<float>(acc[(j * 4 + 3) * 64 + l]));
            } else {
#pragma unroll
                for (int c = 0; c < ND; ++c) o[c] = static_cast<float>(acc[(j * ND + c) * 64 + l]);
            }
        }
}

// The FP32 node block rows from the gathered FP64 rows, a thread per (block row, lane, dof row), for
// operators with a node of more than kFillBlocks column nodes: block slot q sums the element blocks
// wsrc[wptr[q] .. wptr[q + 1]) = 3 * incidence row + vertex, in element order. (A search of the node's incidences
// by every block row takes quadratic time at a hub.)
template <int ND>
__global__ __launch_bounds__(256) void k_node_rows_fill(const int *__restrict__ bptr, const int *__restrict__ wptr,
                                                        const int *__restrict__ wsrc, const double *__restrict__ val,
                                                        float *__restrict__ val32)
{
    constexpr int S = 3 * ND;
    const int sl = blockIdx.x / ND, d = blockIdx.x % ND, l = threadIdx.x & 63;
    for (int j = bptr[sl] + static_cast<int>(threadIdx.x >> 6); j < bptr[sl + 1]; j += 4) {
        const size_t q = static_cast<size_t>(j) * 64 + l;
        double acc[ND];
#pragma unroll
        for (int c = 0; c < ND; ++c) acc[c] = 0.0;
        for (int k = wptr[q]; k < wptr[q + 1]; ++k) {
            const int r = wsrc[k] / 3, a = wsrc[k] % 3;
            const double *v = val + ((static_cast<size_t>(r) * ND + d) * S + ND * a) * 64 + l;
#pragma unroll
            for (int c = 0; c < ND; ++c) acc[c] += v[c * 64];
        }
#pragma unroll
        for (int c = 0; c < ND; ++c)
            val32[((static_cast<size_t>(j) * ND + d) * 64 + l) * ND + c] = static_cast<float>(acc[c]);
    }
}

template <typename CT, int ND, int U, int U32>
static void gather_launch(femgpu_ctx *ctx, const femgpu_ebe *E, const CT *col, const CT *bcol, const double *P, double *Q,
                          const float *P32, float *Q32, const int *skip, const double *xs, float *xout,
                          const ArnoldiTail *tail)
{
    const int grid = xcd_grid((E->ngroups + 255) / 256);
    const int *key = E->col16 ? E->key.p : nullptr;
    if (P32 && tail)   // one block more for the end of the step before
        k_node_rows<CT, ND, kTailRows, true><<<xcd_grid((E->ngroups + kTailThreads - 1) / kTailThreads + 1), kTailThreads, 0,
                                              ctx->stream>>>(
            E->ngroups, E->NEQ, E->bptr.p, E->blen.p, E->eq.p, key, bcol, E->val32.p, P32, xs, xout, Q32, skip, *tail);
    else if (P32)
        k_node_rows<CT, ND, U32, false><<<grid, 256, 0, ctx->stream>>>(E->ngroups, E->NEQ, E->bptr.p, E->blen.p, E->eq.p, key,
                                                                      bcol, E->val32.p, P32, xs, xout, Q32, skip,
                                                                      ArnoldiTail());
    else
        k_ebe_gather<double, CT, ND, U><<<grid, 256, 0, ctx->stream>>>(E->ngroups, E->NEQ, E->iptr.p, E->len.p, E->eq.p, key,
                                                                       col, E->val.p, P, Q, skip);
}

// Q = A P in FP64 (P32 null) or FP32.
static int ebe_product(femgpu_ctx *ctx, const femgpu_ebe *E, const double *P, double *Q, const float *P32, float *Q32,
                       const int *skip, const double *xs = nullptr, float *xout = nullptr,
                       const ArnoldiTail *tail = nullptr)
{
    FG_CHECK(E->has_values, FEMGPU_ERR_STATE, "femgpu_ebemv: element matrices not set");
    if (E->zero_q && E->NEQ > 0) {
        const int grid = std::min(4096, (E->NEQ + 255) / 256);
        if (P32) k_ebe_zero<float><<<grid, 256, 0, ctx->stream>>>(E->NEQ, Q32, skip);
        else k_ebe_zero<double><<<grid, 256, 0, ctx->stream>>>(E->NEQ, Q, skip);
        FG_HIP(hipGetLastError());
    }
    if (E->ngroups == 0) return FEMGPU_OK;
    const short *c16 = E->col16v.p, *b16 = E->bcol16.p;
    const int *c32 = E->col32v.p, *b32 = E->bcol32.p;
    switch (E->ndof) {
    case 1:
        if (E->col16) gather_launch<short, 1, 6, 7>(ctx, E, c16, b16, P, Q, P32, Q32, skip, xs, xout, tail);
        else gather_launch<int, 1, 6, 7>(ctx, E, c32, b32, P, Q, P32, Q32, skip, xs, xout, tail);
        break;
    case 3:
        if (E->col16) gather_launch<short, 3, 1, 4>(ctx, E, c16, b16, P, Q, P32, Q32, skip, xs, xout, tail);
        else gather_launch<int, 3, 1, 4>(ctx, E, c32, b32, P, Q, P32, Q32, skip, xs, xout, tail);
        break;
    default:
        if (E->col16) gather_launch<short, 4, 1, 4>(ctx, E, c16, b16, P, Q, P32, Q32, skip, xs, xout, tail);
        else gather_launch<int, 4, 1, 4>(ctx, E, c32, b32, P, Q, P32, Q32, skip, xs, xout, tail);
        break;
    }
    FG_HIP(hipGetLastError());
    return FEMGPU_OK;
}

int launch_ebemv(femgpu_ctx *ctx, const femgpu_ebe *E, const double *P, double *Q, const int *skip)
{
    return ebe_product(ctx, E, P, Q, nullptr, nullptr, skip);
}

int launch_ebemv32(femgpu_ctx *ctx, const femgpu_ebe *E, const float *P, float *Q, const int *skip, const double *xs,
                   float *xout, const ArnoldiTail *tail)
{
    FG_CHECK(!xout || ebe_scales(E), FEMGPU_ERR_ARG, "EBE product: some unknown has no node row to store its scaled value");
    return ebe_product(ctx, E, nullptr, nullptr, P, Q, skip, xs, xout, tail);
}

int ebe_match_nodes(femgpu_ctx *ctx, const femgpu_ebe *E, const femgpu_blockdiag *B, const int **gnode, int *want)
{
    *gnode = nullptr;
    const int *node_of, *id;
    if (!blockdiag_nodes(B, E->ndof, E->NEQ, &node_of, &id, want) || E->ngroups == 0) return FEMGPU_OK;
    FG_TRY(ctx->node_match.alloc(static_cast<size_t>(E->ngroups) + 2));
    int *found = ctx->node_match.p + E->ngroups;
    FG_HIP(hipMemsetAsync(found, 0, 2 * sizeof(int), ctx->stream));
    k_match_nodes<<<(E->ngroups + 255) / 256, 256, 0, ctx->stream>>>(E->ngroups, E->ndof, E->NEQ, E->eq.p, node_of, id,
                                                                     ctx->node_match.p, found);
    FG_HIP(hipGetLastError());
    FG_HIP(hipMemcpyAsync(ctx->h_pinned + kPinMatch, found, 2 * sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
    *gnode = ctx->node_match.p;
    return FEMGPU_OK;
}

bool ebe_scales(const femgpu_ebe *E) { return !E->zero_q; }

template <int ND>
static int fill_launch(femgpu_ctx *ctx, const femgpu_ebe *E, const double *Ae)
{
    constexpr int S = 3 * ND, RB = ND == 1 ? 6 : 2;
    const int grid = E->nslices * ND;
    const size_t turn = sizeof(double) * RB * 64 * (S + 1);
    if (!E->wide_slots) {
        k_ebe_fill<ND, RB, true><<<grid, 64, turn + sizeof(double) * 64 * ND * E->maxblk, ctx->stream>>>(
            E->iptr.p, E->bptr.p, E->src.p, E->slots.p, Ae, E->val.p, E->val32.p);
    } else {
        k_ebe_fill<ND, RB, false><<<grid, 64, turn, ctx->stream>>>(E->iptr.p, nullptr, E->src.p, nullptr, Ae, E->val.p, nullptr);
        FG_HIP(hipGetLastError());
        k_node_rows_fill<ND><<<grid, 256, 0, ctx->stream>>>(E->bptr.p, E->wptr.p, E->wsrc.p, E->val.p, E->val32.p);
    }
    FG_HIP(hipGetLastError());
    return FEMGPU_OK;
}

// Node block rows of the FP32 product, planned on the device from the gathered columns (on the host the search for a
// node's column nodes took 10 ms for 511 x 640 squares, a third of the creation). One lane per group: its column
// nodes in order of appearance, each known by its first unknown; slots: the positions of every incidence's three
// column nodes among them (8 bits each, 255: none); width: column nodes of the slice's longest group.
constexpr int kBlockCols = 2 * kFillBlocks;   // fewer than kFillBlocks triangles: at most 2 * 23 + 1 column nodes

template <typename CT, int ND>
__global__ __launch_bounds__(64) void k_block_slots(int ngroups, int NEQ, const int *__restrict__ iptr,
                                                    const int *__restrict__ len, const int *__restrict__ key,
                                                    const CT *__restrict__ col, unsigned *__restrict__ slots,
                                                    int *__restrict__ blen, int *__restrict__ width)
{
    constexpr int S = 3 * ND;
    __shared__ int cols[kBlockCols * 64];
    const int sl = blockIdx.x, l = threadIdx.x, g = sl * 64 + l;
    const int n = g < ngroups ? len[g] : 0, kg = key && g < ngroups ? key[g] : 0, r1 = iptr[sl + 1];
    int nc = 0;
    for (int r = iptr[sl], j = 0; r < r1; ++r, ++j) {
        unsigned code = ~0u;
        for (int a = 0; a < 3 && j < n; ++a) {
            int k = -1;
            for (int d = 0; d < ND && k < 0; ++d) k = ebe_col<CT>(col[(static_cast<size_t>(r) * S + ND * a + d) * 64 + l], kg, NEQ);
            if (k < 0) continue;   // a node without unknowns
            int at = 0;
            while (at < nc && cols[at * 64 + l] != k) ++at;
            if (at == nc) cols[nc++ * 64 + l] = k;
            code = (code & ~(255u << (8 * a))) | (static_cast<unsigned>(at) << (8 * a));
        }
        slots[static_cast<size_t>(r) * 64 + l] = code;
    }
    if (g < ngroups) blen[g] = nc;
    for (int o = 32; o > 0; o >>= 1) nc = max(nc, __shfl_xor(nc, o, 64));
    if (l == 0) width[sl] = nc;
}

// The columns of the block rows: those of the first incidence that has the node.
template <typename CT, int ND>
__global__ __launch_bounds__(64) void k_block_cols(int ngroups, CT sink, const int *__restrict__ iptr,
                                                   const int *__restrict__ bptr, const int *__restrict__ len,
                                                   const int *__restrict__ blen, const CT *__restrict__ col,
                                                   const unsigned *__restrict__ slots, CT *__restrict__ bcol)
{
    constexpr int S = 3 * ND;
    const int sl = blockIdx.x, l = threadIdx.x, g = sl * 64 + l;
    const int n = g < ngroups ? len[g] : 0, nc = g < ngroups ? blen[g] : 0, r0 = iptr[sl], b0 = bptr[sl], b1 = bptr[sl + 1];
    int seen = 0;
    for (int j = 0; j < n; ++j) {
        const unsigned code = slots[static_cast<size_t>(r0 + j) * 64 + l];
        for (int a = 0; a < 3; ++a) {
            if (((code >> (8 * a)) & 255u) != static_cast<unsigned>(seen)) continue;
            for (int d = 0; d < ND; ++d)
                bcol[(static_cast<size_t>(b0 + seen) * 64 + l) * ND + d] =
                    col[(static_cast<size_t>(r0 + j) * S + ND * a + d) * 64 + l];
            ++seen;
        }
    }
    for (int b = b0 + nc; b < b1; ++b)
        for (int d = 0; d < ND; ++d) bcol[(static_cast<size_t>(b) * 64 + l) * ND + d] = sink;
}

template <typename CT, int ND>
static int block_rows_of(femgpu_ctx *ctx, femgpu_ebe *E, const CT *col, DevBuf<CT> &bcol, CT sink)
{
    hipStream_t st = ctx->stream;
    DevBuf<int> width;
    std::vector<int> bptr(static_cast<size_t>(E->nslices) + 1, 0);
    FG_TRY(width.alloc(static_cast<size_t>(E->nslices)));
    FG_TRY(E->slots.alloc(static_cast<size_t>(E->nrows) * 64));
    FG_TRY(E->blen.alloc(static_cast<size_t>(E->ngroups)));
    const int *key = E->col16 ? E->key.p : nullptr;
    if (E->nslices > 0) {
        k_block_slots<CT, ND><<<E->nslices, 64, 0, st>>>(E->ngroups, E->NEQ, E->iptr.p, E->len.p, key, col, E->slots.p,
                                                        E->blen.p, width.p);
        FG_HIP(hipGetLastError());
        FG_HIP(hipMemcpyAsync(bptr.data() + 1, width.p, sizeof(int) * E->nslices, hipMemcpyDeviceToHost, st));
        FG_HIP(hipStreamSynchronize(st));
    }
    for (int sl = 0; sl < E->nslices; ++sl) {
        E->maxblk = std::max(E->maxblk, bptr[sl + 1]);
        bptr[sl + 1] += bptr[sl];
    }
    if (E->maxblk > kFillBlocks) return FEMGPU_OK;   // too many column nodes for the fill kernel: planned as hubs
    E->nbrows = bptr[E->nslices];
    FG_TRY(E->bptr.upload(bptr.data(), bptr.size(), st));
    FG_TRY(bcol.alloc(static_cast<size_t>(E->nbrows) * 64 * ND));
    if (E->nslices > 0) {
        k_block_cols<CT, ND><<<E->nslices, 64, 0, st>>>(E->ngroups, sink, E->iptr.p, E->bptr.p, E->len.p, E->blen.p, col,
                                                       E->slots.p, bcol.p);
        FG_HIP(hipGetLastError());
    }
    FG_HIP(hipStreamSynchronize(st));   // the host array ends here
    return FEMGPU_OK;
}

static int block_rows(femgpu_ctx *ctx, femgpu_ebe *E)
{
    const short s16 = kSink16;
    switch (E->ndof) {
    case 1: return E->col16 ? block_rows_of<short, 1>(ctx, E, E->col16v.p, E->bcol16, s16) : block_rows_of<int, 1>(ctx, E, E->col32v.p, E->bcol32, E->NEQ);
    case 3: return E->col16 ? block_rows_of<short, 3>(ctx, E, E->col16v.p, E->bcol16, s16) : block_rows_of<int, 3>(ctx, E, E->col32v.p, E->bcol32, E->NEQ);
    default: return E->col16 ? block_rows_of<short, 4>(ctx, E, E->col16v.p, E->bcol16, s16) : block_rows_of<int, 4>(ctx, E, E->col32v.p, E->bcol32, E->NEQ);
    }
}

// The same on the host, for operators with a node of too many column nodes for the fill kernel's LDS: the block
// slots' element blocks (wptr, wsrc) in place of the incidences' positions. gptr, inc: a group's incidences 3 e + a;
// kinc: the first unknown of every incidence's node (-1: none); gkey: a group's first unknown.
static int hub_block_rows(femgpu_ctx *ctx, femgpu_ebe *E, const std::vector<int> &iptr, const std::vector<int> &inc,
                          const std::vector<int> &gptr, const std::vector<int> &kinc, const std::vector<int> &gkey,
                          const int *lm)
{
    const int ng = E->ngroups, nd = E->ndof, s = E->s;
    hipStream_t st = ctx->stream;
    std::vector<int> bptr(static_cast<size_t>(E->nslices) + 1, 0), blen(static_cast<size_t>(ng), 0);
    std::vector<int> pos(static_cast<size_t>(E->NEQ), -1);   // a column node's position by its key
    std::vector<int> at(3 * static_cast<size_t>(gptr[ng]), -1);
    for (int g = 0; g < ng; ++g) {
        for (int q = gptr[g]; q < gptr[g + 1]; ++q)
            for (int a = 0; a < 3; ++a) {
                const int k = kinc[inc[q] - inc[q] % 3 + a];
                if (k < 0) continue;
                if (pos[k] < 0) pos[k] = blen[g]++;
                at[3 * static_cast<size_t>(q) + a] = pos[k];
            }
        for (int q = gptr[g]; q < gptr[g + 1]; ++q)
            for (int a = 0; a < 3; ++a)
                if (const int k = kinc[inc[q] - inc[q] % 3 + a]; k >= 0) pos[k] = -1;
        bptr[(g >> 6) + 1] = std::max(bptr[(g >> 6) + 1], blen[g]);
    }
    E->maxblk = 0;
    for (int sl = 0; sl < E->nslices; ++sl) {
        E->maxblk = std::max(E->maxblk, bptr[sl + 1]);
        bptr[sl + 1] += bptr[sl];
    }
    const size_t nb = static_cast<size_t>(bptr[E->nslices]) * 64;
    std::vector<int> wptr(nb + 1, 0), wsrc, b32(E->col16 ? 0 : nb * nd, E->NEQ);
    std::vector<short> b16(E->col16 ? nb * nd : 0, kSink16);
    const auto slot_of = [&](int g, int p) { return (static_cast<size_t>(bptr[g >> 6]) + p) * 64 + (g & 63); };
    for (int g = 0; g < ng; ++g)
        for (int q = gptr[g]; q < gptr[g + 1]; ++q)
            for (int a = 0; a < 3; ++a) {
                const int p = at[3 * static_cast<size_t>(q) + a];
                if (p < 0) continue;
                const size_t o = slot_of(g, p);
                if (wptr[o + 1]++ > 0) continue;   // the node's columns from its first incidence
                const int *L = lm + static_cast<size_t>(inc[q] / 3) * s + nd * a;
                for (int d = 0; d < nd; ++d) {
                    if (L[d] >= E->NEQ) continue;
                    if (E->col16) b16[o * nd + d] = static_cast<short>(L[d] - gkey[g]);
                    else b32[o * nd + d] = L[d];
                }
            }
    for (size_t q = 0; q < nb; ++q) wptr[q + 1] += wptr[q];
    wsrc.resize(static_cast<size_t>(wptr[nb]));
    for (int g = 0; g < ng; ++g)
        for (int q = gptr[g]; q < gptr[g + 1]; ++q)
            for (int a = 0; a < 3; ++a)
                if (const int p = at[3 * static_cast<size_t>(q) + a]; p >= 0)
                    wsrc[wptr[slot_of(g, p)]++] = 3 * (iptr[g >> 6] + q - gptr[g]) + a;
    for (size_t q = nb; q > 0; --q) wptr[q] = wptr[q - 1];
    wptr[0] = 0;
    E->wide_slots = true;
    E->nbrows = bptr[E->nslices];
    E->slots.release();
    FG_TRY(E->bptr.upload(bptr.data(), bptr.size(), st));
    FG_TRY(E->blen.upload(blen.data(), blen.size(), st));
    FG_TRY(E->wptr.upload(wptr.data(), wptr.size(), st));
    FG_TRY(E->wsrc.upload(wsrc.data(), wsrc.size(), st));
    if (E->col16) FG_TRY(E->bcol16.upload(b16.data(), b16.size(), st));
    else FG_TRY(E->bcol32.upload(b32.data(), b32.size(), st));
    FG_HIP(hipStreamSynchronize(st));   // the host arrays end here
    return FEMGPU_OK;
}

}  // namespace fg

using namespace fg;

extern "C" int femgpu_ebe_create(femgpu_ctx *ctx, int nel, int s, int NEQ, const int *lm, femgpu_ebe **out)
{
    FG_CHECK(ctx && out && nel >= 0 && NEQ >= 0 && lm && (s == 3 || s == 9 || s == 12), FEMGPU_ERR_ARG,
             "femgpu_ebe_create: bad arguments (s must be 3, 9 or 12)");
    FG_CHECK(static_cast<long long>(nel) * s * s < INT_MAX, FEMGPU_ERR_ARG, "femgpu_ebe_create: %d elements of %dx%d "
             "exceed the int32 element-matrix index", nel, s, s);
    const size_t total = static_cast<size_t>(nel) * s;
    for (size_t q = 0; q < total; ++q)
        FG_CHECK(lm[q] >= 0 && lm[q] <= NEQ, FEMGPU_ERR_ARG, "femgpu_ebe_create: lm entry %d out of [0, NEQ]", lm[q]);
    const int nd = s / 3;
    // incidence (e, a) -> its node's first unknown (the group key); nodes with every dof prescribed
    // contribute no rows
    std::vector<int> kinc(static_cast<size_t>(nel) * 3, -1), cnt(static_cast<size_t>(NEQ) + 1, 0);
    // and whether the columns fit in 16 bits as offsets from it
    bool fits16 = true;
    for (int e = 0; e < nel; ++e) {
        const int *L = lm + static_cast<size_t>(e) * s;
        int *k = kinc.data() + 3 * static_cast<size_t>(e);
        int lo = INT_MAX, hi = -1;   // the element's unknowns
        for (int a = 0; a < 3; ++a)
            for (int d = 0; d < nd; ++d) {
                const int q = L[nd * a + d];
                if (q >= NEQ) continue;
                if (k[a] < 0) k[a] = q;
                lo = std::min(lo, q);
                hi = std::max(hi, q);
            }
        for (int a = 0; a < 3; ++a) {
            if (k[a] < 0) continue;
            ++cnt[k[a]];
            fits16 = fits16 && k[a] - lo <= 32767 && hi - k[a] <= 32767;
        }
    }
    std::vector<int> gid(static_cast<size_t>(NEQ) + 1, -1), gkey;
    for (int k = 0; k < NEQ; ++k)
        if (cnt[k] > 0) {
            gid[k] = static_cast<int>(gkey.size());
            gkey.push_back(k);
        }
    const int ng = static_cast<int>(gkey.size());
    std::vector<int> gptr(static_cast<size_t>(ng) + 1, 0);
    for (int g = 0; g < ng; ++g) gptr[g + 1] = gptr[g] + cnt[gkey[g]];
    std::vector<int> inc(gptr[ng]), fillp(gptr.begin(), gptr.end() - 1);
    for (size_t ea = 0; ea < kinc.size(); ++ea)
        if (kinc[ea] >= 0) inc[fillp[gid[kinc[ea]]]++] = static_cast<int>(ea);   // element order kept
    // the node's unknowns, identical in every element at the node
    const int nslices = (ng + 63) / 64;
    std::vector<int> eq(static_cast<size_t>(nslices) * nd * 64, NEQ);
    std::vector<char> covered(static_cast<size_t>(NEQ) + 1, 0);
    for (int g = 0; g < ng; ++g) {
        const int e0 = inc[gptr[g]] / 3, a0 = inc[gptr[g]] % 3;
        for (int q = gptr[g]; q < gptr[g + 1]; ++q) {
            const int e = inc[q] / 3, a = inc[q] % 3;
            for (int d = 0; d < nd; ++d)
                FG_CHECK(lm[static_cast<size_t>(e) * s + nd * a + d] == lm[static_cast<size_t>(e0) * s + nd * a0 + d],
                         FEMGPU_ERR_ARG, "femgpu_ebe_create: element %d and %d give one node different unknowns", e0, e);
        }
        for (int d = 0; d < nd; ++d) {
            const int u = lm[static_cast<size_t>(e0) * s + nd * a0 + d];
            eq[(static_cast<size_t>(g >> 6) * nd + d) * 64 + (g & 63)] = u;
            covered[u] = 1;
        }
    }
    bool zero_q = false;
    for (int k = 0; k < NEQ; ++k) zero_q = zero_q || !covered[k];
    std::vector<int> iptr(static_cast<size_t>(nslices) + 1, 0), len(ng);
    int maxinc = 0;
    for (int sl = 0; sl < nslices; ++sl) {
        int w = 0;
        for (int g = 64 * sl; g < std::min(ng, 64 * sl + 64); ++g) {
            len[g] = gptr[g + 1] - gptr[g];
            w = std::max(w, len[g]);
        }
        maxinc = std::max(maxinc, w);
        iptr[sl + 1] = iptr[sl] + w;
    }
    const int nrows = iptr[nslices];
    const size_t nslots = static_cast<size_t>(nrows) * 64;
    FG_CHECK(nslots * s * nd < (size_t{1} << 40) && nslots < static_cast<size_t>(INT_MAX), FEMGPU_ERR_ARG,
             "femgpu_ebe_create: operator too large");
    // Per incidence its rows' place and its columns. The slices are independent: large operators take several host
    // threads (below, a thread that waits for a processor, 4 ms beside a pool of threads that spin, would cost more
    // than it saves).
    std::vector<int> src(nslots, -1), c32(fits16 ? 0 : nslots * s, NEQ);
    std::vector<short> c16(fits16 ? nslots * s : 0, kSink16);
    host_pieces(static_cast<size_t>(nslices), nel >= 1 << 18 ? 1 << 8 : SIZE_MAX, [&](size_t s0, size_t s1, size_t) {
        for (int g = static_cast<int>(64 * s0); g < std::min(ng, static_cast<int>(64 * s1)); ++g) {
            const int l = g & 63, key = gkey[g];
            for (int j = 0; j < len[g]; ++j) {
                const int ea = inc[gptr[g] + j], e = ea / 3, a = ea % 3;
                const size_t r = static_cast<size_t>(iptr[g >> 6] + j);
                src[r * 64 + l] = e * s * s + nd * a * s;
                const int *L = lm + static_cast<size_t>(e) * s;
                if (fits16) {
                    short *o = c16.data() + r * s * 64 + l;
                    for (int b = 0; b < s; ++b) o[b * 64] = L[b] < NEQ ? static_cast<short>(L[b] - key) : kSink16;
                } else {
                    int *o = c32.data() + r * s * 64 + l;
                    for (int b = 0; b < s; ++b) o[b * 64] = L[b];
                }
            }
        }
    });
    auto *E = new femgpu_ebe();
    E->ctx = ctx;
    E->nslices = nslices;
    E->nel = nel;
    E->s = s;
    E->ndof = nd;
    E->NEQ = NEQ;
    E->ngroups = ng;
    E->nrows = nrows;
    E->maxinc = maxinc;
    E->col16 = fits16 ? 1 : 0;
    E->zero_q = zero_q;
    E->hiptr = iptr;
    hipStream_t st = ctx->stream;
    int rc = E->iptr.upload(iptr.data(), iptr.size(), st);
    if (!rc) rc = E->len.upload(len.data(), len.size(), st);
    if (!rc) rc = E->eq.upload(eq.data(), eq.size(), st);
    if (!rc) rc = E->src.upload(src.data(), src.size(), st);
    if (!rc && fits16) rc = E->key.upload(gkey.data(), gkey.size(), st);
    if (!rc && fits16) rc = E->col16v.upload(c16.data(), c16.size(), st);
    if (!rc && !fits16) rc = E->col32v.upload(c32.data(), c32.size(), st);
    if (!rc) rc = E->val.alloc(nslots * s * nd);
    if (!rc) rc = maxinc < kFillBlocks ? block_rows(ctx, E) : FEMGPU_OK;
    if (!rc && (maxinc >= kFillBlocks || E->maxblk > kFillBlocks)) rc = hub_block_rows(ctx, E, iptr, inc, gptr, kinc, gkey, lm);
    if (!rc) rc = E->val32.alloc(static_cast<size_t>(E->nbrows) * 64 * nd * nd);
    if (!rc && hipStreamSynchronize(st) != hipSuccess) rc = FEMGPU_ERR_HIP;   // host arrays end here
    if (rc) {
        delete E;
        return rc;
    }
    *out = E;
    return FEMGPU_OK;
}

extern "C" int femgpu_ebe_destroy(femgpu_ebe *E)
{
    delete E;
    return FEMGPU_OK;
}

extern "C" int femgpu_ebe_set_values(femgpu_ebe *E, const double *A, int on_device)
{
    FG_CHECK(E && A, FEMGPU_ERR_ARG, "femgpu_ebe_set_values: bad arguments");
    femgpu_ctx *ctx = E->ctx;
    const size_t total = static_cast<size_t>(E->nel) * E->s * E->s;
    DevBuf<double> tmp;
    const double *dA = A;
    if (!on_device) {
        FG_TRY(tmp.upload(A, total, ctx->stream));
        dA = tmp.p;
    }
    if (E->nrows > 0) switch (E->ndof) {
        case 1: FG_TRY(fill_launch<1>(ctx, E, dA)); break;
        case 3: FG_TRY(fill_launch<3>(ctx, E, dA)); break;
        default: FG_TRY(fill_launch<4>(ctx, E, dA)); break;
        }
    if (!on_device) FG_HIP(hipStreamSynchronize(ctx->stream));
    E->has_values = true;
    return FEMGPU_OK;
}

extern "C" int femgpu_ebe_get_info(femgpu_ebe *E, femgpu_ebe_info *info)
{
    FG_CHECK(E && info, FEMGPU_ERR_ARG, "femgpu_ebe_get_info: bad arguments");
    const long long slots = static_cast<long long>(E->nrows) * 64, s = E->s, nd = E->ndof;
    const long long nsl = static_cast<long long>(E->hiptr.size()) - 1;
    const long long meta = 4LL * E->ngroups * (E->col16 ? 2 : 1) + 4 * (nsl + 1) + 4 * nsl * nd * 64;
    const long long cols = slots * s * (E->col16 ? 2 : 4);
    info->groups = E->ngroups;
    info->max_incidences = E->maxinc;
    info->column_bytes = E->col16 ? 2 : 4;
    info->pad = 0;
    info->bytes_f64 = slots * nd * s * 8 + cols + meta + 16LL * E->NEQ;
    info->bytes_f32 = static_cast<long long>(E->nbrows) * 64 * nd * (4 * nd + (E->col16 ? 2 : 4)) + meta + 8LL * E->NEQ;
    return FEMGPU_OK;
}

extern "C" int femgpu_ebemv(femgpu_ebe *E, const double *d_P, double *d_Q)
{
    FG_CHECK(E && d_P && d_Q && d_P != d_Q, FEMGPU_ERR_ARG, "femgpu_ebemv: bad arguments");
    return launch_ebemv(E->ctx, E, d_P, d_Q);
}

extern "C" int femgpu_ebemv_f32(femgpu_ebe *E, const float *d_P, float *d_Q)
{
    FG_CHECK(E && d_P && d_Q && d_P != d_Q, FEMGPU_ERR_ARG, "femgpu_ebemv_f32: bad arguments");
    return launch_ebemv32(E->ctx, E, d_P, d_Q);
}
