// Per-element SUPG/PSPG/LSIC assembly of the steady incompressible Navier-Stokes equations
// (P1 u, v, p; 9x9 element blocks) on the device: the Picard tangent and residual of
// Build_K_F_SUPG_PSPG.c:8-671 (the branch its call counter selects below 50000, :466-566) with the
// nodal state of eval_U.c:3-38.
//
// Vertex a has the edge vectors b[a] = (y23, y31, y12)[a] and
// c[a] = (x32, x13, x21)[a]; each entry of the element matrix is the reference's expression for
// its vertex pair, evaluated in the reference's operation order with contraction off (for the
// symmetric terms the reference evaluates the (min, max) pair and reuses it, and so does this
// kernel), so element matrices, residuals, CSR values and right-hand sides are bit-identical.
// Global accumulation is a sum in element order, as for the transport assembly: inside the fused
// kernel where the mesh has its plan and CSR values are wanted, through slot lists otherwise.
#include <algorithm>
#include <cstdint>
#include <vector>

#include "common.h"
#include "device_util.h"

namespace fg {

struct NsIn {
    const double *x, *y, *presc, *u, *fx, *fy;
    const int *type, *invP, *ien;
    int neq;
    double Re;
};

// What an element's rows need of it.
struct NsElem {
    double b[3], c[3], C[3];
    double Area, invArea, visc, tau, tau_l, p, dpdx, dpdy, duxdx, duxdy, duydx, duydy, duxduy, ux, uy, fxB, fyB;
};

// The element of vertices v with the nodal state U[vertex][u, v, p].
__device__ __forceinline__ void ns_element(const NsIn &in, const int (&v)[3], const double (&U)[3][3], NsElem &E)
{
#pragma clang fp contract(off)
    const double third = 1.0 / 3.0;
    const double X0 = in.x[v[0]], X1 = in.x[v[1]], X2 = in.x[v[2]];
    const double Y0 = in.y[v[0]], Y1 = in.y[v[1]], Y2 = in.y[v[2]];
    E.b[0] = Y1 - Y2, E.b[1] = Y2 - Y0, E.b[2] = Y0 - Y1;
    E.c[0] = X2 - X1, E.c[1] = X0 - X2, E.c[2] = X1 - X0;
    const double(&b)[3] = E.b, (&c)[3] = E.c;
    const double TwoA = fabs(c[2] * b[1] - c[1] * b[2]);
    E.Area = 0.5 * TwoA;
    const double invArea = E.invArea = 1.0 / E.Area;
    E.ux = third * (U[0][0] + U[1][0] + U[2][0]);
    E.uy = third * (U[0][1] + U[1][1] + U[2][1]);
    E.duxdx = 0.5 * invArea * (U[0][0] * b[0] + U[1][0] * b[1] + U[2][0] * b[2]);
    E.duxdy = 0.5 * invArea * (U[0][0] * c[0] + U[1][0] * c[1] + U[2][0] * c[2]);
    E.duydx = 0.5 * invArea * (U[0][1] * b[0] + U[1][1] * b[1] + U[2][1] * b[2]);
    E.duydy = 0.5 * invArea * (U[0][1] * c[0] + U[1][1] * c[1] + U[2][1] * c[2]);
    E.duxduy = U[0][0] * b[0] + U[0][1] * c[0] + U[1][0] * b[1] + U[1][1] * c[1] + U[2][0] * b[2] + U[2][1] * c[2];
    E.p = third * (U[0][2] + U[1][2] + U[2][2]);
    E.dpdx = 0.5 * invArea * (U[0][2] * b[0] + U[1][2] * b[1] + U[2][2] * b[2]);
    E.dpdy = 0.5 * invArea * (U[0][2] * c[0] + U[1][2] * c[1] + U[2][2] * c[2]);
#pragma unroll
    for (int a = 0; a < 3; ++a) E.C[a] = 0.5 * invArea * (E.ux * b[a] + E.uy * c[a]);
    // tau_SUPG = tau_PSPG and tau_LSIC (:118-131), rho = 1, viscosity 1/Re
    const double h = sqrt(TwoA), visc = 1. / in.Re, rho = 1.;
    const double nu = visc / rho;
    const double unorm = sqrt(E.ux * E.ux + E.uy * E.uy);
    double auxtau = (2.0 * unorm / h) * (2.0 * unorm / h) + 9.0 * (4.0 * nu / (h * h)) * (4.0 * nu / (h * h));
    auxtau = sqrt(auxtau);
    E.visc = visc;
    E.tau = 1.0 / auxtau;
    E.tau_l = sqrt(nu * nu + (0.5 * h * unorm) * (0.5 * h * unorm));
    E.fxB = in.fx ? third * (in.fx[v[0]] + in.fx[v[1]] + in.fx[v[2]]) : 0.0;
    E.fyB = in.fy ? third * (in.fy[v[0]] + in.fy[v[1]] + in.fy[v[2]]) : 0.0;
}

__device__ __forceinline__ double pick3(const double (&x)[3], int a) { return a == 0 ? x[0] : a == 1 ? x[1] : x[2]; }

// The three rows of vertex a: K[9 d + column], and their residual entries R[d] (:392-464).
__device__ __forceinline__ void ns_vertex(const NsElem &E, int a, double (&K)[27], double (&R)[3])
{
#pragma clang fp contract(off)
    const double third = 1.0 / 3.0, sixth = 1.0 / 6.0, rho = 1., invrho = 1.0 / rho;
    const double(&b)[3] = E.b, (&c)[3] = E.c, (&C)[3] = E.C;
    const double ba = pick3(b, a), ca = pick3(c, a), Ca = pick3(C, a);   // a may differ from lane to lane
    const double Area = E.Area, invArea = E.invArea, visc = E.visc, tau = E.tau, tau_l = E.tau_l;
#pragma unroll
    for (int bb = 0; bb < 3; ++bb) {
        const double Clo = a < bb ? Ca : C[bb], Chi = a < bb ? C[bb] : Ca;
        const double Nb = rho * third * Area * C[bb];
        const double Nd = rho * tau * Area * Clo * Chi;
        const double Kuu = visc * 0.25 * invArea * (2 * ba * b[bb] + ca * c[bb]);
        const double Kvv = visc * 0.25 * invArea * (ba * b[bb] + 2 * ca * c[bb]);
        const double Kuv = visc * 0.25 * invArea * (ca * b[bb]);
        const double Kvu = visc * 0.25 * invArea * (ba * c[bb]);
        const double ks = tau_l * rho * 0.25 * invArea;
        const double Ks_uu = ks * b[bb] * ba, Ks_uv = ks * c[bb] * ba;
        const double Ks_vu = ks * b[bb] * ca, Ks_vv = ks * c[bb] * ca;
        const double Gdu_ab = 0.5 * tau * Ca * b[bb], Gdv_ab = 0.5 * tau * Ca * c[bb];
        const double Gdu_ba = 0.5 * tau * C[bb] * ba, Gdv_ba = 0.5 * tau * C[bb] * ca;
        const double Gphi = invrho * 0.25 * tau * invArea * (ba * b[bb] + ca * c[bb]);
        double *r0 = K + 3 * bb;
        r0[0] = Nb + Nd + Kuu + Ks_uu;
        r0[1] = Kuv + Ks_uv;
        r0[2] = -(sixth * ba + Gdu_ab);
        r0[9] = Kvu + Ks_vu;
        r0[10] = Nb + Nd + Kvv + Ks_vv;
        r0[11] = -(sixth * ca + Gdv_ab);
        r0[18] = sixth * b[bb] + Gdu_ba;
        r0[19] = sixth * c[bb] + Gdv_ba;
        r0[20] = Gphi;
    }
    const double f1 = rho * third * Area * E.fxB, f2 = rho * third * Area * E.fyB;
    const double cvx = E.duxdx * E.ux + E.duxdy * E.uy, cvy = E.duydx * E.ux + E.duydy * E.uy;
    const double Nvx = rho * third * Area * cvx, Nvy = rho * third * Area * cvy;
    const double GTv = third * Area * (E.duxdx + E.duydy);
    const double fdx = rho * tau * Area * Ca * E.fxB, fdy = rho * tau * Area * Ca * E.fyB;
    const double fphi = tau * Area * (ba * E.fxB + ca * E.fyB);
    const double Ndx = rho * tau * Area * Ca * cvx, Ndy = rho * tau * Area * Ca * cvy;
    const double Kvx = 0.5 * visc * (2 * ba * E.duxdx + ca * (E.duxdy + E.duydx));
    const double Kvy = 0.5 * visc * (2 * ca * E.duydy + ba * (E.duxdy + E.duydx));
    const double Ksx = tau_l * rho * 0.25 * invArea * ba * E.duxduy;
    const double Ksy = tau_l * rho * 0.25 * invArea * ca * E.duxduy;
    const double Gvx = 0.5 * E.p * ba, Gvy = 0.5 * E.p * ca;
    const double Gdx = tau * Area * Ca * E.dpdx, Gdy = tau * Area * Ca * E.dpdy;
    const double Nphi = 0.5 * tau * ((E.duxdx * E.ux + E.duxdy * E.uy) * ba + (E.duydx * E.ux + E.duydy * E.uy) * ca);
    const double Gphiv = 0.5 * tau * invrho * (ba * E.dpdx + ca * E.dpdy);
    R[0] = (f1 + fdx) - (Nvx + Ndx + Kvx + Ksx - (Gvx + Gdx));
    R[1] = (f2 + fdy) - (Nvy + Ndy + Kvy + Ksy - (Gvy + Gdy));
    R[2] = fphi - (GTv + Nphi + Gphiv);
}

// The nodal values of three vertices whose unknowns' numbers (-1: prescribed) are q[k].
__device__ __forceinline__ void ns_state(const NsIn &in, const int (&v)[3], const int (&q)[9], double (&U)[3][3])
{
#pragma unroll
    for (int k = 0; k < 9; ++k) U[k / 3][k % 3] = in.neq > 0 ? in.u[max(q[k], 0)] : 0.0;
#pragma unroll
    for (int k = 0; k < 9; ++k)
        if (q[k] < 0) U[k / 3][k % 3] = in.presc[3 * v[k / 3] + k % 3];
}

__global__ __launch_bounds__(256) void k_elem_ns(int nel, NsIn in, double *__restrict__ Ke, double *__restrict__ Res)
{
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= nel) return;
    const int v[3] = {in.ien[3 * e], in.ien[3 * e + 1], in.ien[3 * e + 2]};
    double U[3][3];
    int eq[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) {
        const int i = 3 * v[k / 3] + k % 3;
        eq[k] = in.type[i] > 0 ? in.invP[i] : -1;
    }
    ns_state(in, v, eq, U);
    NsElem E;
    ns_element(in, v, U, E);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        double K[27], R[3];
        ns_vertex(E, a, K, R);
#pragma unroll
        for (int q = 0; q < 27; ++q) Ke[81 * static_cast<size_t>(e) + 27 * a + q] = K[q];
#pragma unroll
        for (int d = 0; d < 3; ++d) Res[9 * static_cast<size_t>(e) + 3 * a + d] = R[d];
    }
}

// CSR values and residual with no element arrays in memory. A block takes a compact patch of nodes with at most
// kNfThreads (element, vertex) incidences and (node, neighbour) pairs. A thread per incidence evaluates the
// element and leaves the three rows of its vertex in an LDS slot (27 entries, 3 residual entries, one word
// of padding against bank conflicts); then a thread per pair sums the 3 x 3 block of the node and the
// neighbour over the elements that hold both, in element order, and a thread per (node, dof) the residual.
// The sums are those of the slot lists in the same order (bit-identical). Three kernels with 81 + 9 doubles
// per element written and read again took 112 us of device time at 257 x 257 nodes (135 us a call); this one takes 29, of which a
// third is arithmetic and the rest waits in the chains node -> state -> element and pair -> codes -> slots.
// Patches of 64, 128, 192 and 256 incidences: 29.1, 28.8, 28.5, 29.7 us.
constexpr int kNfThreads = 128, kNfSlot = 31;
// what the plan packs: a node's place in its patch in 8 bits, LDS offsets of contributions and a patch's first codes
// (three per incidence) in 16
static_assert(kNfThreads <= 256 && kNfSlot * kNfThreads <= 65536 && 3 * kNfThreads <= 65536, "packed fields of the plan");

__global__ __launch_bounds__(kNfThreads) void k_ns_fused(int nblocks, NsIn in, const int4 *__restrict__ bptr,
                                                         const int4 *__restrict__ inc, const int4 *__restrict__ eqs,
                                                         const int4 *__restrict__ node, const uint2 *__restrict__ pair,
                                                         const unsigned short *__restrict__ code, int nnz,
                                                         double *__restrict__ AA, double *__restrict__ F)
{
#pragma clang fp contract(off)
    extern __shared__ double slots[];
    const int w = xcd_block(), t = threadIdx.x;
    if (w >= nblocks) return;
    if (w == 0 && t == 0) {
        AA[nnz] = 0.0;
        F[in.neq] = 0.0;
    }
    const int4 p0 = bptr[w], p1 = bptr[w + 1];   // first {incidence, pair, code, 2 x node}
    const bool has = t < p1.y - p0.y;
    // {CSR positions of the three columns (255: none) and node, 8 bits each}, {first code, codes, 16 bits each}
    uint2 pr = make_uint2(0, 0);
    int4 nd = make_int4(-1, -1, -1, 0);   // first CSR slot of the three rows (-1: none), LDS slots
    if (has) {
        pr = pair[p0.y + t];
        nd = node[2 * (p0.w + (pr.x >> 24))];
    }
    if (t < p1.x - p0.x) {
        const int4 A = inc[p0.x + t];   // {v0, v1, v2, vertex}
        const int v[3] = {A.x, A.y, A.z};
        int eq[9];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const int4 q = eqs[v[a]];
            eq[3 * a] = q.x, eq[3 * a + 1] = q.y, eq[3 * a + 2] = q.z;
        }
        double U[3][3], K[27], R[3];
        ns_state(in, v, eq, U);
        NsElem E;
        ns_element(in, v, U, E);
        ns_vertex(E, A.w, K, R);
        double *s = slots + kNfSlot * t;
#pragma unroll
        for (int q = 0; q < 27; ++q) s[q] = K[q];
#pragma unroll
        for (int d = 0; d < 3; ++d) s[27 + d] = R[d];
    }
    __syncthreads();
    if (has) {
        const int first = p0.z + (pr.y & 0xffffu), cnt = pr.y >> 16;
        double S[9] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        for (int c = 0; c < cnt; c += 2) {
            const bool two = c + 1 < cnt;
            const double *s0 = slots + code[first + c], *s1 = slots + code[first + (two ? c + 1 : c)];
            double a[9], b[9];
#pragma unroll
            for (int k = 0; k < 9; ++k) a[k] = s0[9 * (k / 3) + k % 3], b[k] = s1[9 * (k / 3) + k % 3];
#pragma unroll
            for (int k = 0; k < 9; ++k) {
                S[k] += a[k];
                if (two) S[k] += b[k];
            }
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const int row = d == 0 ? nd.x : d == 1 ? nd.y : nd.z;
            if (row < 0) continue;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const unsigned pos = (pr.x >> (8 * k)) & 255u;
                if (pos != 255u) AA[row + static_cast<int>(pos)] = S[3 * d + k];
            }
        }
    }
    for (int q = t; q < 3 * (p1.w - p0.w); q += kNfThreads) {
        const int ln = q / 3, d = q - 3 * ln;
        const int4 n = node[2 * (p0.w + ln)], e4 = node[2 * (p0.w + ln) + 1];
        const int eq = d == 0 ? e4.x : d == 1 ? e4.y : e4.z, s0 = n.w & 0xffff, cnt = n.w >> 16;
        if (eq < 0) continue;
        double f = 0.0;
        for (int c = 0; c < cnt; ++c) f += slots[kNfSlot * (s0 + c) + 27 + d];
        F[eq] = f;
    }
}

// The fused kernel's plan from the mesh's host arrays. ok when every unknown belongs to one dof of one node,
// every CSR slot to one row (contiguous rows), a node's rows have the same columns in the same positions
// (at most 255), each position belongs to one neighbour, and a node has at most 32 elements; else the slot
// lists.
static int build_ns_fused(femgpu_mesh *M, const int *ien, const int *type, const int *invP, const int *lm, const int *scheme)
{
    M->nf_ok = false;
    const int nn = M->nnodes, nel = M->nel, neq = M->neq, nnz = M->nnz;
    if (neq == 0 || nel == 0 || nnz == 0) return FEMGPU_OK;
    std::vector<int> owner(neq, -1), deq(static_cast<size_t>(nn) * 3);
    for (int k = 0; k < 3 * nn; ++k) {
        deq[k] = type[k] > 0 ? invP[k] : -1;
        if (deq[k] < 0) continue;
        if (owner[deq[k]] >= 0) return FEMGPU_OK;
        owner[deq[k]] = k;
    }
    // incidences of every node with unknowns, in element order; lm must be the node numbering
    std::vector<int> iptr(static_cast<size_t>(nn) + 1, 0);
    for (size_t ea = 0; ea < 3 * static_cast<size_t>(nel); ++ea) {
        const int v = ien[ea];
        bool any = false;
        for (int d = 0; d < 3; ++d) {
            const int q = deq[3 * v + d];
            if (lm[3 * ea + d] != (q >= 0 ? q : neq)) return FEMGPU_OK;
            any = any || q >= 0;
        }
        if (any) ++iptr[v + 1];
    }
    int maxinc = 0;
    for (int v = 0; v < nn; ++v) {
        maxinc = std::max(maxinc, iptr[v + 1]);
        iptr[v + 1] += iptr[v];
    }
    if (maxinc > 32) return FEMGPU_OK;
    std::vector<int> inc(static_cast<size_t>(iptr[nn])), fill(iptr.begin(), iptr.end() - 1);
    for (size_t ea = 0; ea < 3 * static_cast<size_t>(nel); ++ea)
        if (iptr[ien[ea] + 1] > iptr[ien[ea]]) inc[fill[ien[ea]]++] = static_cast<int>(ea);
    // rows: first and last slot of every unknown; every slot in exactly one row
    std::vector<int> rfirst(neq, INT32_MAX), rlast(neq, -1);
    for (size_t ea = 0; ea < 3 * static_cast<size_t>(nel); ++ea)
        for (int d = 0; d < 3; ++d) {
            const int q = lm[3 * ea + d], *sc = scheme + 9 * (3 * ea + d);
            for (int b = 0; b < 9; ++b) {
                if (sc[b] >= nnz) continue;
                if (q >= neq) return FEMGPU_OK;
                rfirst[q] = std::min(rfirst[q], sc[b]);
                rlast[q] = std::max(rlast[q], sc[b]);
            }
        }
    std::vector<char> seen(static_cast<size_t>(nnz), 0);
    long long covered = 0;
    for (int q = 0; q < neq; ++q) {
        if (rlast[q] < 0 || rlast[q] - rfirst[q] >= 255) return FEMGPU_OK;
        for (int k = rfirst[q]; k <= rlast[q]; ++k) {
            if (seen[k]) return FEMGPU_OK;
            seen[k] = 1;
        }
        covered += rlast[q] - rfirst[q] + 1;
    }
    if (covered != nnz) return FEMGPU_OK;
    // a node's rows share columns: same length, same relative positions for every incidence; the positions of
    // an element row are distinct
    const auto row_of = [&](int v, int d) { return deq[3 * v + d]; };
    const auto first_dof = [&](int v) { return row_of(v, 0) >= 0 ? 0 : row_of(v, 1) >= 0 ? 1 : 2; };
    for (int v = 0; v < nn; ++v) {
        if (iptr[v] == iptr[v + 1]) {
            for (int d = 0; d < 3; ++d)
                if (row_of(v, d) >= 0) return FEMGPU_OK;
            continue;
        }
        const int d0 = first_dof(v), q0 = row_of(v, d0), len = rlast[q0] - rfirst[q0];
        for (int d = d0 + 1; d < 3; ++d) {
            const int q = row_of(v, d);
            if (q < 0) continue;
            if (rlast[q] - rfirst[q] != len) return FEMGPU_OK;
            for (int p = iptr[v]; p < iptr[v + 1]; ++p)
                for (int b = 0; b < 9; ++b) {
                    const int s0 = scheme[9 * (3 * static_cast<size_t>(inc[p]) + d0) + b];
                    const int s1 = scheme[9 * (3 * static_cast<size_t>(inc[p]) + d) + b];
                    if ((s0 < nnz) != (s1 < nnz) || (s0 < nnz && s0 - rfirst[q0] != s1 - rfirst[q])) return FEMGPU_OK;
                }
        }
    }
    // (node, neighbour) pairs: the elements that hold both, and the CSR positions of the neighbour's three
    // columns in the node's rows, the same for every element; each position belongs to one pair
    struct Pair { int vtx, pos[3], first, cnt; };
    std::vector<Pair> prs;
    std::vector<int> prp(static_cast<size_t>(nn) + 1, 0), pcode, at(nn, -1), held;
    std::vector<char> used(256);
    prs.reserve(static_cast<size_t>(nel) * 4);
    pcode.reserve(static_cast<size_t>(nel) * 9);
    for (int v = 0; v < nn; ++v) {
        const size_t f0 = prs.size();
        held.clear();
        if (iptr[v] < iptr[v + 1]) {
            const int d0 = first_dof(v), q0 = row_of(v, d0), len = rlast[q0] - rfirst[q0] + 1;
            for (int p = iptr[v]; p < iptr[v + 1]; ++p)
                for (int b = 0; b < 3; ++b) {
                    const int u = ien[inc[p] / 3 * 3 + b];
                    const int *sc = scheme + 9 * (3 * static_cast<size_t>(inc[p]) + d0) + 3 * b;
                    int pos[3];
                    for (int k = 0; k < 3; ++k) pos[k] = sc[k] < nnz ? sc[k] - rfirst[q0] : 255;
                    if (at[u] < 0) {
                        at[u] = static_cast<int>(prs.size());
                        held.push_back(u);
                        prs.push_back({u, {pos[0], pos[1], pos[2]}, 0, 0});
                    }
                    Pair &q = prs[at[u]];
                    if (q.pos[0] != pos[0] || q.pos[1] != pos[1] || q.pos[2] != pos[2]) return FEMGPU_OK;
                    ++q.cnt;
                }
            std::fill(used.begin(), used.end(), 0);
            int named = 0;
            for (size_t i = f0; i < prs.size(); ++i)
                for (int k = 0; k < 3; ++k) {
                    const int pos = prs[i].pos[k];
                    if (pos == 255) continue;
                    if (used[pos]) return FEMGPU_OK;
                    used[pos] = 1;
                    ++named;
                }
            if (named != len) return FEMGPU_OK;
            int at0 = static_cast<int>(pcode.size());
            for (size_t i = f0; i < prs.size(); ++i) {
                prs[i].first = at0;
                at0 += prs[i].cnt;
                prs[i].cnt = 0;
            }
            pcode.resize(at0);
            for (int p = iptr[v]; p < iptr[v + 1]; ++p)
                for (int b = 0; b < 3; ++b) {
                    Pair &q = prs[at[ien[inc[p] / 3 * 3 + b]]];
                    pcode[q.first + q.cnt++] = kNfSlot * (p - iptr[v]) + 3 * b;
                }
            for (int u : held) at[u] = -1;
        }
        prp[v + 1] = static_cast<int>(prs.size());
        if (prp[v + 1] - prp[v] > kNfThreads) return FEMGPU_OK;
    }
    // patches: breadth-first over nodes that share elements
    std::vector<int> blk(nn, -1), order;
    std::vector<int4> bptr{make_int4(0, 0, 0, 0)}, ent, node, eqs(nn);
    std::vector<uint2> pair;
    std::vector<unsigned short> code;
    ent.reserve(inc.size());
    pair.reserve(prs.size());
    code.reserve(pcode.size());
    for (int v = 0; v < nn; ++v) eqs[v] = make_int4(row_of(v, 0), row_of(v, 1), row_of(v, 2), 0);
    int slots_max = 0;
    for (int seed = 0; seed < nn; ++seed) {
        if (blk[seed] >= 0 || iptr[seed] == iptr[seed + 1]) continue;
        const size_t start = order.size(), code0 = code.size();
        int slots = iptr[seed + 1] - iptr[seed], pairs = prp[seed + 1] - prp[seed];
        order.push_back(seed);
        blk[seed] = 1;
        for (size_t h = start; h < order.size(); ++h)
            for (int q = prp[order[h]]; q < prp[order[h] + 1]; ++q) {
                const int u = prs[q].vtx, su = iptr[u + 1] - iptr[u], pu = prp[u + 1] - prp[u];
                if (su == 0 || blk[u] >= 0 || slots + su > kNfThreads || pairs + pu > kNfThreads) continue;
                blk[u] = 1;
                order.push_back(u);
                slots += su;
                pairs += pu;
            }
        int ns = 0;
        for (size_t h = start; h < order.size(); ++h) {
            const int v = order[h];
            int rs[3];
            for (int d = 0; d < 3; ++d) rs[d] = row_of(v, d) >= 0 ? rfirst[row_of(v, d)] : -1;
            node.push_back(make_int4(rs[0], rs[1], rs[2], ns | ((iptr[v + 1] - iptr[v]) << 16)));
            node.push_back(eqs[v]);
            for (int q = prp[v]; q < prp[v + 1]; ++q) {
                const Pair &P = prs[q];
                pair.push_back(make_uint2(static_cast<unsigned>(P.pos[0] | P.pos[1] << 8 | P.pos[2] << 16) |
                                              static_cast<unsigned>(h - start) << 24,
                                          static_cast<unsigned>(code.size() - code0) | static_cast<unsigned>(P.cnt) << 16));
                for (int i = 0; i < P.cnt; ++i) code.push_back(static_cast<unsigned short>(kNfSlot * ns + pcode[P.first + i]));
            }
            for (int p = iptr[v]; p < iptr[v + 1]; ++p) {
                const int *ev = ien + inc[p] / 3 * 3;
                ent.push_back(make_int4(ev[0], ev[1], ev[2], inc[p] % 3));
            }
            ns += iptr[v + 1] - iptr[v];
        }
        slots_max = std::max(slots_max, ns);
        bptr.push_back(make_int4(static_cast<int>(ent.size()), static_cast<int>(pair.size()), static_cast<int>(code.size()),
                                 static_cast<int>(order.size())));
    }
    hipStream_t st = M->ctx->stream;
    FG_TRY(M->nf_bptr.upload(bptr.data(), bptr.size(), st));
    FG_TRY(M->nf_inc.upload(ent.data(), ent.size(), st));
    FG_TRY(M->nf_eqs.upload(eqs.data(), eqs.size(), st));
    FG_TRY(M->nf_node.upload(node.data(), node.size(), st));
    FG_TRY(M->nf_pair.upload(pair.data(), pair.size(), st));
    FG_TRY(M->nf_code.upload(code.data(), code.size(), st));
    FG_HIP(hipStreamSynchronize(st));   // the host arrays end here
    M->nf_blocks = static_cast<int>(bptr.size()) - 1;
    M->nf_slots = slots_max;
    M->nf_ok = true;
    return FEMGPU_OK;
}

// F[I] = sum of the residual entries of unknown I in element order (F[lm] += Res, :655-658);
// F[NEQ] = 0. src entries index the per-element residual array (e*s+i).
__global__ void k_rhs_gather(int NEQ, const int *__restrict__ dst, const int *__restrict__ ptr,
                             const int *__restrict__ src, const double *__restrict__ Res, double *__restrict__ F)
{
#pragma clang fp contract(off)
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k > NEQ) return;
    if (k == NEQ) {
        F[NEQ] = 0.0;
        return;
    }
    F[dst[k]] = gather_sum<8>(src, Res, ptr[k], ptr[k + 1]);
}

__global__ void k_aa_gather_blocks(int nnz, const int *__restrict__ dst, const int *__restrict__ ptr,
                                   const int *__restrict__ src, const double *__restrict__ Ke, double *__restrict__ AA)
{
#pragma clang fp contract(off)
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k > nnz) return;
    if (k == nnz) {
        AA[nnz] = 0.0;
        return;
    }
    AA[dst[k]] = gather_sum<8>(src, Ke, ptr[k], ptr[k + 1]);
}

}  // namespace fg

using namespace fg;

namespace fg {

// Device mesh for element blocks of s = 3*ndof dofs (ndof = 3: Navier-Stokes, 4: Euler): per-dof
// Type/invP_id/prescribed values, lm[nel*s], the residual gather map (unknown -> e*s+i in element
// order) and, with a slot table scheme[nel*s*s], the CSR value gather map (slot -> e*s*s+q).
int block_mesh_create(femgpu_ctx *ctx, int ndof, int nnodes, int nel, int neq, const double *x, const double *y,
                      const int *type, const int *invP, const double *presc, const int *ien, const int *lm,
                      const int *scheme, int nnz, femgpu_mesh **out)
{
    const int sb = 3 * ndof, ss = sb * sb;
    FG_CHECK(ctx && nnodes > 0 && nel >= 0 && neq >= 0 && x && y && type && invP && presc && ien && lm && out,
             FEMGPU_ERR_ARG, "mesh create: bad arguments");
    for (size_t q = 0; q < static_cast<size_t>(nel) * 3; ++q)
        FG_CHECK(ien[q] >= 0 && ien[q] < nnodes, FEMGPU_ERR_ARG, "mesh create: vertex %d out of range", ien[q]);
    for (size_t k = 0; k < static_cast<size_t>(nnodes) * ndof; ++k)
        FG_CHECK(type[k] == 0 || (invP[k] >= 0 && invP[k] < neq), FEMGPU_ERR_ARG,
                 "mesh create: dof %zu is an unknown with invP_id %d out of range", k, invP[k]);
    for (size_t q = 0; q < static_cast<size_t>(nel) * sb; ++q)
        FG_CHECK(lm[q] >= 0 && lm[q] <= neq, FEMGPU_ERR_ARG, "mesh create: lm entry %d out of range", lm[q]);
    auto *M = new femgpu_mesh();
    M->ctx = ctx;
    M->ndof = ndof;
    M->nnodes = nnodes;
    M->nel = nel;
    M->neq = neq;
    M->nnz = scheme ? nnz : 0;
    hipStream_t s = ctx->stream;
    int rc = FEMGPU_OK;
    auto up = [&](auto &buf, auto *h, size_t n) {
        if (rc == FEMGPU_OK) rc = buf.upload(h, n, s);
    };
    const size_t nd = static_cast<size_t>(nnodes) * ndof;
    up(M->x, x, nnodes);
    up(M->y, y, nnodes);
    up(M->ubc, presc, nd);
    up(M->type, type, nd);
    up(M->invP, invP, nd);
    up(M->ien, ien, static_cast<size_t>(nel) * 3);
    up(M->lm, lm, static_cast<size_t>(nel) * sb);
    std::vector<std::pair<int, int>> pairs;
    pairs.reserve(static_cast<size_t>(nel) * sb);
    for (int e = 0; e < nel; ++e)
        for (int i = 0; i < sb; ++i) {
            const int I = lm[static_cast<size_t>(sb) * e + i];
            if (I < neq) pairs.emplace_back(I, sb * e + i);
        }
    std::vector<int> ptr, src, dst;
    csr_map(neq, pairs, ptr, src, dst);
    up(M->rhs_ptr, ptr.data(), ptr.size());
    up(M->rhs_src, src.data(), src.size());
    up(M->rhs_dst, dst.data(), dst.size());
    // the uploads are asynchronous: the host lists must outlive them (the aa map uses new vectors)
    std::vector<int> aptr, asrc, adst;
    if (rc == FEMGPU_OK && scheme) {
        for (size_t q = 0; q < static_cast<size_t>(nel) * ss; ++q)
            if (scheme[q] < 0 || scheme[q] > nnz) rc = FEMGPU_ERR_ARG;
        if (rc == FEMGPU_ERR_ARG) set_error("mesh create: scheme slot out of range");
        if (rc == FEMGPU_OK && static_cast<long long>(nel) * ss >= (1LL << 31)) {
            set_error("mesh create: too many element entries");
            rc = FEMGPU_ERR_ARG;
        }
        if (rc == FEMGPU_OK && ndof == 3) rc = build_ns_fused(M, ien, type, invP, lm, scheme);
        M->has_scheme = rc == FEMGPU_OK;
        if (rc == FEMGPU_OK && !M->nf_ok) {   // slot lists, where the fused assembly does not apply
            pairs.clear();
            for (int e = 0; e < nel; ++e)
                for (int q = 0; q < ss; ++q) {
                    const int slot = scheme[static_cast<size_t>(ss) * e + q];
                    if (slot < nnz) pairs.emplace_back(slot, ss * e + q);
                }
            csr_map(nnz, pairs, aptr, asrc, adst);
            up(M->aa_ptr, aptr.data(), aptr.size());
            up(M->aa_src, asrc.data(), asrc.size());
            up(M->aa_dst, adst.data(), adst.size());
        }
    }
    if (rc == FEMGPU_OK) rc = M->fe.alloc(static_cast<size_t>(nel) * sb);
    if (rc == FEMGPU_OK) rc = M->ke.alloc(static_cast<size_t>(nel) * ss);
    if (rc == FEMGPU_OK && hipStreamSynchronize(s) != hipSuccess) rc = FEMGPU_ERR_HIP;
    if (rc != FEMGPU_OK) {
        delete M;
        return rc;
    }
    *out = M;
    return FEMGPU_OK;
}

int launch_block_gathers(femgpu_mesh *M, const double *Ke, double *F, double *AA)
{
    femgpu_ctx *ctx = M->ctx;
    k_rhs_gather<<<(M->neq + 1 + 255) / 256, 256, 0, ctx->stream>>>(M->neq, M->rhs_dst.p, M->rhs_ptr.p, M->rhs_src.p,
                                                                    M->fe.p, F);
    FG_HIP(hipGetLastError());
    if (AA) {
        k_aa_gather_blocks<<<(M->nnz + 1 + 255) / 256, 256, 0, ctx->stream>>>(M->nnz, M->aa_dst.p, M->aa_ptr.p,
                                                                              M->aa_src.p, Ke, AA);
        FG_HIP(hipGetLastError());
    }
    return FEMGPU_OK;
}

}  // namespace fg

extern "C" int femgpu_ns_mesh_create(femgpu_ctx *ctx, int nnodes, int nel, int neq, const double *x, const double *y,
                                     const int *type3, const int *invP3, const double *presc3, const int *ien,
                                     const int *lm, const int *scheme, int nnz, femgpu_mesh **out)
{
    return block_mesh_create(ctx, 3, nnodes, nel, neq, x, y, type3, invP3, presc3, ien, lm, scheme, nnz, out);
}

extern "C" int femgpu_assemble_ns(femgpu_mesh *M, double Re, const double *d_u, const double *d_fx,
                                  const double *d_fy, double *d_Ke, double *d_F, double *d_AA)
{
    FG_CHECK(M && d_u && d_F && Re > 0.0, FEMGPU_ERR_ARG, "femgpu_assemble_ns: bad arguments");
    FG_CHECK(M->ndof == 3, FEMGPU_ERR_STATE, "femgpu_assemble_ns: not a Navier-Stokes mesh");
    FG_CHECK(!d_AA || M->has_scheme, FEMGPU_ERR_STATE, "femgpu_assemble_ns: mesh created without a CSR slot table");
    femgpu_ctx *ctx = M->ctx;
    double *Ke = d_Ke ? d_Ke : M->ke.p;
    NsIn in;
    in.x = M->x.p;
    in.y = M->y.p;
    in.presc = M->ubc.p;
    in.u = d_u;
    in.fx = d_fx;
    in.fy = d_fy;
    in.type = M->type.p;
    in.invP = M->invP.p;
    in.ien = M->ien.p;
    in.neq = M->neq;
    in.Re = Re;
    const bool fused = d_AA && M->nf_ok;
    if (fused) {
        const size_t lds = sizeof(double) * kNfSlot * static_cast<size_t>(M->nf_slots);
        k_ns_fused<<<xcd_grid(M->nf_blocks), kNfThreads, lds, ctx->stream>>>(
            M->nf_blocks, in, M->nf_bptr.p, M->nf_inc.p, M->nf_eqs.p, M->nf_node.p, M->nf_pair.p, M->nf_code.p, M->nnz, d_AA,
            d_F);
        FG_HIP(hipGetLastError());
        if (!d_Ke) return FEMGPU_OK;
    }
    if (M->nel > 0) {
        k_elem_ns<<<(M->nel + 255) / 256, 256, 0, ctx->stream>>>(M->nel, in, Ke, M->fe.p);
        FG_HIP(hipGetLastError());
    }
    if (fused) return FEMGPU_OK;
    return launch_block_gathers(M, Ke, d_F, d_AA);
}
