// Small device arrays of a GMRES cycle and the parts of an Arnoldi step that more than one kernel carries: the
// fixed-order sum of per-block partials and the Givens update of a column.
#pragma once

#include <hip/hip_runtime.h>

#include "device_util.h"

namespace fg {

struct GDev {
    double *H;        // (ld x ld) Hessenberg, H[r*ld + c]
    double *c, *s, *e, *y, *hnorm, *invh;   // ld each
    double *scal;     // [0] eps  [1] rho  [2] normb
    int *flags;       // [0] cycle done  [1] steps in cycle
    int ld, kmax;
    double *partials;
    int *h_status;    // host-mapped: per step {done} ; h_rho host-mapped rho per step
    double *h_rho;
    int prec_mode;    // FP32 preconditioner (host side only): 0 exact sweeps, k > 0 Jacobi iterations
    int cgs;          // FP32 inner Arnoldi with classical Gram-Schmidt (host side only)
    int graphs;       // FP32 inner Arnoldi steps replayed from captured hipGraphs (host side only)
};

__device__ __forceinline__ double &Hat(const GDev &G, int r, int c) { return G.H[r * G.ld + c]; }

// Host-mapped doubles (G.h_rho): [0, kmax) the residual estimate after each step, kMapE0 / kMapEps
// the cycle's starting residual and its target, 248..255 norms of the mixed solver.
constexpr int kMapE0 = 246, kMapEps = 247;

constexpr int kMaxBasis = 150;   // largest GMRES basis (make_gdev)

// Givens update of column i and the convergence test (pgmres.c:118-159), with h_{i+1,i} = hn.
// Called by every thread of the block: the block stages the column, the earlier rotations and
// e[i] in LDS with loads issued together, then one thread applies the rotations -- the operations
// of a serial update in the same order -- and stores the results.
static __device__ void givens_column(const GDev &G, int i, double hn)
{
#pragma clang fp contract(off)
    __shared__ double col[kMaxBasis + 1], cs[kMaxBasis], sn[kMaxBasis], ei_s;
    for (int k = threadIdx.x; k <= i; k += blockDim.x) col[k] = Hat(G, k, i);
    for (int k = threadIdx.x; k < i; k += blockDim.x) {
        cs[k] = G.c[k];
        sn[k] = G.s[k];
    }
    if (threadIdx.x == 0) ei_s = G.e[i];
    __syncthreads();
    if (threadIdx.x != 0) return;
    // the entry that the rotations carry along stays in a register and eight rotations' operands are read
    // ahead: an LDS round trip per rotation would be most of this kernel's time
    double run = col[0];
    int j0 = 0;
    for (; j0 + 8 <= i; j0 += 8) {
        double cj[8], sj[8], hj[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            cj[u] = cs[j0 + u];
            sj[u] = sn[j0 + u];
            hj[u] = col[j0 + u + 1];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            Hat(G, j0 + u, i) = cj[u] * run + sj[u] * hj[u];
            run = -sj[u] * run + cj[u] * hj[u];
        }
    }
    for (; j0 < i; ++j0) {
        const double hj = col[j0 + 1];
        Hat(G, j0, i) = cs[j0] * run + sn[j0] * hj;
        run = -sn[j0] * run + cs[j0] * hj;
    }
    const double a = run, b = hn;
    const double r = sqrt(a * a + b * b);
    const double ci = a / r, si = b / r;
    G.c[i] = ci;
    G.s[i] = si;
    Hat(G, i, i) = r;
    Hat(G, i + 1, i) = 0.0;
    const double ei = ei_s;
    G.e[i + 1] = -si * ei;
    G.e[i] = ci * ei;
    const double rho = fabs(G.e[i + 1]);
    const int steps = i + 1;
    const int done = !(rho > G.scal[0]) || (steps >= G.kmax - 1);
    G.scal[1] = rho;
    G.flags[1] = steps;
    G.flags[0] = done;
    __hip_atomic_store(&G.h_rho[i], rho, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(&G.h_status[i], done ? 1 : 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Sum of the nb partials in a fixed order by one block of 256 threads (valid in every thread).
// Each thread adds its entries b, b + 256, ... in order, with four loads issued together.
template <int BS = 256>
__device__ __forceinline__ double sum_partials(const double *partials, int nb, double *red)
{
    double v = 0;
    int b = threadIdx.x;
    for (; b + 3 * BS < nb; b += 4 * BS) {
        const double a0 = partials[b], a1 = partials[b + BS], a2 = partials[b + 2 * BS], a3 = partials[b + 3 * BS];
        v += a0;
        v += a1;
        v += a2;
        v += a3;
    }
    for (; b < nb; b += BS) v += partials[b];
    v = block_sum<BS>(v, red);
    __shared__ double total;
    if (threadIdx.x == 0) total = v;
    __syncthreads();
    return total;
}

// What the EBE product of Arnoldi step i takes over from its neighbours: with nb > 0 the end of step i - 1
// (||w|| from its nb partials, the scaling of the operand by 1 / ||w||, and in a block of its own the Givens
// update of column i - 1), with gnode the nodal block-diagonal preconditioner (node of every group, -1: none).
struct ArnoldiTail {
    GDev G;
    const double *part = nullptr;
    int nb = 0, col = 0;
    const int *gnode = nullptr;
    const float *inv = nullptr;
};

}  // namespace fg
