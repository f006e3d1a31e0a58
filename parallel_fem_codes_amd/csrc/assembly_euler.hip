// Per-element SUPG assembly of the 2D compressible Euler equations (P1, conservative variables
// rho, rho u, rho v, rho E; 12x12 element blocks) on the device: Ae = Me + alpha*dt*Ke and the
// residual R = -(Me dU + Ke U) of Build_M_K_F_SUPG.c:6-1057, with eval_U_dU.c:3-55, the flux
// Jacobians of Ax_Ay_calculations.c (dimensionless :3-53 or dimensional :55-99) and the CAU
// shock-capture coefficient of Delta_CAU.c:4-83.
//
// The element matrices are built row by row: for dof row i of vertex a, the Galerkin/SUPG convection
// block C_a = (b_a Ax + c_a Ay)/6, the SUPG products b_a (AxAx, AxAy) + c_a (AyAx, AyAy) and the CAU
// coupling give every column, and the row's residual and Ae entries are formed on the spot. Each
// quantity is evaluated in the reference's operation order with contraction off; the reference's
// hand-expanded 4x4 products skip only terms with a structural zero factor, so the dense products
// used here have equal values.
// Global accumulation is the element-order gather shared with the Navier-Stokes assembly.
#include "common.h"
#include "device_util.h"

namespace fg {

struct EulerIn {
    const double *x, *y, *presc, *u, *du;
    const int *type, *invP, *ien;
    int neq;
    femgpu_euler_problem pb;
};

__device__ __forceinline__ void euler_jacobians_dev(const femgpu_euler_problem &p, const double Ub[4],
                                                    double Ax[4][4], double Ay[4][4])
{
#pragma clang fp contract(off)
    const double g = p.gamma;
    const double v1 = Ub[1] / Ub[0], v2 = Ub[2] / Ub[0], E = Ub[3] / Ub[0];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            Ax[i][j] = 0.0;
            Ay[i][j] = 0.0;
        }
    Ax[0][1] = 1.0;
    Ay[0][2] = 1.0;
    Ax[2][0] = -v1 * v2;
    Ax[2][1] = v2;
    Ax[2][2] = v1;
    Ax[1][1] = (3.0 - g) * v1;
    Ax[1][2] = -(g - 1.0) * v2;
    Ax[3][3] = g * v1;
    Ay[1][1] = v2;
    Ay[1][2] = v1;
    Ay[2][1] = -(g - 1.0) * v1;
    Ay[2][2] = (3.0 - g) * v2;
    Ay[3][3] = g * v2;
    if (p.dimensionless) {
        const double nv = v1 * v1 + v2 * v2, eps2 = p.Mach * p.Mach;
        Ax[1][0] = -(v1 * v1) + ((g - 1) * nv * 0.5);
        Ax[1][3] = (g - 1.0) / eps2;
        Ax[3][0] = -v1 * (g * E - ((g - 1.0) * eps2 * nv));
        Ax[3][1] = g * E - (g - 1.0) * eps2 * (0.5 * nv + v1 * v1);
        Ax[3][2] = -(g - 1.0) * eps2 * v1 * v2;
        Ay[2][0] = -(v2 * v2) + (((g - 1.0) * nv * 0.5));
        Ay[3][0] = -v2 * (g * E - (g - 1.0) * eps2 * nv);
        Ay[3][2] = g * E - (g - 1.0) * eps2 * (0.5 * nv + v2 * v2);
    } else {
        const double rho = Ub[0], nU = (Ub[1] * Ub[1]) + (Ub[2] * Ub[2]);
        Ax[1][0] = -(v1 * v1) + (((g - 1) * nU * 0.5) / (rho * rho));
        Ax[1][3] = g - 1.0;
        Ax[3][0] = (-g * v1 * E) + ((g - 1.0) * v1 * (nU / (rho * rho)));
        Ax[3][1] = (g * E) - ((g - 1.0) * 0.5 * ((nU / (rho * rho)) + (2.0 * v1 * v1)));
        Ax[3][2] = -((g - 1.0) * v1 * v2);
        Ay[2][0] = -(v2 * v2) + (((g - 1.0) * nU * 0.5) / (rho * rho));
        Ay[3][0] = (-g * v2 * E) + (((g - 1.0) * v2 * nU) / (rho * rho));
        Ay[3][2] = (g * E) - ((g - 1.0) * 0.5 * ((nU / (rho * rho)) + (2.0 * v2 * v2)));
    }
    Ay[1][0] = Ax[2][0];
    Ay[2][3] = Ax[1][3];
    Ay[3][1] = Ax[3][2];
}

// w^T A0 w grouped as Delta_CAU.c:39-73 groups it.
__device__ __forceinline__ double a0_form_dev(const double A0[4][4], const double w[4])
{
#pragma clang fp contract(off)
    return w[0] * (A0[0][0] * w[0] + 2.0 * A0[0][1] * w[1] + 2.0 * A0[0][2] * w[2] + 2.0 * A0[0][3] * w[3]) +
           w[1] * (A0[1][1] * w[1] + 2.0 * A0[1][2] * w[2] + 2.0 * A0[1][3] * w[3]) +
           w[2] * (A0[2][2] * w[2] + 2.0 * A0[2][3] * w[3]) + w[3] * A0[3][3] * w[3];
}

// Orders a wavefront's LDS writes before its later LDS reads of other lanes' words, and the reverse.
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Component j of a quad's value: lane j of each four lanes to all four.
template <int J>
__device__ __forceinline__ double quad_bcast(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(b), J * 0x55, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(b >> 32), J * 0x55, 0xf, 0xf, true);
    return __longlong_as_double(static_cast<long long>(static_cast<unsigned>(lo)) | (static_cast<long long>(hi) << 32));
}
__device__ __forceinline__ void quad_all(double v, double (&all)[4])
{
    all[0] = quad_bcast<0>(v);
    all[1] = quad_bcast<1>(v);
    all[2] = quad_bcast<2>(v);
    all[3] = quad_bcast<3>(v);
}
__device__ __forceinline__ double sel4(int i, double v0, double v1, double v2, double v3)
{
    return i < 2 ? (i == 0 ? v0 : v1) : (i == 2 ? v2 : v3);
}

// Four lanes per element, lane i of a quad on dof i: it loads its dof of the three vertices, forms its
// component of the element's state and gradients, exchanges components with the quad (DPP moves), evaluates
// the rest of the element's state, and forms rows i, 4 + i and 8 + i. What bounds it: the 1 152 bytes an
// element writes (184 MB at 401 x 201 nodes), about forty FP64 divisions (half of them shared out over the
// quad) and 2 900 FP64 operations of entries. One thread per element held the whole element in registers
// (one wavefront per SIMD) and stored its rows 64 cache lines per instruction: 105 us. Here a wavefront turns
// its rows through LDS and stores runs of 384 bytes: 74 us (160 000 elements; about 2 200 instructions a
// lane, 36 us of issue at two wavefronts per SIMD).
__global__ __launch_bounds__(256, 2) void k_elem_euler(int nel, EulerIn in, double *__restrict__ Ae, double *__restrict__ Res)
{
#pragma clang fp contract(off)
    __shared__ double turn_all[4 * 64 * 13];
    const int l = threadIdx.x & 63, i = l & 3;
    const int ew = xcd_block() * 64 + static_cast<int>(threadIdx.x >> 6) * 16;   // the wavefront's 16 elements
    if (ew >= nel) return;
    const int n = min(16, nel - ew), e = ew + min(l >> 2, n - 1);   // idle quads repeat the last element
    double *turn = turn_all + (threadIdx.x >> 6) * (64 * 13);
    const femgpu_euler_problem &p = in.pb;
    const double third = 1.0 / 3.0, sixth = 1.0 / 6.0;
    const double gamma = p.gamma, alpha = p.alpha, delta_t = p.dt;
    int v[3], eq[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) v[a] = in.ien[3 * e + a];
    const double X0 = in.x[v[0]], X1 = in.x[v[1]], X2 = in.x[v[2]];
    const double Y0 = in.y[v[0]], Y1 = in.y[v[1]], Y2 = in.y[v[2]];
    // this lane's dof of the vertices: mark, number and prescribed value, then state
    double U[3], dU[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int q = 4 * v[a] + i;
        eq[a] = in.type[q] > 0 ? in.invP[q] : -1;
        U[a] = in.presc[q];
        dU[a] = 0.0;
    }
    if (in.neq > 0)   // else every dof is prescribed
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const int q = eq[a] >= 0 ? eq[a] : 0;
            const double un = in.u[q], dn = in.du[q];
            U[a] = eq[a] >= 0 ? un : U[a];
            dU[a] = eq[a] >= 0 ? dn : 0.0;
        }
    const double b[3] = {Y1 - Y2, Y2 - Y0, Y0 - Y1};
    const double c[3] = {X2 - X1, X0 - X2, X1 - X0};
    const double twoArea = fabs(c[2] * b[1] - c[1] * b[2]);
    const double Area = 0.5 * twoArea;
    const double gxi = (U[0] * b[0] + U[1] * b[1] + U[2] * b[2]) / twoArea;
    const double gyi = (U[0] * c[0] + U[1] * c[1] + U[2] * c[2]) / twoArea;
    double Ub[4], gUx[4], gUy[4];
    quad_all((U[0] + U[1] + U[2]) * third, Ub);
    quad_all(gxi, gUx);
    quad_all(gyi, gUy);
    const double v1 = Ub[1] / Ub[0], v2 = Ub[2] / Ub[0], E = Ub[3] / Ub[0];
    double Ax[4][4], Ay[4][4];
    euler_jacobians_dev(p, Ub, Ax, Ay);
    // CAU coefficient (Delta_CAU.c) with the entropy-variable metric A0^-1 (:134-160)
    double delta = 0.0;
    if (p.shock) {
        double dUb[4], gkx[4], gky[4], LUh[4];
        quad_all((dU[0] + dU[1] + dU[2]) * third, dUb);
        quad_all((b[0] * gxi + c[0] * gyi) / twoArea, gkx);
        quad_all((b[1] * gxi + c[1] * gyi) / twoArea, gky);
        const double nU = (Ub[1] * Ub[1]) + (Ub[2] * Ub[2]);
        const double rho_i = Ub[3] - ((nU * 0.5) / Ub[0]);
        const double V2 = Ub[1] / rho_i, V3 = Ub[2] / rho_i, V4 = (-Ub[0]) / rho_i;
        const double rhoi_e = -1.0 / (rho_i * V4);
        const double k1 = (V2 * V2 + V3 * V3) * 0.5 / V4;
        double A0[4][4];
        A0[0][0] = rhoi_e * (k1 * k1 + gamma);
        A0[0][1] = rhoi_e * (k1 * V2);
        A0[0][2] = rhoi_e * (k1 * V3);
        A0[0][3] = rhoi_e * ((k1 + 1.0) * V4);
        A0[1][1] = rhoi_e * (V2 * V2 - V4);
        A0[1][2] = rhoi_e * (V2 * V3);
        A0[1][3] = rhoi_e * (V2 * V4);
        A0[2][2] = rhoi_e * (V3 * V3 - V4);
        A0[2][3] = rhoi_e * (V3 * V4);
        A0[3][3] = rhoi_e * V4 * V4;
        double AgUx[4], AgUy[4];
        AgUx[0] = gUx[1];
        AgUx[1] = Ax[1][0] * gUx[0] + Ax[1][1] * gUx[1] + Ax[1][2] * gUx[2] + Ax[1][3] * gUx[3];
        AgUx[2] = Ax[2][0] * gUx[0] + Ax[2][1] * gUx[1] + Ax[2][2] * gUx[2];
        AgUx[3] = Ax[3][0] * gUx[0] + Ax[3][1] * gUx[1] + Ax[3][2] * gUx[2] + Ax[3][3] * gUx[3];
        AgUy[0] = gUy[2];
        AgUy[1] = Ay[1][0] * gUy[0] + Ay[1][1] * gUy[1] + Ay[1][2] * gUy[2];
        AgUy[2] = Ay[2][0] * gUy[0] + Ay[2][1] * gUy[1] + Ay[2][2] * gUy[2] + Ay[2][3] * gUy[3];
        AgUy[3] = Ay[3][0] * gUy[0] + Ay[3][1] * gUy[1] + Ay[3][2] * gUy[2] + Ay[3][3] * gUy[3];
#pragma unroll
        for (int k = 0; k < 4; ++k) LUh[k] = dUb[k] + AgUx[k] + AgUy[k];
        const double n_gk = sqrt(a0_form_dev(A0, gkx) + a0_form_dev(A0, gky));
        const double n_LUh = sqrt(a0_form_dev(A0, LUh));
        const double n_gU = sqrt(a0_form_dev(A0, gUx) + a0_form_dev(A0, gUy));
        delta = (n_gU >= p.tolerance) ? n_LUh / n_gk : 0.0;
    }
    // SUPG parameter (:246-271)
    double betax = 2.0 * (gUx[0] * Ub[0] + gUx[1] * Ub[1] + gUx[2] * Ub[2] + gUx[3] * Ub[3]);
    double betay = 2.0 * (gUy[0] * Ub[0] + gUy[1] * Ub[1] + gUy[2] * Ub[2] + gUy[3] * Ub[3]);
    const double betaxy = sqrt(betax * betax + betay * betay);
    if (betaxy != 0.0) {
        betax = betax / betaxy;
        betay = betay / betaxy;
    }
    const double h = sqrt(twoArea);
    const double abs_vbeta = fabs(v1 * betax + v2 * betay);
    const double cs = sqrt(gamma * (gamma - 1.0) * (E - 0.5 * (v1 * v1 + v2 * v2)));
    const double CFL = ((cs + abs_vbeta) * delta_t) / h;
    const double psi = (2.0 * alpha * CFL) * (1.0 / (1.0 + 2.0 * alpha * CFL));
    const double tau_d = delta / ((cs + abs_vbeta) * (cs + abs_vbeta));
    const double tau_a = h / (2.0 * (cs + abs_vbeta));
    const double tau_t = (2.0 / (3.0 * (1.0 + 2.0 * alpha * CFL))) * tau_a;
    double tau = tau_t + psi * (tau_a - tau_d);
    if (tau < 0.0) tau = 0.0;
    const double Mg1 = Area * sixth, Mg2 = Area / 12.0;
    const double tau4area = tau / (4 * Area), delta4area = delta / (4.0 * Area);
    const double Kc01 = delta4area * (b[0] * b[1] + c[0] * c[1]);
    const double Kc02 = delta4area * (b[0] * b[2] + c[0] * c[2]);
    const double Kc12 = delta4area * (b[1] * b[2] + c[1] * c[2]);
    // row i of the Jacobians and of their four products, each entry accumulated over k from the k = 0 term;
    // the rows 4a + i share them
    double xi[4], yi[4], Pxx[4], Pxy[4], Pyx[4], Pyy[4], C[3][4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        xi[k] = sel4(i, Ax[0][k], Ax[1][k], Ax[2][k], Ax[3][k]);
        yi[k] = sel4(i, Ay[0][k], Ay[1][k], Ay[2][k], Ay[3][k]);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            Pxx[j] = k == 0 ? xi[0] * Ax[0][j] : Pxx[j] + xi[k] * Ax[k][j];
            Pxy[j] = k == 0 ? xi[0] * Ay[0][j] : Pxy[j] + xi[k] * Ay[k][j];
            Pyx[j] = k == 0 ? yi[0] * Ax[0][j] : Pyx[j] + yi[k] * Ax[k][j];
            Pyy[j] = k == 0 ? yi[0] * Ay[0][j] : Pyy[j] + yi[k] * Ay[k][j];
        }
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int j = 0; j < 4; ++j) C[a][j] = (b[a] * xi[j] + c[a] * yi[j]) * sixth;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const int o1 = a == 0 ? 1 : 0, o2 = a == 2 ? 1 : 2;
        const double Kca1 = a == 2 ? Kc02 : Kc01, Kca2 = a == 0 ? Kc02 : Kc12;   // Kcau(a, o1), Kcau(a, o2)
        double AX[4], AY[4], row[12];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            AX[j] = b[a] * Pxx[j] + c[a] * Pyx[j];
            AY[j] = b[a] * Pxy[j] + c[a] * Pyy[j];
        }
        double MdU = 0, KU = 0;
#pragma unroll
        for (int bb = 0; bb < 3; ++bb) {
            const double Kab = a + bb == 1 ? Kc01 : a + bb == 2 ? Kc02 : Kc12;   // a != bb
            double Ue[4], dUe[4];
            quad_all(U[bb], Ue);
            quad_all(dU[bb], dUe);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool diag = i == j;
                const double Mpg = C[a][j] * tau;
                const double m = diag ? (a == bb ? Mg1 : Mg2) + Mpg : Mpg;
                double k;
                if (a == bb) {
                    const double k1v = tau4area * (b[o1] * AX[j] + c[o1] * AY[j]);
                    const double k2v = tau4area * (b[o2] * AX[j] + c[o2] * AY[j]);
                    k = C[a][j] - (k1v + k2v);
                    k = diag ? k - (Kca1 + Kca2) : k;
                } else {
                    const double kp = tau4area * (b[bb] * AX[j] + c[bb] * AY[j]);
                    k = C[bb][j] + kp;
                    k = diag ? k + Kab : k;
                }
                MdU += m * dUe[j];
                KU += k * Ue[j];
                row[4 * bb + j] = m + alpha * delta_t * k;
            }
        }
        if ((l >> 2) < n) Res[12 * static_cast<size_t>(e) + 4 * a + i] = -MdU - KU;
        // value k of row i of element r at 144 r + 48 a + 12 i + k: turned so that lanes store in order
        double *dst = Ae + 144 * static_cast<size_t>(ew) + 48 * a;
#pragma unroll
        for (int k = 0; k < 12; ++k) turn[l * 13 + k] = row[k];
        wave_lds_fence();
        double w[12];
#pragma unroll
        for (int k = 0; k < 12; ++k) {
            const int q = k * 64 + l, r = q / 12;
            w[k] = turn[r * 13 + (q - 12 * r)];
        }
        wave_lds_fence();   // the next rows reuse the part
#pragma unroll
        for (int k = 0; k < 12; ++k) {
            const int q = k * 64 + l, r = q / 48;
            if (r < n) dst[144 * r + (q - 48 * r)] = w[k];
        }
        __builtin_amdgcn_sched_barrier(0);   // one vertex's rows at a time: their registers are reused
    }
}

}  // namespace fg

using namespace fg;

extern "C" int femgpu_euler_mesh_create(femgpu_ctx *ctx, int nnodes, int nel, int neq, const double *x,
                                        const double *y, const int *type4, const int *invP4, const double *presc4,
                                        const int *ien, const int *lm, const int *scheme, int nnz, femgpu_mesh **out)
{
    return block_mesh_create(ctx, 4, nnodes, nel, neq, x, y, type4, invP4, presc4, ien, lm, scheme, nnz, out);
}

extern "C" int femgpu_assemble_euler(femgpu_mesh *M, const femgpu_euler_problem *pb, const double *d_u,
                                     const double *d_du, double *d_Ae, double *d_R, double *d_AA)
{
    FG_CHECK(M && pb && d_u && d_du && d_R, FEMGPU_ERR_ARG, "femgpu_assemble_euler: bad arguments");
    FG_CHECK(M->ndof == 4, FEMGPU_ERR_STATE, "femgpu_assemble_euler: not an Euler mesh");
    FG_CHECK(!d_AA || M->has_scheme, FEMGPU_ERR_STATE, "femgpu_assemble_euler: mesh created without a CSR slot table");
    femgpu_ctx *ctx = M->ctx;
    double *Ae = d_Ae ? d_Ae : M->ke.p;
    EulerIn in;
    in.x = M->x.p;
    in.y = M->y.p;
    in.presc = M->ubc.p;
    in.u = d_u;
    in.du = d_du;
    in.type = M->type.p;
    in.invP = M->invP.p;
    in.ien = M->ien.p;
    in.neq = M->neq;
    in.pb = *pb;
    if (M->nel > 0) {
        k_elem_euler<<<xcd_grid((M->nel + 63) / 64), 256, 0, ctx->stream>>>(M->nel, in, Ae, M->fe.p);
        FG_HIP(hipGetLastError());
    }
    return launch_block_gathers(M, Ae, d_R, d_AA);
}
