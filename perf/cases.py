"""Performance cases of the library: the work its users have it do, through the public Python layer.

Each case is one pass of a step that the drivers of the four equations repeat: the assembly of a
system on the device, the set-up of its preconditioner, its solve, and the operator products that a
program with its own solver calls. Meshes are triangulations whose interior nodes are moved by the
seed (so geometry, state and right-hand sides change with it while the connectivity, which a
program plans once, stays); unknowns are SYMRCM-ordered for CSR storage, as the drivers order them.

``exact`` computes the same results with numpy and torch alone in 64 bits, from the element
integrals of the discretisations.
"""
import functools
import math

import numpy as np
import torch

from parallel_fem_codes_amd import fem, serving

F64, F32 = torch.float64, torch.float32


def listed():
    return [
        # one multicorrection of the transient transport at the size the library's benchmark quotes:
        # assembly, mixed-precision GMRES(30) with the parallel ILU(0)
        {"name": "transient_mixed_1000x1000", "kind": "transient", "solver": "mixed", "mx": 1000, "my": 1000,
         "cau": False},
        # the same step on a coarse mesh (a first run, a parameter study): launches and host waits
        {"name": "transient_mixed_47x33", "kind": "transient", "solver": "mixed", "mx": 47, "my": 33, "cau": True},
        # the reference's own FP64 pair on a mid-size mesh: exact ILU(0) set-up and pgmres
        {"name": "transient_fp64_300x261", "kind": "transient", "solver": "fp64", "mx": 300, "my": 261, "cau": False},
        # assembly of one fixed-point iteration of the steady transport with CAU shock capture
        {"name": "steady_assembly_640x501", "kind": "steady_assembly", "mx": 640, "my": 501, "cau": True},
        # assembly of one Picard iteration of the steady Navier-Stokes equations into CSR
        {"name": "ns_assembly_256x256", "kind": "ns_assembly", "mx": 256, "my": 256, "Re": 1000.0, "force": False},
        # ILU(0) set-up of a Picard system (rows of up to 21 entries) and its first application
        {"name": "ns_ilu_setup_80x80", "kind": "ns_ilu", "mx": 80, "my": 80, "Re": 400.0},
        # set-up of one multicorrection of the Euler equations with element-by-element storage:
        # element matrices, operator, nodal blocks, preconditioned residual, first product
        {"name": "euler_setup_400x200", "kind": "euler_setup", "mx": 400, "my": 200, "dimensionless": 0},
        # a whole pseudo-time step of the Euler driver, mixed precision
        {"name": "euler_step_200x100", "kind": "euler_step", "mx": 200, "my": 100, "orth": "CGS"},
        # the operator products on their own, as a program with its own Krylov loop calls them
        {"name": "csrmv_f64_1236x811", "kind": "csrmv", "mx": 1236, "my": 811, "ndof": 1, "dtype": "f64"},
        {"name": "ebemv3_f64_511x640", "kind": "ebemv", "mx": 511, "my": 640, "ndof": 1, "dtype": "f64"},
        {"name": "ebemv12_f32_800x400", "kind": "ebemv", "mx": 800, "my": 400, "ndof": 4, "dtype": "f32"},
        # a batch of small steady systems on unstructured meshes, as the request loop packs them
        {"name": "batched_steady_24", "kind": "batched", "systems": 24, "nmin": 300, "nmax": 3000},
    ]


def _size(rng, lo, hi):
    """Mesh cells per direction: log-uniform, with an aspect ratio of up to 2."""
    a = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    r = math.exp(rng.uniform(-math.log(2.0), math.log(2.0)))
    return max(4, int(a * math.sqrt(r))), max(4, int(a / math.sqrt(r)))


def draw(rng):
    kind = rng.choice(["transient", "transient", "steady_assembly", "ns_assembly", "ns_ilu", "euler_setup", "euler_step",
                       "csrmv", "ebemv", "batched"])
    c = {"kind": kind}
    if kind == "transient":
        c["solver"] = rng.choice(["mixed", "mixed", "fp64"])
        c["mx"], c["my"] = _size(rng, 24, 700 if c["solver"] == "mixed" else 300)
        c["cau"] = rng.random() < 0.5
    elif kind == "steady_assembly":
        c["mx"], c["my"] = _size(rng, 24, 640)
        c["cau"] = rng.random() < 0.7
    elif kind == "ns_assembly":
        c["mx"], c["my"] = _size(rng, 16, 256)
        c["Re"], c["force"] = float(rng.choice([100, 400, 1000, 5000])), rng.random() < 0.5
    elif kind == "ns_ilu":
        c["mx"], c["my"] = _size(rng, 16, 90)
        c["Re"] = float(rng.choice([100, 400, 1000]))
    elif kind == "euler_setup":
        c["mx"], c["my"] = _size(rng, 16, 280)
        c["dimensionless"] = rng.choice([0, 1])
    elif kind == "euler_step":
        c["mx"], c["my"] = _size(rng, 16, 140)
        c["orth"] = rng.choice(["CGS", "MGS"])
    elif kind == "csrmv":
        c["mx"], c["my"] = _size(rng, 24, 1000)
        c["ndof"], c["dtype"] = 1, rng.choice(["f64", "f32"])
        if rng.random() < 0.4:
            c["ndof"] = 3
            c["mx"], c["my"] = _size(rng, 16, 200)
    elif kind == "ebemv":
        c["ndof"], c["dtype"] = rng.choice([1, 3, 4]), rng.choice(["f64", "f32"])
        c["mx"], c["my"] = _size(rng, 24, {1: 900, 3: 350, 4: 400}[c["ndof"]])
    else:
        c["systems"], c["nmin"], c["nmax"] = rng.randint(4, 32), rng.randint(150, 400), rng.randint(1000, 3000)
    return c


# ------------------------------------------------------------------------------ meshes and numbering

BOX = {1: (0.0, 0.0, 1.0, 1.0), 3: (0.0, 0.0, 1.0, 1.0), 4: (0.0, 0.0, 2.0, 1.0)}


@functools.lru_cache(maxsize=6)
def _structure(mx, my, ndof, csr):
    """Connectivity, marks and numbering of an mx x my mesh (host arrays, the same for every seed):
    what a program plans once. ndof 1: transport, 3: cavity, 4: oblique shock."""
    x, y, ien = fem.structured_mesh(mx, my, box=BOX[ndof])
    if ndof == 1:
        t = fem.boundary_types(x, y)
    else:
        t = fem.structured_marks({3: "CAVITY", 4: "OBLIQUO"}[ndof], x, y)[2]
        if ndof == 3 and (t.reshape(-1, 3)[:, 2] != 0).all():   # no node at the centre: pin the first pressure
            t = t.copy()
            t[2] = 0
    inv, neq = fem.number_unknowns(t, ndof)
    lm = fem.Fill_LM(ien, t, inv, neq, ndof)
    S = {"x": x, "y": y, "ien": ien, "type": t, "inv": inv, "neq": neq, "lm": lm}
    if csr:
        c = fem.csr_Initialization(lm, 3 * ndof, neq, "SYMRCM", permute_lm=True, type_=t, invP_id=inv)
        S.update(inv=c.invP_id, lm=c.lm, IA=c.IA, JA=c.JA, scheme=c.scheme, nnz=c.nnz)
    return S


def _moved(S, mx, my, ndof, seed):
    """The nodes, interior ones moved by up to a fifth of a cell."""
    rng = np.random.default_rng([seed, 1])
    x0, y0, x1, y1 = BOX[ndof]
    x, y = S["x"], S["y"]
    inner = (x > x0 + 1e-12) & (x < x1 - 1e-12) & (y > y0 + 1e-12) & (y < y1 - 1e-12)
    dx = rng.uniform(-0.2, 0.2, len(x)) * (x1 - x0) / mx
    dy = rng.uniform(-0.2, 0.2, len(x)) * (y1 - y0) / my
    return np.where(inner, x + dx, x), np.where(inner, y + dy, y)


def _smooth(x, y, rng, modes=6):
    """A smooth random field of the nodes."""
    f = np.zeros(len(x))
    for _ in range(modes):
        kx, ky, ph = rng.uniform(-12, 12), rng.uniform(-12, 12), rng.uniform(0, 2 * np.pi)
        f += rng.normal() * np.sin(kx * x + ky * y + ph)
    return f / modes


def _at_unknowns(S, nodal, ndof):
    """A dof field (nnodes*ndof) at the unknowns, in the solve numbering."""
    u = np.zeros(S["neq"])
    m = S["type"] != 0
    u[S["inv"][m]] = nodal[m]
    return u


def _dev(a, dtype=F64):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dtype)


# ------------------------------------------------------------------------------ inputs

TT = {"k": 1e-4, "alpha": 0.5}   # the rotating-field workload


def _transport_inputs(case, seed):
    S = _structure(case["mx"], case["my"], 1, True)
    rng = np.random.default_rng([seed, 2])
    x, y = _moved(S, case["mx"], case["my"], 1, seed)
    ubc = np.where((np.abs(x) <= 1e-15) & (y > 0.25) & (y < 0.5), 1.0, 0.0)
    cx, cy, sg = rng.uniform(0.25, 0.75), rng.uniform(0.25, 0.75), rng.uniform(0.05, 0.15)
    pulse = np.exp(-((x - cx) ** 2 + (y - cy) ** 2) / (2 * sg ** 2)) + 0.05 * _smooth(x, y, rng)
    u, du = _at_unknowns(S, pulse, 1), _at_unknowns(S, 0.1 * _smooth(x, y, rng), 1)
    return S, x, y, ubc, u, du, 1.0 / max(case["mx"], case["my"])


def _ns_inputs(case, seed):
    S = _structure(case["mx"], case["my"], 3, True)
    rng = np.random.default_rng([seed, 3])
    x, y = _moved(S, case["mx"], case["my"], 3, seed)
    presc = np.zeros((len(x), 3))
    presc[np.abs(y - 1.0) <= 1e-15, 0] = 1.0
    state = np.stack([y * y + 0.1 * _smooth(x, y, rng), 0.2 * _smooth(x, y, rng), 0.1 * _smooth(x, y, rng)], 1)
    u = _at_unknowns(S, state.ravel(), 3)
    f = [_smooth(x, y, rng) for _ in range(2)] if case.get("force") else None
    return S, x, y, presc.ravel(), u, f


def _euler_inputs(case, seed):
    S = _structure(case["mx"], case["my"], 4, False)
    rng = np.random.default_rng([seed, 4])
    x, y = _moved(S, case["mx"], case["my"], 4, seed)
    free = np.array(fem.OBLIQUO_STATE)
    presc = np.tile(free, (len(x), 1))
    presc[(np.abs(y) <= 1e-15) & (np.abs(x) > 0), 2] = 0.0
    state = np.tile(free, (len(x), 1))
    state *= 1.0 + 0.05 * np.stack([_smooth(x, y, rng) for _ in range(4)], 1)
    u = _at_unknowns(S, state.ravel(), 4)
    du = _at_unknowns(S, (0.02 * np.stack([_smooth(x, y, rng) for _ in range(4)], 1)).ravel(), 4)
    h = math.sqrt(2.0 / (case["mx"] * case["my"]))
    rho, m1, m2, rE = free
    v = math.hypot(m1, m2) / rho
    c = math.sqrt(0.56 * (rE / rho - 0.5 * v * v))
    pb = {"gamma": 1.4, "Mach": v / c, "alpha": 0.5, "dt": 5.0 * h / (c + v), "tolerance": 1e-8,
          "dimensionless": int(case.get("dimensionless", 0)), "shock": 1}
    return S, x, y, presc.ravel(), u, du, pb


def _ebe_values(case, seed, nel):
    """Element matrices with a mass part and a part of any sign, on the GPU."""
    s = 3 * case["ndof"]
    g = torch.Generator(device="cuda").manual_seed(seed * 7 + 5)
    A = torch.randn(nel, s, s, dtype=F64, device="cuda", generator=g).mul_(0.05)
    mass = torch.kron(torch.eye(3, dtype=F64) + 1.0, torch.eye(case["ndof"], dtype=F64)).cuda() / 12.0
    return A.add_(mass)


@functools.lru_cache(maxsize=4)
def _requests(systems, nmin, nmax, seed):
    """Steady systems on Delaunay meshes of the unit square, of nmin to nmax points (spaced evenly over
    the logarithm): per request its CSR structure and data."""
    rng = np.random.default_rng([seed, 7])
    sizes = np.exp(np.linspace(math.log(nmin), math.log(nmax), systems)).astype(int)
    out = []
    for npts in rng.permutation(sizes):
        x, y, typ, ubc, ien = serving.square_mesh(int(npts), rng)
        k, th = math.exp(rng.uniform(math.log(1e-4), math.log(1e-2))), rng.uniform(0.0, 2 * math.pi)
        inv, neq = fem.number_unknowns(typ)
        lm = fem.Fill_LM(ien, typ, inv, neq)
        c = fem.csr_Initialization(lm, 3, neq, "SYMRCM", type_=typ, invP_id=inv)
        S = {"ien": ien, "type": typ, "inv": c.invP_id, "neq": neq, "scheme": c.scheme, "nnz": c.nnz, "IA": c.IA,
             "JA": c.JA}
        Ke, Fe = _transport_elements(S, x, y, ubc, np.zeros(neq), None, k, False, 0.0, 0.0, (math.cos(th), 0.0, 0.0),
                                     (math.sin(th), 0.0, 0.0))
        out.append((S, _csr_sum(S, Ke), _row_sum(S, Fe, 1)[:neq]))
    return out


# ------------------------------------------------------------------------------ prepare and run

def prepare(case, seed):
    kind = case["kind"]
    dev = fem.Device(0)
    st = {"case": case, "dev": dev}
    if kind in ("transient", "steady_assembly"):
        S, x, y, ubc, u, du, dt = _transport_inputs(case, seed)
        st["M"] = fem.Mesh(dev, x, y, S["type"], S["inv"], ubc, S["ien"], S["neq"], lm=S["lm"], scheme=S["scheme"],
                           nnz=S["nnz"])
        st["pb"] = fem.make_problem(k=TT["k"], f0=0.0 if kind == "transient" else 1.0, shock=1 if case["cau"] else 0)
        st["u"], st["du"], st["dt"] = _dev(u), _dev(du), dt
        if kind == "transient":
            st["A"] = fem.CsrMatrix(dev, S["IA"], S["JA"])
            st["R"] = torch.zeros(S["neq"] + 1, dtype=F64, device="cuda")
            st["X"] = torch.zeros(S["neq"], dtype=F64, device="cuda")
            st["B"] = torch.zeros_like(st["X"])
        else:
            st["F"] = torch.zeros(S["neq"], dtype=F64, device="cuda")
            st["AA"] = torch.zeros(S["nnz"] + 1, dtype=F64, device="cuda")
    elif kind == "ns_assembly":
        S, x, y, presc, u, f = _ns_inputs(case, seed)
        st["M"] = fem.NsMesh(dev, x, y, S["type"], S["inv"], presc, S["ien"], S["lm"], S["neq"], scheme=S["scheme"],
                             nnz=S["nnz"])
        st["u"] = _dev(u)
        st["f"] = [_dev(v) for v in f] if f else [None, None]
        st["F"] = torch.zeros(S["neq"] + 1, dtype=F64, device="cuda")
        st["AA"] = torch.zeros(S["nnz"] + 1, dtype=F64, device="cuda")
    elif kind == "ns_ilu":
        S, x, y, presc, u, f = _ns_inputs(case, seed)
        Ke, Fe = _ns_elements(S, x, y, presc, u, f, case["Re"])
        st["A"] = fem.CsrMatrix(dev, S["IA"], S["JA"])
        st["AA"], st["F0"] = _dev(_csr_sum(S, Ke)), _dev(_row_sum(S, Fe, 3)[:S["neq"]])
        st["F"] = torch.zeros_like(st["F0"])
    elif kind in ("euler_setup", "euler_step"):
        S, x, y, presc, u, du, pb = _euler_inputs(case, seed)
        st["M"] = fem.EulerMesh(dev, x, y, S["type"], S["inv"], presc, S["ien"], S["lm"], S["neq"])
        st["E"] = fem.EbeMatrix(dev, S["lm"], 12, S["neq"])
        st["D"] = fem.BlockDiag(dev, len(x), S["ien"], 4, S["type"], S["inv"], S["neq"])
        st["pb"] = fem.make_euler_problem(**pb)
        st["u0"], st["du0"] = _dev(u), _dev(du)
        st["u"], st["du"] = _dev(u), _dev(du)
        st["R"] = torch.zeros(S["neq"] + 1, dtype=F64, device="cuda")
        st["Z"], st["Q"] = torch.zeros(S["neq"], dtype=F64, device="cuda"), torch.zeros(S["neq"], dtype=F64, device="cuda")
        if kind == "euler_setup":
            st["Ae"] = torch.zeros(len(S["ien"]) // 3, 12, 12, dtype=F64, device="cuda")
        st["opts"] = fem.driver_opts("mixed", kmax=50, lmax=400, tol=1e-8, nonlinear_tol=1e-30, nonlinear_maxiter=2,
                                     stop_by_norm=False, inner_kmax=50, inner_tol=1e-4,
                                     orthogonalization=case.get("orth", "MGS"))
    elif kind == "csrmv":
        S = _structure(case["mx"], case["my"], case["ndof"], True)
        rng = np.random.default_rng([seed, 5])
        dt = F64 if case["dtype"] == "f64" else F32
        st["A"] = fem.CsrMatrix(dev, S["IA"], S["JA"])
        st["A"].set_values(_dev(rng.standard_normal(S["nnz"])))
        st["P"] = _dev(rng.standard_normal(S["neq"]), dt)
        st["Q"] = torch.zeros_like(st["P"])
    elif kind == "ebemv":
        S = _structure(case["mx"], case["my"], case["ndof"], False)
        dt = F64 if case["dtype"] == "f64" else F32
        st["E"] = fem.EbeMatrix(dev, S["lm"], 3 * case["ndof"], S["neq"])
        st["E"].set_values(_ebe_values(case, seed, len(S["ien"]) // 3))
        st["P"] = _dev(np.random.default_rng([seed, 6]).standard_normal(S["neq"]), dt)
        st["Q"] = torch.zeros_like(st["P"])
        torch.cuda.synchronize()
    else:
        reqs = _requests(case["systems"], case["nmin"], case["nmax"], seed)
        IA, JA, st["off"], _ = fem.concat_csr([(S["IA"], S["JA"]) for S, _, _ in reqs])
        st["A"] = fem.CsrMatrix(dev, IA, JA)
        st["A"].set_values(np.concatenate([a for _, a, _ in reqs]))
        st["F"] = _dev(np.concatenate([f for _, _, f in reqs]))
        st["X"] = torch.zeros_like(st["F"])
    return st


def run(st):
    kind = st["case"]["kind"]
    if kind == "transient":
        A, n = st["A"], st["X"].numel()
        st["M"].Build_M_K_R_SUPG(st["pb"], TT["alpha"], st["dt"], st["u"], st["du"], st["R"], AA_ptr=A.values_ptr())
        A.values_changed()
        if st["case"]["solver"] == "mixed":
            fem.gmres_mixed(st["dev"], A, st["R"][:n], st["X"], tol=1e-8, inner_kmax=30, inner_tol=1e-4, sweep_mode=2,
                            factor_sweeps=1)
            return {"R": st["R"], "X": st["X"]}
        st["B"].copy_(st["R"][:n])
        A.ILUp_precond_setup(st["B"])
        fem.pgmres(st["dev"], A, st["B"], st["X"], 30, 1000, 1e-8, precond=A)
        return {"R": st["R"], "B": st["B"], "X": st["X"]}
    if kind == "steady_assembly":
        st["M"].Build_K_F_SUPG(st["pb"], st["u"], st["F"], AA_ptr=st["AA"].data_ptr())
        return {"F": st["F"], "AA": st["AA"]}
    if kind == "ns_assembly":
        st["M"].Build_K_F_SUPG_PSPG(st["case"]["Re"], st["u"], st["F"], *st["f"], AA_ptr=st["AA"].data_ptr())
        return {"F": st["F"], "AA": st["AA"]}
    if kind == "ns_ilu":
        st["A"].set_values(st["AA"])
        st["F"].copy_(st["F0"])
        st["A"].ILUp_precond_setup(st["F"])
        return {"F": st["F"]}
    if kind == "euler_setup":
        n = st["Z"].numel()
        st["M"].Build_M_K_F_SUPG(st["pb"], st["u0"], st["du0"], st["R"], Ae=st["Ae"])
        st["E"].set_values(st["Ae"])
        st["D"].setup(st["Ae"])
        st["D"].apply(st["R"][:n], st["Z"])
        st["E"].ebemv(st["Z"], st["Q"])
        return {"Ae": st["Ae"], "R": st["R"], "Z": st["Z"], "Q": st["Q"]}
    if kind == "euler_step":
        st["u"].copy_(st["u0"])
        st["du"].copy_(st["du0"])
        fem.Predictor_Old_step_Euler(st["M"], st["E"], st["D"], st["pb"], st["u"], st["du"], st["opts"])
        return {"u": st["u"], "a": st["du"]}
    if kind == "csrmv":
        st["A"].csrmv(st["P"], st["Q"])
        return st["Q"]
    if kind == "ebemv":
        st["E"].ebemv(st["P"], st["Q"])
        return st["Q"]
    fem.gmres_mixed_batched(st["dev"], st["A"], st["off"], st["F"], st["X"], tol=1e-8, sweep_mode=2, factor_sweeps=2,
                            orthogonalization="CGS")
    return st["X"]


# ------------------------------------------------------------------------------ work and tolerances

def work(case):
    """Inputs read once and results written once; operations of the products and element integrals.
    The solves add one product with the assembled operator, which any solver needs."""
    kind = case["kind"]
    if kind == "batched":
        n = case["systems"] * (case["nmax"] - case["nmin"]) / math.log(case["nmax"] / case["nmin"])
        return {"bytes": 7 * n * 12 + 16 * n, "flops": 14 * n}
    mx, my = case["mx"], case["my"]
    nn, nel = (mx + 1) * (my + 1), 2 * mx * my
    ndof = {"ns_assembly": 3, "ns_ilu": 3, "euler_setup": 4, "euler_step": 4}.get(kind, case.get("ndof", 1))
    n = ndof * nn
    nnz = 7 * ndof * n
    mesh = 16 * nn + 12 * nel
    if kind == "transient":
        return {"bytes": mesh + 8 * nn + 16 * n + 16 * n, "flops": 350 * nel + 2 * nnz}
    if kind == "steady_assembly":
        return {"bytes": mesh + 8 * nn + 8 * n + 8 * n + 8 * nnz, "flops": 300 * nel}
    if kind == "ns_assembly":
        return {"bytes": mesh + 24 * nn + 8 * n + 8 * n + 8 * nnz, "flops": 600 * nel}
    if kind == "ns_ilu":
        return {"bytes": 12 * nnz + 16 * n, "flops": 2 * nnz * 10 + 2 * nnz}
    if kind == "euler_setup":
        return {"bytes": mesh + 32 * nn + 16 * n + 8 * 144 * nel + 24 * n, "flops": 3000 * nel + 2 * 144 * nel}
    if kind == "euler_step":
        return {"bytes": mesh + 32 * nn + 32 * n, "flops": 2 * (3000 * nel + 2 * 144 * nel)}
    w = 8 if case["dtype"] == "f64" else 4
    if kind == "csrmv":
        return {"bytes": nnz * (w + 4) + 4 * n + 2 * w * n, "flops": 2 * nnz}
    s = 3 * ndof
    return {"bytes": nel * (w * s * s + 4 * s) + 2 * w * n, "flops": 2 * nel * s * s}


def tolerance(case):
    """About four times the largest distance from exact() seen over the ranges. Products: rounding of
    the data type over a row. Assemblies and factors: the same, with the cancellations of the
    shock-capture terms. Solves stop at a relative residual of 1e-8, and a correct solver may stop just
    below it (measured 1e-9 to 3e-9 in the transient solution; in the steady systems the condition
    number comes on top; the Euler step's second multicorrection reduces the first one's error)."""
    kind = case["kind"]
    if kind == "transient":
        return {"rel": 3e-8}
    if kind == "batched":
        return {"rel": 5e-8}
    if kind == "euler_step":
        return {"rel": 1e-10}
    if kind in ("csrmv", "ebemv"):
        return {"rel": 1e-15 if case["dtype"] == "f64" else 3e-7}
    return {"rel": 1e-12}


# ------------------------------------------------------------------------------ results in 64 bits

def _csr_sum(S, Ke):
    """CSR values: element entries summed into their slots (the dummy slot, last, dropped)."""
    return np.bincount(S["scheme"], weights=Ke.reshape(-1), minlength=S["nnz"] + 1)[:S["nnz"]]


def _row_sum(S, Fe, ndof):
    """Element loads summed into the unknowns; one entry more, 0, for prescribed dofs."""
    ien = S["ien"].reshape(-1, 3)
    dofs = (ndof * ien[:, :, None] + np.arange(ndof)).reshape(len(ien), -1)
    rows = np.where(S["type"][dofs] != 0, S["inv"][dofs], S["neq"])
    F = np.bincount(rows.reshape(-1), weights=Fe.reshape(-1), minlength=S["neq"] + 1)
    F[S["neq"]] = 0.0
    return F


def _dof_values(S, u, presc, ndof):
    """Per element and vertex the ndof values: the state at unknowns, prescribed values elsewhere."""
    full = np.array(presc, dtype=np.float64)
    m = S["type"] != 0
    full[m] = u[S["inv"][m]]
    return full.reshape(-1, ndof)[S["ien"].reshape(-1, 3)]


def _edges(S, x, y):
    v = S["ien"].reshape(-1, 3)
    X, Y = x[v], y[v]
    b = np.roll(Y, -1, 1) - np.roll(Y, -2, 1)   # y2 - y3, y3 - y1, y1 - y2
    c = np.roll(X, -2, 1) - np.roll(X, -1, 1)   # x3 - x2, x1 - x3, x2 - x1
    return X, Y, b, c, c[:, 2] * b[:, 1] - c[:, 1] * b[:, 2]


def _transport_elements(S, x, y, ubc, u, du, k, cau, f0, alpha_dt, bx=(0.5, 0.0, -1.0), by=(-0.5, 1.0, 0.0)):
    """SUPG element matrices and loads of the transport problem: steady (du None; K and F minus the
    lifted Dirichlet values) or transient (M + alpha dt K and f - M du - K u)."""
    X, Y, b, c, twoA = _edges(S, x, y)
    A = 0.5 * twoA
    ue = _dof_values(S, u, ubc, 1)[:, :, 0]
    XB, YB = X.mean(1), Y.mean(1)
    wx, wy = bx[0] + bx[1] * XB + bx[2] * YB, by[0] + by[1] * XB + by[2] * YB
    nw = np.hypot(wx, wy)
    h = np.sqrt(np.abs(twoA))
    tau = np.where(nw > 0, 0.5 * h / np.where(nw > 0, nw, 1.0), 0.0)
    g = (wx[:, None] * b + wy[:, None] * c)            # 2A w . grad N
    E = lambda v: v[:, None, None]
    bb, cc = b[:, :, None] * b[:, None, :], c[:, :, None] * c[:, None, :]
    K = E(0.25 * k / A) * (bb + cc) + g[:, None, :] / 6.0 + E(0.25 * tau / A) * g[:, :, None] * g[:, None, :]
    due = np.zeros_like(ue) if du is None else _dof_values(S, du, np.zeros(len(x)), 1)[:, :, 0]
    if cau:
        adv = (g * ue).sum(1) / twoA
        g0, g1 = (b * ue).sum(1) / twoA, (c * ue).sum(1) / twoA
        ng = np.hypot(g0, g1)
        ok = ng > 0
        ngs = np.where(ok, ng, 1.0)
        Ru = due.mean(1) + adv - f0
        px, py = adv * g0 / ngs ** 2, adv * g1 / ngs ** 2
        kp = px * px * k + py * py * k
        with np.errstate(divide="ignore", invalid="ignore"):
            Pe = 0.5 * h * np.hypot(px, py) ** 3 / kp
        fac = np.where(Pe / 3.0 < 0.7, Pe / 3.0, 0.7)
        Eu = np.where(ok, 0.5 * h * fac * np.abs(Ru) / ngs, 0.0)
        K = K + E(0.25 * Eu / A) * (bb + cc)
    Fe = (A / 3.0 * f0)[:, None] + (tau * f0 / 2.0)[:, None] * g
    if du is None:
        dirichlet = (S["type"][S["ien"].reshape(-1, 3)] == 0)
        ub = np.where(dirichlet, ubc[S["ien"].reshape(-1, 3)], 0.0)
        return K, Fe - np.einsum("eab,eb->ea", K, ub)
    M = E(A / 12.0) * (np.eye(3) + 1.0) + E(tau) * g[:, :, None] / 6.0
    return M + alpha_dt * K, Fe - np.einsum("eab,eb->ea", M, due) - np.einsum("eab,eb->ea", K, ue)


def _ns_elements(S, x, y, presc, u, f, Re):
    """SUPG/PSPG/LSIC element matrices (Picard tangent) and residuals of the steady Navier-Stokes
    equations, unit density, viscosity 1/Re."""
    X, Y, b, c, twoA = _edges(S, x, y)
    twoA = np.abs(twoA)
    A, nu = 0.5 * twoA, 1.0 / Re
    W = _dof_values(S, u, presc, 3)
    U, V, Pn = W[:, :, 0], W[:, :, 1], W[:, :, 2]
    ux, uy, p = U.mean(1), V.mean(1), Pn.mean(1)
    gr = lambda q: ((q * b).sum(1) / twoA, (q * c).sum(1) / twoA)
    (uxx, uxy), (uyx, uyy), (px, py) = gr(U), gr(V), gr(Pn)
    div2A = (U * b).sum(1) + (V * c).sum(1)
    C = (ux[:, None] * b + uy[:, None] * c) / twoA[:, None]
    h, un = np.sqrt(twoA), np.hypot(ux, uy)
    tau = 1.0 / np.sqrt((2 * un / h) ** 2 + 9.0 * (4 * nu / (h * h)) ** 2)
    tl = np.sqrt(nu * nu + (0.5 * h * un) ** 2)
    E = lambda v: v[:, None, None]
    r, q = (lambda v: v[:, :, None]), (lambda v: v[:, None, :])   # row vertex, column vertex
    K = np.zeros((len(A), 3, 3, 3, 3))   # element, row vertex, row dof, column vertex, column dof
    conv = E(A / 3) * q(C) + E(tau * A) * r(C) * q(C)
    kv, ks = E(0.25 * nu / A), E(0.25 * tl / A)
    K[:, :, 0, :, 0] = conv + kv * (2 * r(b) * q(b) + r(c) * q(c)) + ks * r(b) * q(b)
    K[:, :, 0, :, 1] = kv * r(c) * q(b) + ks * r(b) * q(c)
    K[:, :, 1, :, 0] = kv * r(b) * q(c) + ks * r(c) * q(b)
    K[:, :, 1, :, 1] = conv + kv * (r(b) * q(b) + 2 * r(c) * q(c)) + ks * r(c) * q(c)
    K[:, :, 0, :, 2] = -(r(b) / 6 + E(0.5 * tau) * r(C) * q(b))
    K[:, :, 1, :, 2] = -(r(c) / 6 + E(0.5 * tau) * r(C) * q(c))
    K[:, :, 2, :, 0] = q(b) / 6 + E(0.5 * tau) * q(C) * r(b)
    K[:, :, 2, :, 1] = q(c) / 6 + E(0.5 * tau) * q(C) * r(c)
    K[:, :, 2, :, 2] = E(0.25 * tau / A) * (r(b) * q(b) + r(c) * q(c))
    fx, fy = (w[S["ien"].reshape(-1, 3)].mean(1) if f else np.zeros(len(A)) for w in (f or [None, None]))
    cx, cy = uxx * ux + uxy * uy, uyx * ux + uyy * uy
    R = np.zeros((len(A), 3, 3))
    e = lambda v: v[:, None]
    test = e(A / 3) + e(tau * A) * C
    R[:, :, 0] = test * e(fx - cx) - 0.5 * nu * (2 * b * e(uxx) + c * e(uxy + uyx)) - e(0.25 * tl / A * div2A) * b + \
        0.5 * e(p) * b + e(tau * A * px) * C
    R[:, :, 1] = test * e(fy - cy) - 0.5 * nu * (2 * c * e(uyy) + b * e(uxy + uyx)) - e(0.25 * tl / A * div2A) * c + \
        0.5 * e(p) * c + e(tau * A * py) * C
    R[:, :, 2] = e(tau * A) * (b * e(fx) + c * e(fy)) - e(A / 3 * (uxx + uyy)) - e(0.5 * tau) * (b * e(cx) + c * e(cy)) - \
        e(0.5 * tau) * (b * e(px) + c * e(py))
    return K, R


def _euler_elements(S, x, y, presc, u, du, pb):
    """SUPG element matrices M + alpha dt K with CAU shock capture and residuals -(M dU + K U) of the
    2D Euler equations in conservative variables."""
    X, Y, b, c, twoA = _edges(S, x, y)
    twoA = np.abs(twoA)
    A = 0.5 * twoA
    Ue = _dof_values(S, u, presc, 4)
    dUe = _dof_values(S, du, np.zeros(4 * len(x)), 4)
    Ub, dUb = Ue.mean(1), dUe.mean(1)
    gx = np.einsum("eav,ea->ev", Ue, b) / twoA[:, None]
    gy = np.einsum("eav,ea->ev", Ue, c) / twoA[:, None]
    g = pb["gamma"]
    v1, v2, En = Ub[:, 1] / Ub[:, 0], Ub[:, 2] / Ub[:, 0], Ub[:, 3] / Ub[:, 0]
    q2 = v1 * v1 + v2 * v2
    eps2 = pb["Mach"] ** 2 if pb["dimensionless"] else 1.0
    z, one = np.zeros_like(v1), np.ones_like(v1)
    st = lambda rows: np.stack([np.stack(r, -1) for r in rows], -2)
    Ax = st([[z, one, z, z],
             [(g - 1) * q2 / 2 - v1 * v1, (3 - g) * v1, -(g - 1) * v2, (g - 1) / eps2 * one],
             [-v1 * v2, v2, v1, z],
             [-v1 * (g * En - (g - 1) * eps2 * q2), g * En - (g - 1) * eps2 * (q2 / 2 + v1 * v1),
              -(g - 1) * eps2 * v1 * v2, g * v1]])
    Ay = st([[z, z, one, z],
             [-v1 * v2, v2, v1, z],
             [(g - 1) * q2 / 2 - v2 * v2, -(g - 1) * v1, (3 - g) * v2, (g - 1) / eps2 * one],
             [-v2 * (g * En - (g - 1) * eps2 * q2), -(g - 1) * eps2 * v1 * v2,
              g * En - (g - 1) * eps2 * (q2 / 2 + v2 * v2), g * v2]])
    # entropy-variable metric
    ri = Ub[:, 3] - (Ub[:, 1] ** 2 + Ub[:, 2] ** 2) / (2 * Ub[:, 0])
    V2, V3, V4 = Ub[:, 1] / ri, Ub[:, 2] / ri, -Ub[:, 0] / ri
    k1 = (V2 ** 2 + V3 ** 2) / (2 * V4)
    A0 = st([[k1 * k1 + g, k1 * V2, k1 * V3, (k1 + 1) * V4], [k1 * V2, V2 * V2 - V4, V2 * V3, V2 * V4],
             [k1 * V3, V2 * V3, V3 * V3 - V4, V3 * V4], [(k1 + 1) * V4, V2 * V4, V3 * V4, V4 * V4]])
    A0 *= (-1.0 / (ri * V4))[:, None, None]
    form = lambda w: np.einsum("ei,eij,ej->e", w, A0, w)
    kx = (b[:, :1] * gx + c[:, :1] * gy) / twoA[:, None]
    ky = (b[:, 1:2] * gx + c[:, 1:2] * gy) / twoA[:, None]
    res = dUb + np.einsum("eij,ej->ei", Ax, gx) + np.einsum("eij,ej->ei", Ay, gy)
    delta = np.zeros_like(A)
    if pb["shock"]:
        act = np.sqrt(form(gx) + form(gy)) >= pb["tolerance"]
        delta[act] = np.sqrt(form(res)[act]) / np.sqrt((form(kx) + form(ky))[act])
    be, ce = 2 * (gx * Ub).sum(1), 2 * (gy * Ub).sum(1)
    nb = np.hypot(be, ce)
    nb = np.where(nb != 0, nb, 1.0)
    h = np.sqrt(twoA)
    s = np.sqrt(g * (g - 1) * (En - q2 / 2)) + np.abs(v1 * be / nb + v2 * ce / nb)
    al, dt = pb["alpha"], pb["dt"]
    cfl = 2 * al * s * dt / h
    ta = h / (2 * s)
    tau = 2.0 / (3.0 * (1 + cfl)) * ta + cfl / (1 + cfl) * (ta - delta / s ** 2)
    tau = np.maximum(tau, 0.0)
    G = b[:, :, None, None] * Ax[:, None] + c[:, :, None, None] * Ay[:, None]   # 2A A . grad N_a
    I4 = np.eye(4)
    E = lambda v: v[:, None, None, None, None]
    M = np.einsum("e,ab,ij->eaibj", A / 12, np.eye(3) + 1.0, I4) + E(tau / 6) * G[:, :, :, None, :]
    K = np.repeat(G.transpose(0, 2, 1, 3)[:, None] / 6, 3, axis=1)
    K = K + E(tau / (4 * A)) * np.einsum("eaik,ebkj->eaibj", G, G, optimize=True)
    K += np.einsum("eab,ij->eaibj", (delta / (4 * A))[:, None, None] * (b[:, :, None] * b[:, None] + c[:, :, None] * c[:, None]),
                   I4)
    R = -np.einsum("eaibj,ebj->eai", M, dUe, optimize=True) - np.einsum("eaibj,ebj->eai", K, Ue, optimize=True)
    return M + al * dt * K, R


def _block_inverses(S, Ae, nn):
    """Nodal 4x4 blocks summed over the elements and inverted as the reference inverts them: the
    adjugate with one cofactor (row 4, column 3) taken with the entry of row 3, column 2 of the block
    in place of that of row 2, column 2."""
    ien = S["ien"].reshape(-1, 3)
    D = np.zeros((nn, 16))
    for a in range(3):
        blk = Ae.reshape(-1, 3, 4, 3, 4)[:, a, :, a, :].reshape(-1, 16)
        for q in range(16):
            D[:, q] += np.bincount(ien[:, a], weights=blk[:, q], minlength=nn)
    D = D.reshape(nn, 4, 4)
    inv = np.linalg.inv(D)
    inv[:, 3, 2] += D[:, 0, 2] * D[:, 3, 0] * (D[:, 2, 1] - D[:, 1, 1]) / np.linalg.det(D)
    return inv


def _apply_blocks(S, inv, r):
    full = np.zeros(len(S["type"]))
    m = S["type"] != 0
    full[m] = r[S["inv"][m]]
    zf = np.einsum("nij,nj->ni", inv, full.reshape(-1, 4)).reshape(-1)
    out = np.zeros(S["neq"])
    out[S["inv"][m]] = zf[m]
    return out


def _ebe_product(lm, Ae, p, neq):
    """Sum over the elements of A_e p_e, on the device of Ae."""
    pe = torch.cat([p, p.new_zeros(1)])[lm]
    q = torch.zeros(neq + 1, dtype=F64, device=Ae.device)
    q.index_add_(0, lm.reshape(-1), torch.bmm(Ae, pe.unsqueeze(2)).reshape(-1))
    return q[:neq]


def _ell(IA, JA, AA, dev):
    """Rows padded to the longest one: columns and values, for products with plain torch."""
    n, ln = len(IA) - 1, np.diff(IA)
    w = int(ln.max())
    k = np.arange(len(JA)) - np.repeat(IA[:-1], ln)
    rows = np.repeat(np.arange(n), ln)
    col, val = np.zeros((n, w), np.int64), np.zeros((n, w))
    col[rows, k], val[rows, k] = JA, AA
    col, val = torch.from_numpy(col).to(dev), torch.from_numpy(val).to(dev)
    return lambda x: (val * x[col]).sum(1)


def _bicgstab(mv, prec, f, tol=1e-14, restarts=30, its=400):
    """Right-preconditioned BiCGSTAB in 64 bits, restarted on the true residual."""
    x, nf, best = torch.zeros_like(f), f.norm(), None
    for _ in range(restarts):
        r = f - mv(x)
        if best is None or r.norm() < best[0]:
            best = (r.norm(), x.clone())
        if best[0] <= tol * nf:
            break
        x, target = best[1].clone(), max(tol * nf, 1e-6 * best[0])
        r = f - mv(x)
        r0, p, rr = r.clone(), r.clone(), None
        rr = r0 @ r
        for _ in range(its):
            ph = prec(p)
            v = mv(ph)
            a = rr / (r0 @ v)
            s = r - a * v
            sh = prec(s)
            t = mv(sh)
            w = (t @ s) / (t @ t)
            x, r = x + a * ph + w * sh, s - w * t
            if r.norm() <= target or not torch.isfinite(r).all():
                break
            rn = r0 @ r
            p = r + (rn / rr) * (a / w) * (p - w * v)
            rr = rn
    return best[1]


def _ilu_solve(IA, JA, AA, f):
    """U^-1 L^-1 f with the ILU(0) factors of the serial row elimination."""
    IA, JA, n = IA.tolist(), JA.tolist(), len(IA) - 1
    rows, up, f = [], [], f.tolist()
    AA = AA.tolist()
    y = [0.0] * n
    for i in range(n):
        w = dict(zip(JA[IA[i]:IA[i + 1]], AA[IA[i]:IA[i + 1]]))
        yi = f[i]
        for k in JA[IA[i]:IA[i + 1]]:
            if k >= i:
                break
            d, rest = up[k]
            m = w[k] / d
            for j, v in rest:
                if j in w:
                    w[j] -= m * v
            yi -= m * y[k]
        y[i] = yi
        up.append((w[i], [(j, v) for j, v in w.items() if j > i]))
    z = [0.0] * n
    for i in range(n - 1, -1, -1):
        d, rest = up[i]
        s = y[i]
        for j, v in rest:
            s -= v * z[j]
        z[i] = s / d
    return np.array(z)


def exact(case, seed):
    kind = case["kind"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a))
    if kind in ("transient", "steady_assembly"):
        S, x, y, ubc, u, du, dt = _transport_inputs(case, seed)
        if kind == "steady_assembly":
            Ke, Fe = _transport_elements(S, x, y, ubc, u, None, TT["k"], case["cau"], 1.0, 0.0)
            return {"F": t(_row_sum(S, Fe, 1)[:S["neq"]]), "AA": t(np.append(_csr_sum(S, Ke), 0.0))}
        Ae, Re = _transport_elements(S, x, y, ubc, u, du, TT["k"], case["cau"], 0.0, TT["alpha"] * dt)
        R, AA = _row_sum(S, Re, 1), _csr_sum(S, Ae)
        d = _row_diag(S, AA)
        dg = t(d).to(dev)
        X = _bicgstab(_ell(S["IA"], S["JA"], AA, dev), lambda v: v / dg, t(R[:-1]).to(dev)).cpu()
        if case["solver"] == "mixed":
            return {"R": t(R), "X": X}
        return {"R": t(R), "B": t(_ilu_solve(S["IA"], S["JA"], AA, R[:-1])), "X": X}
    if kind in ("ns_assembly", "ns_ilu"):
        S, x, y, presc, u, f = _ns_inputs(case, seed)
        Ke, Fe = _ns_elements(S, x, y, presc, u, f, case["Re"])
        F, AA = _row_sum(S, Fe, 3), _csr_sum(S, Ke)
        if kind == "ns_assembly":
            return {"F": t(F), "AA": t(np.append(AA, 0.0))}
        return {"F": t(_ilu_solve(S["IA"], S["JA"], AA, F[:-1]))}
    if kind in ("euler_setup", "euler_step"):
        S, x, y, presc, u, du, pb = _euler_inputs(case, seed)
        lm = t(S["lm"].reshape(-1, 12).astype(np.int64)).to(dev)
        if kind == "euler_setup":
            Ae, Re = _euler_elements(S, x, y, presc, u, du, pb)
            R = _row_sum(S, Re, 4)
            Z = _apply_blocks(S, _block_inverses(S, Ae, len(x)), R[:-1])
            Ad = t(Ae.reshape(-1, 12, 12))
            return {"Ae": Ad, "R": t(R), "Z": t(Z), "Q": _ebe_product(lm, Ad.to(dev), t(Z).to(dev), S["neq"]).cpu()}
        al, dt = pb["alpha"], pb["dt"]
        u = u + (1 - al) * dt * du
        a = np.zeros_like(u)
        for _ in range(2):
            Ae, Re = _euler_elements(S, x, y, presc, u, a, pb)
            Ad = t(Ae.reshape(-1, 12, 12)).to(dev)
            inv = t(_block_inverses(S, Ae, len(x))).to(dev)
            m = t(S["type"] != 0).to(dev)
            eq = t(S["inv"].astype(np.int64)).to(dev)[m]

            def prec(v):
                full = torch.zeros(len(S["type"]), dtype=F64, device=dev)
                full[m] = v[eq]
                z = (inv * full.reshape(-1, 1, 4)).sum(2).reshape(-1)
                out = torch.zeros_like(v)
                out[eq] = z[m]
                return out

            Da = _bicgstab(lambda v: _ebe_product(lm, Ad, v, S["neq"]), prec, t(_row_sum(S, Re, 4)[:-1]).to(dev),
                           tol=1e-13).cpu().numpy()
            a = a + Da
            u = u + al * dt * Da
        return {"u": t(u), "a": t(a)}
    if kind == "csrmv":
        S = _structure(case["mx"], case["my"], case["ndof"], True)
        rng = np.random.default_rng([seed, 5])
        AA = rng.standard_normal(S["nnz"])
        p = rng.standard_normal(S["neq"]).astype(np.float64 if case["dtype"] == "f64" else np.float32)
        return t(np.add.reduceat(AA * p.astype(np.float64)[S["JA"]], S["IA"][:-1]))
    if kind == "ebemv":
        S = _structure(case["mx"], case["my"], case["ndof"], False)
        s = 3 * case["ndof"]
        p = np.random.default_rng([seed, 6]).standard_normal(S["neq"])
        p = p.astype(np.float64 if case["dtype"] == "f64" else np.float32).astype(np.float64)
        lm = t(S["lm"].reshape(-1, s).astype(np.int64)).cuda()
        return _ebe_product(lm, _ebe_values(case, seed, len(lm)), t(p).cuda(), S["neq"]).cpu()
    xs = []
    for S, AA, F in _requests(case["systems"], case["nmin"], case["nmax"], seed):
        D = torch.zeros(S["neq"], S["neq"], dtype=F64)
        D[t(np.repeat(np.arange(S["neq"]), np.diff(S["IA"]))), t(S["JA"].astype(np.int64))] = t(AA)
        xs.append(torch.linalg.solve(D.to(dev), t(F).to(dev)).cpu())
    return torch.cat(xs)


def _row_diag(S, AA):
    rows = np.repeat(np.arange(S["neq"]), np.diff(S["IA"]))
    return AA[S["JA"] == rows]
