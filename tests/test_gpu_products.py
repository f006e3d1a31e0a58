"""The large-matrix default of the FP64 CSR products (staged through LDS) against a 64-bit numpy sum:
slices cut by the last row, uneven rows, columns within and beyond 16-bit distances, a slice too dense
for it, and the fused residual of the mixed solver."""
import numpy as np
import pytest

from parallel_fem_codes_amd import fem

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_cuda():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def banded(n, offsets, keep, rng, dense_rows=()):
    """CSR pattern: row i holds i and a random part of i + offsets; dense_rows hold 60 entries each."""
    off = np.unique(np.concatenate([[0], offsets]))
    col = np.arange(n)[:, None] + off[None, :]
    ok = (col >= 0) & (col < n) & ((rng.random(col.shape) < keep) | (off == 0)[None, :])
    if len(dense_rows):
        ok[list(dense_rows)] = False
    ln = ok.sum(1)
    for i in dense_rows:
        ln[i] = 60
    IA = np.concatenate([[0], np.cumsum(ln)])
    JA = np.empty(IA[-1], np.int64)
    r, c = np.nonzero(ok)
    k = np.arange(len(r)) - np.searchsorted(r, r, side="left")
    JA[IA[r] + k] = col[r, c]
    for i in dense_rows:
        lo = min(max(i - 30, 0), n - 60)
        JA[IA[i]:IA[i + 1]] = np.arange(lo, lo + 60)
    return IA.astype(np.int32), JA.astype(np.int32)


@pytest.mark.parametrize("n,offsets,keep,dense", [
    (320001, [-600, -599, -1, 1, 599, 600], 1.0, False),        # the 7-point stencil, one row past a slice
    (320063, [-600, -599, -1, 1, 599, 600, 7, -9], 0.9, False),   # uneven rows, a slice of 63 rows
    (320256, [-70000, -599, -1, 1, 599, 70000], 1.0, False),    # columns beyond 16 bits
    (120000, list(range(-12, 13)), 0.8, False),                 # rows of about 20
    (320001, [-600, -599, -1, 1, 599, 600], 1.0, True),         # a slice of 64 x 60 entries: lanes per row
])
def test_large_csr_products(torch_cuda, n, offsets, keep, dense):
    torch = torch_cuda
    rng = np.random.default_rng(n)
    IA, JA = banded(n, offsets, keep, rng, range(64 * 11, 64 * 12) if dense else ())
    assert len(JA) > 2 << 20
    dev = fem.Device(0)
    A = fem.CsrMatrix(dev, IA, JA)
    AA = rng.standard_normal(len(JA))
    A.set_values(AA)
    p = rng.standard_normal(n)
    prod = AA * p[JA]
    ref = np.add.reduceat(prod, IA[:-1])
    # each row: at most len roundings of partial sums bounded by the row's sum of |products|
    bound = 64 * np.finfo(np.float64).eps * np.add.reduceat(np.abs(prod), IA[:-1])
    q = torch.full((n,), float("nan"), dtype=torch.float64, device="cuda")
    A.csrmv(torch.from_numpy(p).cuda(), q)
    assert (np.abs(q.cpu().numpy() - ref) <= bound).all()


@pytest.mark.parametrize("offsets", [list(range(-12, 13)), [-600, -599, -1, 1, 599, 600]])
def test_autotune_times_the_default(torch_cuda, offsets):
    """A large matrix, with and without sliced ELL: the default is among the candidates, the kept kernel is
    the fastest measured, and -1 brings the default back (its sums, bit for bit)."""
    torch = torch_cuda
    n = 120000 if len(offsets) > 16 else 320001
    rng = np.random.default_rng(n)
    IA, JA = banded(n, offsets, 1.0, rng)
    dev = fem.Device(0)
    A = fem.CsrMatrix(dev, IA, JA)
    A.set_values(rng.standard_normal(len(JA)))
    p = torch.from_numpy(rng.standard_normal(n)).cuda()
    default, q = torch.empty_like(p), torch.empty_like(p)
    A.csrmv(p, default)
    lanes, us = A.autotune()
    assert set(us) == {-1, 1, 2, 4, 8, 16} | ({0} if len(offsets) <= 16 else set())
    assert us[lanes] == min(us.values())
    A.set_lanes(16)
    A.set_lanes(-1)
    A.csrmv(p, q)
    assert torch.equal(q, default)
    empty = fem.CsrMatrix(dev, np.zeros(1, np.int32), np.zeros(0, np.int32))
    assert empty.autotune()[0] == -1   # nothing to time: the default stays


def test_large_residual(torch_cuda):
    """The mixed solver on a diagonally dominant matrix of that size: its FP64 residual (the staged
    kernel with the fused norm) is the one numpy computes."""
    torch = torch_cuda
    n = 320001
    rng = np.random.default_rng(2)
    IA, JA = banded(n, [-600, -599, -1, 1, 599, 600], 1.0, rng)
    AA = 0.1 * rng.standard_normal(len(JA))
    rows = np.repeat(np.arange(n), np.diff(IA))
    AA[JA == rows] = 2.0
    F = rng.standard_normal(n)
    dev = fem.Device(0)
    A = fem.CsrMatrix(dev, IA, JA)
    A.set_values(AA)
    X = torch.empty(n, dtype=torch.float64, device="cuda")
    info = fem.gmres_mixed(dev, A, torch.from_numpy(F).cuda(), X, tol=1e-10, sweep_mode=2, factor_sweeps=2)
    r = F - np.add.reduceat(AA * X.cpu().numpy()[JA], IA[:-1])
    res = np.linalg.norm(r) / np.linalg.norm(F)
    assert info.status == 0 and res <= 1e-10
    assert abs(res - info.true_rel_residual) <= 1e-5 * res + 1e-16
