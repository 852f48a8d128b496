"""Pass kernels with the line plan compiled in and twiddles in LDS, at every
2^a 3^b 5^c length from 36 to 1024 that has no other compiled-in kernel.  An
untuned plan takes them; a tuning override of the same elements per thread
with FF_TUNE_GENERIC selects the generic kernel, which performs the same
rounded operations, so every solve must agree with it to the bit: column
passes (x and y) and row passes, FP64 in the plain and pencil layouts, FP32
with a refinement step (the residual passes), and the finite-difference
symbol.  The default's result also meets the FP64 bound against the oracle.
Planes of 40 columns leave partial tiles and 20 rows partial workgroups at
the wider tiles; wider lines have one or several tiles to a plane."""
import json

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import fishfry_amd as ff  # noqa: E402
import oracle  # noqa: E402

pytestmark = pytest.mark.gpu
TOL = 1e-13


def smooth(m):
    for q in (2, 3, 5):
        while m % q == 0:
            m //= q
    return m == 1


COLS = [n for n in range(36, 1024) if smooth(n) and n not in (48, 64, 96, 128)]  # (160: x only)
ROWS = [m for m in range(18, 512) if smooth(m) and m not in (24, 32, 48, 64, 80, 128, 256, 384, 500)]
KINDS = [("fp64", {}), ("pencil", {"flags": ff.FF_PENCIL_LAYOUT}),
         ("fp32+1", {"precision": ff.FF_FP32_REFINE, "refine_steps": 1}),
         ("3pt", {"flags": ff.FF_SYMBOL_3PT}),
         ("fp32 5pt", {"precision": ff.FF_FP32_REFINE, "refine_steps": 1, "flags": ff.FF_SYMBOL_5PT})]


def solve(f, kw):
    n = f.shape
    lo, hi, _ = ff.benchmark_grid(n)
    p = ff.ParisPencil(n, lo, hi, **kw)
    d = json.loads(p.describe())
    nb = p.bytes()
    a = torch.zeros(nb // 8, dtype=torch.float64, device="cuda")
    b = torch.full_like(a, float("nan"))
    a[: f.size] = torch.from_numpy(f.reshape(-1)).cuda()
    p.solve(nb, a, b)
    torch.cuda.synchronize()
    out = b[: f.size].cpu().numpy().reshape(n)
    p.close()
    return out, d


def compare(n, keys, part):
    rng = np.random.default_rng(51)
    f = rng.standard_normal(n)
    for name, kw in KINDS:
        ff.tune_reset()
        print("lines", n, name, flush=True)
        got, d = solve(f, kw)
        try:
            for kind, length in keys:
                for prec in (0, 1):
                    cur = ff.tune_query(kind, length, prec, n[2] // 2 + 1)
                    ff.tune_set(kind, length, prec, cur.E, cur.T, ff.FF_TUNE_GENERIC)
            want, g = solve(f, kw)
        finally:
            ff.tune_reset()
        assert d[part]["E"] == g[part]["E"] and d[part]["lds"] != g[part]["lds"]  # another kernel of the same plan
        assert np.array_equal(got, want), (n, name, np.max(np.abs(got - want)))
        if name == "fp64":
            ref = oracle.solve(f)
            assert np.linalg.norm(got - ref) / np.linalg.norm(ref) < TOL


@pytest.mark.parametrize("length", COLS)
def test_columns(length):
    compare((length, 20, 78), [(2, length)], "x")
    if length != 160:
        compare((20, length, 78), [(1, length)], "y")


@pytest.mark.parametrize("m", ROWS)
def test_rows(m):
    compare((5, 7, 2 * m), [(0, m), (3, m)], "z")
