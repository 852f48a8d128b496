"""Lengths with prime factors above 5 and odd-length rows (the mixed-radix pass
kernels) against the oracle and against the register engine's Bluestein path,
which a tuning override of the same length selects.

Line lengths: one stage of each kind (7, 11, 13; 17, 97), two and three stages,
two dense stages (289, 323), the largest dense radix of each precision (199;
293) and the next prime (211; 307: Bluestein), partial tiles, and odd rows with
ny odd and even (rows are transformed in pairs of one plane)."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import fishfry_amd as ff  # noqa: E402
import oracle  # noqa: E402

pytestmark = pytest.mark.gpu

TOL = 1e-13  # relative L2 against the oracle, as for every FP64 solve


def solve(f, **kw):
    n = f.shape
    lo, hi, _ = ff.benchmark_grid(n)
    plan = ff.ParisPencil(n, lo, hi, **kw)
    nb = plan.bytes()
    a = torch.zeros(nb // 8, dtype=torch.float64, device="cuda")
    b = torch.full_like(a, float("nan"))
    a[:f.size] = torch.from_numpy(f.reshape(-1)).cuda()
    plan.solve(nb, a, b)
    out = b[:f.size].cpu().numpy().reshape(n)
    plan.close()
    return out


def rel(x, y):
    return np.linalg.norm(x - y) / np.linalg.norm(y)


def field(n):
    f = np.random.default_rng(n[0] * 10007 + n[1] * 101 + n[2]).standard_normal(n)
    return f - f.mean()


LENGTHS = [7, 11, 13, 14, 17, 26, 34, 49, 66, 91, 97, 131, 169, 199, 211, 289, 293, 301, 307, 323, 385, 451, 1001]


@pytest.mark.parametrize("n", LENGTHS)
def test_column_and_row_lengths(n):
    """The length on each axis in turn: columns of y and x, packed rows (nz = 2n)
    and rows in pairs (odd nz)."""
    shapes = [(n, 6, 10), (5, n, 8), (3, 4, 2 * n)] + ([(4, 5, n), (3, 2, n)] if n % 2 else [])
    for g in shapes:
        print("mixed", g, flush=True)
        f = field(g)
        want = oracle.solve(f)
        assert rel(solve(f), want) < TOL, g
        assert rel(solve(f, precision=ff.FF_FP32_REFINE, refine_steps=2), want) < 1e-12, g
        assert rel(solve(f, precision=ff.FF_FP32_REFINE, refine_steps=0), want) < 1e-5, g


@pytest.mark.parametrize("nz", [3, 5, 9, 15, 27, 81, 243, 675])
def test_odd_smooth_rows(nz):
    for g in ((4, 6, nz), (3, 5, nz), (70, 3, nz)):
        print("odd rows", g, flush=True)
        f = field(g)
        assert rel(solve(f), oracle.solve(f)) < TOL, g


@pytest.mark.parametrize("n", [(77, 26, 34), (34, 91, 49), (14, 301, 17), (13, 7, 11), (119, 33, 38)])
@pytest.mark.parametrize("symbol", [0, ff.FF_SYMBOL_3PT, ff.FF_SYMBOL_5PT])
def test_against_bluestein(n, symbol):
    """Every layout and symbol: bit-identical to the plain layout, and as close
    to the oracle as the Bluestein path."""
    f = field(n)
    want = oracle.solve(f, symbol={0: 0, ff.FF_SYMBOL_3PT: 3, ff.FF_SYMBOL_5PT: 5}[symbol])
    M = n[2] if n[2] % 2 else n[2] // 2
    for prec, steps, tol in ((ff.FF_FP64, 0, TOL), (ff.FF_FP32_REFINE, 1, 1e-9)):
        layouts = [0, ff.FF_PENCIL_LAYOUT] + ([ff.FF_BLOCKED_LAYOUT, ff.FF_SLAB_PIPELINE] if prec == ff.FF_FP64 else [])
        outs = [solve(f, precision=prec, refine_steps=steps, flags=symbol | lay, slab_planes=3) for lay in layouts]
        for o in outs[1:]:
            assert np.array_equal(outs[0], o)
        assert rel(outs[0], want) < tol
        try:
            for kind, length in ((0, M), (3, M), (1, n[1]), (2, n[0])):
                for p in (0, 1):
                    t = ff.tune_query(kind, length, p, n[2] // 2 + 1)
                    ff.tune_set(kind, length, p, t.E, t.T, 0)
            blue = solve(f, precision=prec, refine_steps=steps, flags=symbol)
        finally:
            ff.tune_reset()
        assert rel(blue, want) < tol and rel(outs[0], blue) < tol


def test_batch_modes_bitwise():
    """Mixed-radix instances in the stream, grouped and step-batched modes."""
    shapes = [(77, 26, 34), (32, 32, 32), (77, 26, 34), (34, 91, 49), (64, 32, 98), (34, 91, 49)]
    for prec, steps in ((ff.FF_FP64, 0), (ff.FF_FP32_REFINE, 1)):
        ref = [solve(field(n), precision=prec, refine_steps=steps) for n in shapes]
        for flags in (0, ff.FF_BATCH_GROUPED, ff.FF_BATCH_STEPS):
            b = ff.Batch([dict(n=n, precision=prec, refine_steps=steps) for n in shapes], flags=flags)
            d, p = [], []
            for i, n in enumerate(shapes):
                a = torch.zeros(b.bytes(i) // 8, dtype=torch.float64, device="cuda")
                a[:n[0] * n[1] * n[2]] = torch.from_numpy(field(n).reshape(-1)).cuda()
                d.append(a)
                p.append(torch.full_like(a, float("nan")))
            b.solve(d, p)
            b.wait()
            for i, n in enumerate(shapes):
                got = p[i][:n[0] * n[1] * n[2]].cpu().numpy().reshape(n)
                assert np.array_equal(got, ref[i]), (flags, prec, n)
            b.close()
