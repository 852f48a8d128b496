"""Which kernels a plan takes, as its description reports them: plane kernels for
the shapes and mixed radices for the lengths that test_gpu_plane.py and
test_gpu_mixed.py compare, so that those comparisons are with another kernel; none of
them under the overrides that those tests use, nor where a rule excludes them."""
import json

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import fishfry_amd as ff  # noqa: E402
import oracle  # noqa: E402
from test_gpu_mixed import LENGTHS  # noqa: E402
from test_gpu_plane import SHAPES  # noqa: E402

pytestmark = pytest.mark.gpu


def described(n, **kw):
    lo, hi, _ = ff.benchmark_grid(n)
    with ff.ParisPencil(n, lo, hi, **kw) as p:
        return json.loads(p.describe())


REFINED = dict(precision=ff.FF_FP32_REFINE, refine_steps=2)


@pytest.mark.parametrize("n", SHAPES)
def test_planes(n):
    assert described(n)["planes"] == [1, 0]
    assert described(n, **REFINED)["planes"] == [1, 1]
    for flags in (ff.FF_PENCIL_LAYOUT, ff.FF_BLOCKED_LAYOUT):
        assert described(n, flags=flags)["planes"] == [0, 0]
    try:
        for p in (0, 1):
            t = ff.tune_query(0, n[2] // 2, p, 1)
            ff.tune_set(0, n[2] // 2, p, t.E, t.T, 0)
        assert described(n)["planes"] == [0, 0]
        assert described(n, **REFINED)["planes"] == [0, 0]
    finally:
        ff.tune_reset()


def largest_prime(n):
    p, top = 2, 1
    while n > 1:
        while n % p == 0:
            n //= p
            top = p
        p += 1
    return top


@pytest.mark.parametrize("n", LENGTHS)
def test_mixed(n):
    top = largest_prime(n)
    # (pairs of FP64 rows to 300 only where their tiles fill the chip: test_engine_by_size)
    for prec, key, limit, pairs in ((0, "mixed", 200, 200), (1, "mixed_fp32", 300, 420)):
        kw = REFINED if prec else {}
        for g, axes, most in (((n, 6, 10), ["x"], limit), ((5, n, 8), ["y"], limit), ((3, 4, 2 * n), ["z", "zi"], limit),
                              ((4, 5, n), ["z", "zi"], pairs)):
            if g[2] == n and n % 2 == 0:
                continue
            got = described(g, **kw)[key]
            assert sorted(a for a in got if got[a]["n"] == n) == (sorted(axes) if top <= most else []), (g, key)
        # a plain FP32 solve stays on the register engine
        assert described((5, n, 8), precision=ff.FF_FP32_REFINE)["mixed_fp32"] == {}
        try:
            t = ff.tune_query(1, n, prec, 5)
            ff.tune_set(1, n, prec, t.E, t.T, 0)
            assert "y" not in described((5, n, 8), **kw)[key]
        finally:
            ff.tune_reset()


# length, axis and grid: mixed radices in FP64 and in refined FP32, or the register engine
SIZES = [
    # odd rows of 2^a 3^b 5^c: 3^k and 5^k, and 3^a 5^b of few and many engine passes
    ("z", (128, 128, 125), (0, 0)), ("z", (8, 8, 125), (0, 0)), ("z", (96, 97, 243), (0, 0)),
    ("z", (128, 128, 243), (1, 0)), ("z", (31, 45, 225), (1, 1)), ("z", (96, 97, 225), (1, 0)),
    ("z", (96, 97, 675), (1, 1)), ("z", (31, 45, 729), (0, 0)), ("z", (64, 64, 729), (1, 0)),
    # dense stages where the tiles do not fill the chip, and where they do
    ("z", (16, 48, 283), (0, 1)), ("z", (64, 66, 283), (1, 1)), ("x", (969, 20, 60), (0, 0)),
    ("y", (96, 969, 62), (0, 0)), ("y", (20, 566, 60), (0, 0)), ("y", (96, 566, 62), (0, 1)),
    ("y", (20, 493, 60), (1, 0)), ("y", (96, 493, 62), (1, 1)), ("y", (20, 398, 60), (0, 1)),
    ("y", (96, 398, 62), (1, 1)), ("x", (940, 20, 60), (1, 0)), ("x", (940, 96, 62), (1, 1)),
]


@pytest.mark.parametrize("axis,n,want", SIZES)
def test_engine_by_size(axis, n, want):
    got = (described(n)["mixed"], described(n, precision=ff.FF_FP32_REFINE, refine_steps=1)["mixed_fp32"])
    assert tuple(int(axis in g) for g in got) == want
    f = np.random.default_rng(sum(n)).standard_normal(n)
    w = oracle.solve(f)
    lo, hi, _ = ff.benchmark_grid(n)
    for kw in (dict(), REFINED):
        with ff.ParisPencil(n, lo, hi, **kw) as p:
            d = torch.zeros(p.bytes() // 8, dtype=torch.float64, device="cuda")
            phi = torch.full_like(d, float("nan"))
            d[:f.size] = torch.from_numpy(f.reshape(-1)).cuda()
            print("size", n, kw, flush=True)
            p.solve(p.bytes(), d, phi)
            e = np.linalg.norm(phi[:f.size].cpu().numpy().reshape(n) - w) / np.linalg.norm(w)
            assert e < (1e-13 if not kw else 1e-12), e  # as in test_gpu_mixed.py


@pytest.mark.parametrize("m", [72, 160, 320, 400, 500])
def test_row_lines_by_size(m):
    """Rows whose kernel depends on their number: the FP64 z inverse of some lengths is the generic
    one beyond 8192 rows, rows of 500 take their twiddles from LDS beyond them; one result."""
    def lds(n):
        d = described(n)
        try:
            for kind in (0, 3):
                t = ff.tune_query(kind, m, 0, m + 1)
                ff.tune_set(kind, m, 0, t.E, t.T, ff.FF_TUNE_GENERIC)
            g = described(n)
        finally:
            ff.tune_reset()
        return d["z"]["lds"] > g["z"]["lds"], d["zi"]["lds"] > g["zi"]["lds"]

    few, many = (64, 128, 2 * m), (64, 129, 2 * m)
    assert lds(few) == ((False, False) if m == 500 else (True, True))
    assert lds(many) == ((True, True) if m == 500 else (True, False))
    f = torch.from_numpy(np.random.default_rng(m).standard_normal(many)).cuda()
    lo, hi, _ = ff.benchmark_grid(many)
    out = []
    for tuned in (0, 1):
        try:
            for kind in (0, 3) if tuned else ():
                t = ff.tune_query(kind, m, 0, m + 1)
                ff.tune_set(kind, m, 0, t.E, t.T, ff.FF_TUNE_GENERIC)
            with ff.ParisPencil(many, lo, hi) as p:
                d = torch.zeros(p.bytes() // 8, dtype=torch.float64, device="cuda")
                d[:f.numel()] = f.reshape(-1)
                out.append(torch.full_like(d, float("nan")))
                p.solve(p.bytes(), d, out[-1])
        finally:
            ff.tune_reset()
    assert torch.equal(out[0][:f.numel()], out[1][:f.numel()])


def test_groups_and_long_descriptions():
    """Planes that a group fills the chip with, and a batch whose plans' descriptions are long."""
    b = ff.Batch([dict(n=(40, 128, 128))] * 5, flags=ff.FF_BATCH_GROUPED)
    d = [torch.zeros(b.bytes(i) // 8, dtype=torch.float64, device="cuda") for i in range(5)]
    p = [torch.zeros_like(x) for x in d]
    b.solve(d, p)
    b.wait()
    got = json.loads(b.describe())
    assert [g["planes"] for g in got["groups"]] == [[1, 0]] and got["plans"][0]["planes"] == [0, 0]
    b.close()
    shapes = [(1001, 924, 819 + 2 * k) for k in range(48)]
    b = ff.Batch([dict(n=n) for n in shapes])
    assert [tuple(q["n"]) for q in json.loads(b.describe())["plans"]] == shapes
    b.close()
