"""Plane kernels (the z and y passes of whole planes as one) against the passes
one by one, which a tuning override of the row length selects: the same
operations, so the results are bit-identical."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import fishfry_amd as ff  # noqa: E402
import oracle  # noqa: E402

pytestmark = pytest.mark.gpu


def solve(f, **kw):
    n = f.shape
    lo, hi, _ = ff.benchmark_grid(n)
    plan = ff.ParisPencil(n, lo, hi, **kw)
    nb = plan.bytes()
    a = torch.zeros(nb // 8, dtype=torch.float64, device="cuda")
    b = torch.full_like(a, float("nan"))
    a[:f.size] = torch.from_numpy(f.reshape(-1)).cuda()
    stamps = []
    plan.solve(nb, a, b, stamps)
    assert len(stamps) == 14 and all(s[1] <= t[1] for s, t in zip(stamps, stamps[1:]))
    out = b[:f.size].cpu().numpy().reshape(n)
    if kw.get("flags", 0) & ff.FF_PRESERVE_INPUT:
        assert np.array_equal(a[:f.size].cpu().numpy().reshape(n), f)
    plan.close()
    return out


# one plane to a workgroup: idle threads in rows and in columns, the smallest
# and largest planes, every row and column length, planes that need 128 of them
SHAPES = [(3, 32, 32), (2, 36, 50), (5, 160, 32), (4, 128, 48), (3, 48, 128), (7, 40, 80), (2, 50, 100), (3, 64, 72),
          (2, 72, 36), (3, 80, 40), (2, 96, 64), (3, 100, 48), (2, 108, 50), (2, 32, 108), (3, 40, 96),
          (192, 128, 128), (192, 160, 64), (192, 108, 108), (193, 96, 100)]


@pytest.mark.parametrize("n", SHAPES)
def test_planes_bitwise(n):
    f = np.random.default_rng(sum(n)).standard_normal(n)
    f -= f.mean()
    S3 = ff.FF_SYMBOL_3PT
    cases = [dict(), dict(flags=ff.FF_PRESERVE_INPUT), dict(flags=S3),
             dict(precision=ff.FF_FP32_REFINE, refine_steps=0), dict(precision=ff.FF_FP32_REFINE, refine_steps=2),
             dict(precision=ff.FF_FP32_REFINE, refine_steps=1, flags=S3)]
    print("planes", n, flush=True)
    got = [solve(f, **c) for c in cases]
    try:
        for p in (0, 1):
            t = ff.tune_query(0, n[2] // 2, p, 1)
            ff.tune_set(0, n[2] // 2, p, t.E, t.T, 0)
        want = [solve(f, **c) for c in cases]
    finally:
        ff.tune_reset()
    for c, g, w in zip(cases, got, want):
        assert np.array_equal(g, w), c
    assert np.linalg.norm(got[0] - oracle.solve(f)) < 1e-13 * np.linalg.norm(got[0])


def test_group_fills_the_chip():
    """Four 40x128x128 instances: passes alone, planes as one group of 160."""
    n = (40, 128, 128)
    for prec, steps in ((ff.FF_FP64, 0), (ff.FF_FP32_REFINE, 1)):
        fs = [np.random.default_rng(k).standard_normal(n) for k in range(5)]
        ref = [solve(f, precision=prec, refine_steps=steps) for f in fs]
        b = ff.Batch([dict(n=n, precision=prec, refine_steps=steps)] * len(fs), flags=ff.FF_BATCH_GROUPED)
        d = [torch.zeros(b.bytes(i) // 8, dtype=torch.float64, device="cuda") for i in range(len(fs))]
        p = [torch.full_like(x, float("nan")) for x in d]
        for x, f in zip(d, fs):
            x[:f.size] = torch.from_numpy(f.reshape(-1)).cuda()
        b.solve(d, p)
        b.wait()
        for x, r in zip(p, ref):
            assert np.array_equal(x[:r.size].cpu().numpy().reshape(n), r)
        b.close()
