"""The batch autotuner's overrides (kept by pass kind and line length, for every
plan) configure the register engine's passes: no plan leaves its plane kernels or
mixed radices for one, whichever grids it was recorded on, results stay what they are,
and a batch is not left slower than it was."""
import json

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import fishfry_amd as ff  # noqa: E402
import oracle  # noqa: E402

pytestmark = pytest.mark.gpu


def described(n, **kw):
    lo, hi, _ = ff.benchmark_grid(n)
    with ff.ParisPencil(n, lo, hi, **kw) as p:
        return json.loads(p.describe())


def buffers(b):
    d = [torch.zeros(b.bytes(i) // 8, dtype=torch.float64, device="cuda") for i in range(b.count)]
    return d, [torch.zeros_like(x) for x in d]


# grids whose passes are tuned, and others with their line lengths
TUNED = [(128, 128, 128), (64, 96, 150), (100, 160, 96), (96, 128, 200), (128, 108, 160)]
PLANES = [(192, 128, 64), (192, 64, 128), (32, 32, 32), (100, 40, 96), (20, 48, 100), (192, 108, 80)]
REFINED = dict(precision=ff.FF_FP32_REFINE, refine_steps=1)


def test_other_plans_keep_their_kernels():
    before = [(described(n)["planes"], described(n, **REFINED)["planes"]) for n in PLANES]
    odd = [described((20, 30, 75), **kw) for kw in ({}, REFINED)]
    assert all(q == ([1, 0], [1, 1]) for q in before) and "z" in odd[0]["mixed"] and "z" in odd[1]["mixed_fp32"]
    try:
        for kw in ({}, dict(precision=ff.FF_FP32_REFINE)):
            b = ff.Batch([dict(n=n, **kw) for n in TUNED])
            d, p = buffers(b)
            print("autotune", kw, b.autotune(d, p, reps=2), flush=True)
            b.close()
        assert [(described(n)["planes"], described(n, **REFINED)["planes"]) for n in PLANES] == before
        assert "z" in described((20, 30, 75))["mixed"] and "z" in described((20, 30, 75), **REFINED)["mixed_fp32"]
        # (FP32 plans without refinement run 97 on the register engine, refined ones in mixed radices)
        b = ff.Batch([dict(n=(64, 97, 64), precision=ff.FF_FP32_REFINE)])
        d, p = buffers(b)
        print("autotune 97", b.autotune(d, p, reps=2), flush=True)
        b.close()
        assert "y" in described((64, 97, 64), **REFINED)["mixed_fp32"]
    finally:
        ff.tune_reset()


@pytest.mark.parametrize("flags", [0, ff.FF_BATCH_GROUPED, ff.FF_BATCH_STEPS])
def test_batch_keeps_its_kernels(flags):
    """Groups that run planes together (their plans alone do not), beside grids of the same lengths."""
    shapes = [(128, 128, 128), (96, 96, 96), (128, 64, 96), (128, 128, 128), (96, 96, 96), (48, 36, 50)]
    rng = np.random.default_rng(3)
    fields = [rng.standard_normal(n) for n in shapes]
    b = ff.Batch([dict(n=n) for n in shapes], flags=flags)
    d, p = buffers(b)
    b.solve(d, p)
    b.wait()
    groups = [g["planes"] for g in json.loads(b.describe())["groups"]]
    plans = [q["planes"] for q in json.loads(b.describe())["plans"]]
    try:
        tuned, before, after = b.autotune(d, p, reps=3)
        print("autotune", flags, tuned, before, after, flush=True)
        assert tuned >= 3 and before > 0 and after > 0
        for x, f in zip(d, fields):
            x[:f.size] = torch.from_numpy(f.reshape(-1)).cuda()
        b.solve(d, p)
        b.wait()
        got = json.loads(b.describe())
        assert [g["planes"] for g in got["groups"]] == groups and [q["planes"] for q in got["plans"]] == plans
        if flags == ff.FF_BATCH_GROUPED:
            assert all(g == [1, 0] for g in groups)
        for x, f in zip(p, fields):
            w = oracle.solve(f)
            assert np.linalg.norm(x[:f.size].cpu().numpy().reshape(f.shape) - w) < 1e-13 * np.linalg.norm(w)
    finally:
        ff.tune_reset()
        b.close()
