"""Refined FP32 solves of densities with a mean, against long double transforms:
what is left of the mean in the residual must not set the error's floor.  The
grids run each kind of FP32 x pass that takes the sum (register engine, planes,
LDS lines, butterflies and dense stages of the mixed radices), each layout and the
batch modes, with the spectral symbol and the stencil's.

Tolerance: the floor of a refined solve is its FP64 residual's rounding, three
passes of about 2e-16 each way, in the modes that dominate the solution, whose share of
f can be ten times below the others': 10 * sqrt(6) * 2e-16 = 5e-15.  f - mean f is
exact to an ulp of the mean's constant, so the mean adds nothing."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
scipy_fft = pytest.importorskip("scipy.fft")

import fishfry_amd as ff  # noqa: E402

pytestmark = pytest.mark.gpu
TOL = 5e-15
L = np.longdouble


def exact(f, symbol):
    n = f.shape
    spec = scipy_fft.rfftn(f.astype(L))
    total = 0
    for a, m in enumerate(n):
        k = np.arange(m if a < 2 else m // 2 + 1)
        k = np.minimum(k, m - k).astype(L)
        extent = L(2 * np.pi - 2 * np.pi / m)
        if symbol == 0:
            lam = (k * (2 * L(np.pi) * (m - 1) / (m * extent))) ** 2
        else:
            s2 = np.sin(L(np.pi) * k / m) ** 2
            lam = 4 * s2 * (1 + s2 / 3 if symbol == ff.FF_SYMBOL_5PT else 1) * ((m - 1) / extent) ** 2
        total = total + lam.reshape([-1 if q == a else 1 for q in range(3)])
    total[0, 0, 0] = np.inf
    return scipy_fft.irfftn(-spec / total, s=n)


def err(phi, want):
    d = phi.astype(L) - want
    return float(np.sqrt((d * d).sum() / (want * want).sum()))


GRIDS = [(131, 6, 10), (6, 131, 10), (77, 26, 34), (32, 32, 32), (45, 20, 50), (30, 25, 27)]


def solve(p, f):
    d = torch.zeros(p.bytes() // 8, dtype=torch.float64, device="cuda")
    phi = torch.full_like(d, float("nan"))
    d[:f.size] = torch.from_numpy(f.reshape(-1)).cuda()
    print("mean", f.shape, p.refine_steps, flush=True)
    p.solve(p.bytes(), d, phi)
    return phi[:f.size].cpu().numpy().reshape(f.shape)


def plan(n, steps, flags):
    lo, hi, _ = ff.benchmark_grid(n)
    return ff.ParisPencil(n, lo, hi, precision=ff.FF_FP32_REFINE, refine_steps=steps, flags=flags)


@pytest.mark.parametrize("n", GRIDS)
def test_mean_of_f(n):
    rng = np.random.default_rng(5)
    plans = [plan(n, s, lay) for s in (2, 3) for lay in (0, ff.FF_PENCIL_LAYOUT)]
    for k in range(3):
        base = rng.standard_normal(n)
        base -= base.mean()
        for mean in (0.0, 1.0, 1000.0):
            f = base + mean
            want = exact(f, 0)
            for p in plans:
                e = err(solve(p, f), want)
                assert e < TOL, (k, mean, p.refine_steps, e)
    for p in plans:
        p.close()


@pytest.mark.parametrize("n", GRIDS)
def test_mean_adds_nothing(n):
    """The stencil's floor is higher by its own rounding (1/h^2 of phi's): a mean may add TOL
    to the error that the same density has without it."""
    rng = np.random.default_rng(5)
    p = plan(n, 2, ff.FF_SYMBOL_5PT)
    for k in range(3):
        base = rng.standard_normal(n)
        base -= base.mean()
        errs = [err(solve(p, base + mean), exact(base + mean, ff.FF_SYMBOL_5PT)) for mean in (0.0, 1.0)]
        assert errs[1] < errs[0] + TOL, (k, errs)
    p.close()


def test_batches_with_means():
    """Every batch mode, twice over the same buffers, to the bit of the single solves."""
    shapes = [(32, 32, 32), (77, 26, 34), (32, 32, 32), (48, 48, 48), (77, 26, 34)]
    rng = np.random.default_rng(9)
    fields = [rng.standard_normal(n) + 3.0 for n in shapes]
    want = []
    for n, f in zip(shapes, fields):
        p = plan(n, 3, 0)
        want.append(solve(p, f))
        p.close()
        assert err(want[-1], exact(f, 0)) < TOL
    for flags in (0, ff.FF_BATCH_GROUPED, ff.FF_BATCH_STEPS):
        b = ff.Batch([dict(n=n, precision=ff.FF_FP32_REFINE, refine_steps=3) for n in shapes], flags=flags)
        d = [torch.zeros(b.bytes(i) // 8, dtype=torch.float64, device="cuda") for i in range(len(shapes))]
        phi = [torch.full_like(x, float("nan")) for x in d]
        for x, f in zip(d, fields):
            x[:f.size] = torch.from_numpy(f.reshape(-1)).cuda()
        for _ in range(2):
            b.solve(d, phi)
            b.wait()
            for x, n, w in zip(phi, shapes, want):
                assert np.array_equal(x[:w.size].cpu().numpy().reshape(n), w), (flags, n)
        b.close()
