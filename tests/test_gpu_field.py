"""The right-hand side and the error sums of the driver kernels at sizes around
their tiles (16 rows by 64 columns, up to 64 planes; 16 or 32 modes), against
extended-precision numpy."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _terms(n, f):
    """Coordinates, analytic factors (FishFry.hpp:22-44, 71-86) and mode factors in long double."""
    L = np.longdouble
    axes = [np.array([f.lo[a] + i * f.d[a] + f.shift[a] for i in range(n[a])]).astype(L) for a in range(3)]
    x, y, z = axes
    px, py, pz = np.cos(x) * np.exp(np.sin(x)), np.sin(y) * np.exp(np.cos(y)), np.cos(z) * np.exp(np.cos(z))
    dpx = -np.exp(np.sin(x)) * np.sin(x) * np.cos(x) * (np.sin(x) + 3)
    dpy = np.sin(y) * np.exp(np.cos(y)) * (np.sin(y) ** 2 - 3 * np.cos(y) - 1)
    dpz = np.exp(np.cos(z)) * (3 * np.sin(z) ** 2 - np.cos(z) ** 3 - 1)
    return axes, (px, py, pz), (dpx, dpy, dpz)


def _outer(a, b, c):
    return a[:, None, None] * b[None, :, None] * c[None, None, :]


@pytest.mark.parametrize("nmodes", [0, 1, 16, 17, 32])
@pytest.mark.parametrize("n", [(1, 1, 1), (2, 3, 5), (5, 16, 64), (9, 17, 65), (70, 33, 130)])
def test_field_tiles(n, nmodes):
    import torch

    import fishfry_amd as ff

    rng = np.random.default_rng(17 * nmodes + n[2])
    f = ff.field_default(n)
    for a in range(3):
        f.shift[a] = float(rng.uniform(0, 2 * math.pi))
        f.dd[a] = 1.0
    f.scale = 1.5
    modes = [(rng.integers(-12, 13, 3), float(rng.standard_normal()), float(rng.standard_normal()))
             for _ in range(nmodes)]
    ff.field_set_modes(f, modes)
    axes, p, d = _terms(n, f)
    want = f.scale * (_outer(p[0], p[1], d[2]) + _outer(p[0], d[1], p[2]) + _outer(d[0], p[1], p[2]))
    pot = f.scale * _outer(*p)
    for k, a, b in modes:
        th = sum(int(k[c]) * axes[c].reshape([-1 if q == c else 1 for q in range(3)]) for c in range(3))
        v = a * np.cos(th) + b * np.sin(th)
        want = want + v
        folded = [min(int(k[c]) % n[c], n[c] - int(k[c]) % n[c]) for c in range(3)]
        lam = float(sum(q * q for q in folded))
        pot = pot + (-v / lam if lam else 0 * v)
    # each axis's angle is at most 12 * 3 pi, rounded once in the coordinate and
    # once in the product: 2 * 113 * 2^-53 per axis and unit of amplitude; the
    # analytic factors (below e^2 in all) carry a few roundings each
    amp = sum(abs(a) + abs(b) for _, a, b in modes)
    eps = 2.0 ** -53
    tol = amp * (3 * 2 * 113 + 16) * eps + 64 * math.exp(3) * f.scale * eps
    out = torch.full(n, float("nan"), dtype=torch.float64, device="cuda")
    ff.field_init(f, out)
    assert np.abs(out.cpu().numpy() - want.astype(np.float64)).max() <= tol
    # the error sums of a known phi: e = potential - phi
    phi = rng.standard_normal(n)
    got = ff.field_diff(f, torch.from_numpy(phi).cuda())
    e = np.abs(pot - phi)
    N = e.size
    assert abs(got[0] - float(e.sum())) <= N * tol + 1e-13 * float(e.sum())
    assert abs(got[1] - float((e * e).sum())) <= 2 * float(e.max()) * N * tol + 1e-13 * float((e * e).sum())
    assert abs(got[2] - float(e.max())) <= tol
