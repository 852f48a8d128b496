"""The right-hand side and the error sums on grids whose tiles hold more than the
fewest planes (test_gpu_field.py's all hold four): 11 planes with a last tile of
4, and 64 with a last one of 2, rows and columns partial, for each number of
mode registers; 17 and 32 modes at 64 planes take the most LDS (76 KB).  Whole
planes of f against long double, the sums against FP64 products on the GPU."""
import math

import numpy as np
import pytest

from test_gpu_field import _outer, _terms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nmodes", [0, 16, 17, 32])
@pytest.mark.parametrize("n", [(37, 631, 450), (130, 1021, 520)])
def test_planes_per_tile(n, nmodes):
    import torch

    import fishfry_amd as ff

    across = -(-n[1] // 16) * -(-n[2] // 64)
    planes = max(4, min(64, n[0] * across // 1024))
    assert planes == {37: 11, 130: 64}[n[0]] and n[0] % planes
    rng = np.random.default_rng(31 * nmodes + n[2])
    f = ff.field_default(n)
    for a in range(3):
        f.shift[a] = float(rng.uniform(0, 2 * math.pi))
        f.dd[a] = 1.0
    f.scale = 1.5
    modes = [(rng.integers(-12, 13, 3), float(rng.standard_normal()), float(rng.standard_normal()))
             for _ in range(nmodes)]
    ff.field_set_modes(f, modes)
    axes, p, d = _terms(n, f)
    # each axis's angle is at most 12 * 3 pi, rounded once in the coordinate and once in the product
    amp = sum(abs(a) + abs(b) for _, a, b in modes)
    eps = 2.0 ** -53
    tol = amp * (3 * 2 * 113 + 16) * eps + 64 * math.exp(3) * f.scale * eps
    out = torch.full(n, float("nan"), dtype=torch.float64, device="cuda")
    print("field", n, nmodes, flush=True)
    ff.field_init(f, out)
    assert not torch.isnan(out).any()
    for i in sorted({0, 1, planes - 1, planes, n[0] - 1}):
        cut = [c[i:i + 1] if a == 0 else c for a, c in enumerate(axes)]
        px, dx = p[0][i:i + 1], d[0][i:i + 1]
        want = f.scale * (_outer(px, p[1], d[2]) + _outer(px, d[1], p[2]) + _outer(dx, p[1], p[2]))
        for k, a, b in modes:
            c, s = zip(*((np.cos(int(k[q]) * cut[q]), np.sin(int(k[q]) * cut[q])) for q in range(3)))
            re = (_outer(c[0], c[1], c[2]) - _outer(s[0], s[1], c[2]) - _outer(s[0], c[1], s[2])
                  - _outer(c[0], s[1], s[2]))
            im = (_outer(s[0], c[1], c[2]) + _outer(c[0], s[1], c[2]) + _outer(c[0], c[1], s[2])
                  - _outer(s[0], s[1], s[2]))
            want = want + a * re + b * im
        assert np.abs(out[i:i + 1].cpu().numpy() - want.astype(np.float64)).max() <= tol, i
    # the error sums against phi = 0: the potential's own norms, as sums of products of one factor per axis
    left, right = [f.scale * np.multiply.outer(p[0], p[1])], [p[2]]
    for k, a, b in modes:
        lam = float(sum(min(int(k[q]) % n[q], n[q] - int(k[q]) % n[q]) ** 2 for q in range(3)))
        iv = -1.0 / lam if lam else 0.0
        ex, ey, ez = ((np.cos(int(k[q]) * axes[q]), np.sin(int(k[q]) * axes[q])) for q in range(3))
        gx = (iv * (a * ex[0] + b * ex[1]), iv * (a * ex[1] - b * ex[0]))  # (a - ib) e^{ikx}
        left.append(np.multiply.outer(gx[0], ey[0]) - np.multiply.outer(gx[1], ey[1]))
        right.append(ez[0])
        left.append(-np.multiply.outer(gx[0], ey[1]) - np.multiply.outer(gx[1], ey[0]))
        right.append(ez[1])
    lt = torch.from_numpy(np.stack([v.reshape(-1) for v in left], 1).astype(np.float64)).cuda()
    rt = torch.from_numpy(np.stack(right).astype(np.float64)).cuda()
    pot = (lt @ rt).abs()
    N = pot.numel()
    tol += (2 * len(right) + 8) * eps * 2 * (amp + f.scale * math.exp(3))  # the products' own rounding
    one, two, top = float(pot.sum()), float((pot * pot).sum()), float(pot.max())
    got = ff.field_diff(f, torch.zeros(n, dtype=torch.float64, device="cuda"))
    assert abs(got[0] - one) <= N * tol + 1e-13 * one
    assert abs(got[1] - two) <= 2 * top * N * tol + 1e-13 * two
    assert abs(got[2] - top) <= tol
