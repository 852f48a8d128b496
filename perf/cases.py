"""Workloads the solver's speed is measured on.

Each case is one pass of a user's program through the Python entry points:
a solve of one grid (``ParisPencil.solve_async``), a batch of small grids
(``Batch.solve``) or the right-hand side evaluated on the device
(``field_init``).  The sizes are those of the benchmark, its precision,
batching and serving workloads and the reference's example run.

  listed()            the named cases
  draw(rng)           one more case of the same ranges
  prepare(case, seed) plan, inputs and output buffers on the GPU
  run(state)          one pass; returns its outputs
  work(case)          bytes and flops one pass cannot do without
  exact(case, seed)   the outputs by torch's FP64 transforms
"""
import math

import torch

import fishfry_amd as ff

# The batching workload's grids (the cubes and the one non-cubic shape).
BATCH_SHAPES = [(32, 32, 32), (48, 48, 48), (64, 64, 64), (96, 96, 96), (128, 128, 128), (160, 160, 160),
                (128, 64, 96)]
BATCH_FLAGS = {"streams": 0, "grouped": ff.FF_BATCH_GROUPED, "steps": ff.FF_BATCH_STEPS}
SYMBOLS = {"spectral": 0, "3pt": ff.FF_SYMBOL_3PT, "5pt": ff.FF_SYMBOL_5PT}
# Points of the largest grid of any case.
MAX_POINTS = 1024 ** 3
# Largest grid with an extent that has a prime factor above 5 (serving).
MAX_RAGGED_POINTS = 385 ** 3
MODES = 16  # extra Fourier modes of f, 1 <= |k| <= 12


def _solve(name, n, refine=-1, symbol="spectral"):
    """refine: -1 an FP64 solve, otherwise FP32 passes with that many FP64-residual corrections."""
    return {"name": name, "kind": "solve", "nx": n[0], "ny": n[1], "nz": n[2], "refine": refine, "symbol": symbol}


def listed():
    return [
        # The reference's plain solve at its smallest: five launches, all latency.
        _solve("f64_64", (64, 64, 64)),
        # The reference's example run (bjob.sh): a non-cubic grid, one time step of a simulation.
        _solve("f64_128x256x384", (128, 256, 384)),
        # The plain method at the benchmark's sizes: what one GPU is given.
        _solve("f64_512", (512, 512, 512)),
        _solve("f64_1000", (1000, 1000, 1000)),
        _solve("f64_1024", (1024, 1024, 1024)),
        # FP32 passes with FP64-accurate results: an ordinary grid and the headline one.
        _solve("f32r2_256", (256, 256, 256), refine=2),
        _solve("f32r2_1024", (1024, 1024, 1024), refine=2),
        # The 5-point finite-difference symbol: FP32 passes and one stencil-residual correction reach its accuracy.
        _solve("f32r1_5pt_512", (512, 512, 512), refine=1, symbol="5pt"),
        # Grids as requests bring them: any integer extents, non-cubic, odd, in both precisions.
        _solve("f64_385x301x338", (385, 301, 338)),
        _solve("f32r2_131x97x150", (131, 97, 150), refine=2),
        # Many small grids at once, with new densities for every pass.
        {"name": "batch_f64", "kind": "batch", "count": 32, "mode": "grouped", "refine": -1, "shapes": 20261202},
        # f of the precision and serving workloads, evaluated on the device for a request.
        {"name": "field_484", "kind": "field", "nx": 484, "ny": 484, "nz": 484},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _smooth(v):
    """The nearest 2^a 3^b 5^c extent at or below v."""
    while True:
        m = v
        for p in (2, 3, 5):
            while m % p == 0:
                m //= p
        if m == 1:
            return v
        v -= 1


def draw(rng):
    kind = rng.choice(["smooth", "smooth", "ragged", "ragged", "batch", "field"])
    if kind == "batch":
        return {"kind": "batch", "count": rng.randint(8, 32), "mode": rng.choice(sorted(BATCH_FLAGS)),
                "refine": rng.choice([-1, 0, 2]), "shapes": rng.randrange(1 << 30)}
    hi = 1024 if kind == "smooth" else 512
    cap = MAX_POINTS if kind == "smooth" else 512 ** 3 if kind == "field" else MAX_RAGGED_POINTS
    while True:
        if rng.random() < 0.5:
            n = [_log_int(rng, 32, hi)] * 3
        else:
            n = [_log_int(rng, 32, hi) for _ in range(3)]
        if kind == "smooth":
            n = [_smooth(v) for v in n]
        if n[0] * n[1] * n[2] <= cap:
            break
    if kind == "field":
        return {"kind": "field", "nx": n[0], "ny": n[1], "nz": n[2]}
    return {"kind": "solve", "nx": n[0], "ny": n[1], "nz": n[2], "refine": rng.choice([-1, -1, 0, 1, 2]),
            "symbol": rng.choice(["spectral", "spectral", "3pt", "5pt"])}


def _modes(gen):
    """MODES distinct wave vectors with 1 <= |k| <= 12 (+-k counted once) and N(0,1) amplitudes."""
    got, seen = [], set()
    while len(got) < MODES:
        k = tuple(torch.randint(-12, 13, (3,), generator=gen).tolist())
        if not 1 <= sum(v * v for v in k) <= 144 or k in seen or tuple(-v for v in k) in seen:
            continue
        seen.add(k)
        a, b = torch.randn(2, generator=gen, dtype=torch.float64).tolist()
        got.append((k, a, b))
    return got


def _axes(n, shift):
    """Cell coordinates of the benchmark grid, shifted, on the GPU."""
    return [-math.pi + torch.arange(n[a], dtype=torch.float64, device="cuda") * (2.0 * math.pi / n[a]) + shift[a]
            for a in range(3)]


def _analytic_terms(n, shift):
    """The benchmark's f as a sum of three products of one factor per axis."""
    x, y, z = _axes(n, shift)
    cx, sx, cy, sy, cz, sz = x.cos(), x.sin(), y.cos(), y.sin(), z.cos(), z.sin()
    ex, ey, ez = sx.exp(), cy.exp(), cz.exp()
    px, dpx = cx * ex, -ex * sx * cx * (sx + 3.0)
    py, dpy = sy * ey, sy * ey * (sy * sy - 3.0 * cy - 1.0)
    pz, dpz = cz * ez, ez * (3.0 * sz * sz - cz * cz * cz - 1.0)
    return [(px, py, dpz), (px, dpy, pz), (dpx, py, pz)]


def _mode_terms(n, shift, modes):
    """a cos(k.x) + b sin(k.x) as products of one factor per axis."""
    x, y, z = _axes(n, shift)
    out = []
    for k, a, b in modes:
        ex, ey, ez = (torch.polar(torch.ones_like(t), kk * t) for kk, t in zip(k, (x, y, z)))
        # Re((a - ib) ex ey ez), split over the real and imaginary parts of the x and z factors
        cx = torch.complex(torch.tensor(a, dtype=torch.float64), torch.tensor(-b, dtype=torch.float64)).to(ex) * ex
        out += [(cx.real, ey.real, ez.real), (-cx.imag, ey.imag, ez.real),
                (-cx.imag, ey.real, ez.imag), (-cx.real, ey.imag, ez.imag)]
    return out


def _fill(out, n, terms):
    """out[i, j, k] += sum of the products, plane by plane (a matrix product per block of planes)."""
    fx, fy, fz = (torch.stack([t[a] for t in terms]) for a in range(3))
    step = max(1, (1 << 26) // (n[1] * len(terms)))
    for i in range(0, n[0], step):
        m = min(step, n[0] - i)
        left = (fx[:, i:i + m, None] * fy[:, None, :]).reshape(len(terms), m * n[1]).t().contiguous()
        out[i:i + m].reshape(m * n[1], n[2]).addmm_(left, fz)


def _density(out, n, seed):
    """The precision workload's f -- the analytic field at a random phase and scale plus 16 random modes --
    with a broadband part, as densities deposited from particles have one."""
    cpu = torch.Generator().manual_seed(seed)
    gpu = torch.Generator(device="cuda").manual_seed(seed)
    shift = (torch.rand(3, generator=cpu, dtype=torch.float64) * 2.0 * math.pi).tolist()
    scale = 0.5 + 1.5 * float(torch.rand(1, generator=cpu, dtype=torch.float64))
    torch.randn(n, generator=gpu, dtype=torch.float64, device="cuda", out=out)
    out.mul_(0.1)
    terms = [(scale * tx, ty, tz) for tx, ty, tz in _analytic_terms(n, shift)]
    _fill(out, n, terms + _mode_terms(n, (0.0, 0.0, 0.0), _modes(cpu)))


def _batch_shapes(case):
    gen = torch.Generator().manual_seed(case["shapes"])
    return [BATCH_SHAPES[i] for i in torch.randint(0, len(BATCH_SHAPES), (case["count"],), generator=gen).tolist()]


def _extents(case):
    return case["nx"], case["ny"], case["nz"]


def _precision(case):
    return dict(precision=ff.FF_FP64 if case["refine"] < 0 else ff.FF_FP32_REFINE, refine_steps=max(0, case["refine"]))


def _prepare_solve(case, seed):
    n = _extents(case)
    points = n[0] * n[1] * n[2]
    lo, hi, _ = ff.benchmark_grid(n)
    flags = SYMBOLS[case["symbol"]] | (ff.FF_PRESERVE_INPUT if case["refine"] < 0 else 0)
    plan = ff.ParisPencil(n, lo, hi, flags=flags, **_precision(case))
    nbytes = plan.bytes()
    f = torch.empty(nbytes // 8, dtype=torch.float64, device="cuda")
    phi = torch.empty_like(f)
    _density(f[:points].view(n), n, seed)
    return {"kind": "solve", "plan": plan, "bytes": nbytes, "f": f, "phi": phi, "out": phi[:points].view(n)}


def _prepare_batch(case, seed):
    shapes = _batch_shapes(case)
    batch = ff.Batch([dict(n=n, **_precision(case)) for n in shapes], flags=BATCH_FLAGS[case["mode"]])
    words = [batch.bytes(i) // 8 for i in range(len(shapes))]
    # one allocation for all densities and one for all potentials, each grid on a 256-byte boundary
    starts = [0]
    for w in words:
        starts.append(starts[-1] + (w + 31) // 32 * 32)
    source, density, phi = (torch.zeros(starts[-1], dtype=torch.float64, device="cuda") for _ in range(3))
    for i, n in enumerate(shapes):
        _density(source[starts[i]:starts[i] + n[0] * n[1] * n[2]].view(n), n, seed * 1009 + i)
    cut = lambda buf: [buf[starts[i]:starts[i] + words[i]] for i in range(len(shapes))]  # noqa: E731
    outs = [phi[starts[i]:starts[i] + n[0] * n[1] * n[2]].view(n) for i, n in enumerate(shapes)]
    return {"kind": "batch", "batch": batch, "source": source, "density": density, "densities": cut(density),
            "potentials": cut(phi), "out": outs}


def _prepare_field(case, seed):
    n = _extents(case)
    modes = _modes(torch.Generator().manual_seed(seed))
    field = ff.field_set_modes(ff.field_default(n), modes)
    return {"kind": "field", "field": field, "out": torch.empty(n, dtype=torch.float64, device="cuda")}


def prepare(case, seed):
    return {"solve": _prepare_solve, "batch": _prepare_batch, "field": _prepare_field}[case["kind"]](case, seed)


def run(state):
    if state["kind"] == "solve":
        state["plan"].solve_async(state["bytes"], state["f"], state["phi"])
    elif state["kind"] == "batch":
        # an FP64 batch overwrites its densities: every pass brings new ones
        state["density"].copy_(state["source"])
        state["batch"].solve(state["densities"], state["potentials"])
    else:
        ff.field_init(state["field"], state["out"])
    return state["out"]


def _solve_flops(n, refine, symbol):
    """5 N log2 N per forward and inverse transform pair of real data and 10 N for the filter; a spectral
    correction takes two more pairs, a finite-difference one a pair and the stencil."""
    points = n[0] * n[1] * n[2]
    pair = 5.0 * points * math.log2(points) + 10.0 * points
    r = max(0, refine)
    return pair * (1 + r * (2 if symbol == "spectral" else 1)) + (0 if symbol == "spectral" else 20.0 * r * points)


def work(case):
    if case["kind"] == "batch":
        shapes = _batch_shapes(case)
        points = sum(a * b * c for a, b, c in shapes)
        # the source read, the density written and read, the potential written
        return {"bytes": 32.0 * points, "flops": sum(_solve_flops(n, case["refine"], "spectral") for n in shapes)}
    n = _extents(case)
    points = n[0] * n[1] * n[2]
    if case["kind"] == "field":
        # the analytic part and every mode as products of per-axis factors
        return {"bytes": 8.0 * points, "flops": (6.0 + 4.0 * MODES) * points}
    return {"bytes": 16.0 * points, "flops": _solve_flops(n, case["refine"], case["symbol"])}


def _eigenvalues(n, symbol):
    """Per axis, the (non-negative) eigenvalues of -L_h on the half spectrum of the benchmark grid."""
    out = []
    for a in range(3):
        extent = 2.0 * math.pi - 2.0 * math.pi / n[a]  # from the first cell to the last
        k = torch.arange(n[a] if a < 2 else n[2] // 2 + 1, dtype=torch.float64, device="cuda")
        if symbol == "spectral":
            lam = (torch.minimum(k, n[a] - k) * (2.0 * math.pi * (n[a] - 1) / (n[a] * extent))) ** 2
        else:
            s2 = torch.sin(math.pi * torch.minimum(k, n[a] - k) / n[a]) ** 2
            lam = 4.0 * s2 * (1.0 if symbol == "3pt" else 1.0 + s2 / 3.0) * ((n[a] - 1) / extent) ** 2
        out.append(lam)
    return out


def _exact_solve(n, seed, symbol):
    f = torch.empty(n, dtype=torch.float64, device="cuda")
    _density(f, n, seed)
    spec = torch.fft.rfftn(f)
    del f
    lx, ly, lz = _eigenvalues(n, symbol)
    for i in range(n[0]):  # plane by plane: no array of all eigenvalues
        lam = lx[i] + ly[:, None] + lz[None, :]
        if i == 0:
            lam[0, 0] = math.inf
        spec[i] /= -lam
    return torch.fft.irfftn(spec, s=n)


def exact(case, seed):
    if case["kind"] == "solve":
        return _exact_solve(_extents(case), seed, case["symbol"])
    if case["kind"] == "batch":
        return [_exact_solve(n, seed * 1009 + i, "spectral") for i, n in enumerate(_batch_shapes(case))]
    n = _extents(case)
    out = torch.zeros(n, dtype=torch.float64, device="cuda")
    modes = _modes(torch.Generator().manual_seed(seed))
    _fill(out, n, _analytic_terms(n, (0.0, 0.0, 0.0)) + _mode_terms(n, (0.0, 0.0, 0.0), modes))
    return out
