"""The walk's code paths give the oracle's bits at the edges of their ranges.

The count walk has a short arithmetic for operands in a stated range, a
per-step fallback inside it and a full-sequence walk for terrains outside it;
each case below drives one of them.  All comparisons are bit for bit: the
paths evaluate the same correctly rounded operations.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


def bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


def plane(nx, ny, a=3 / 1024, b=-2 / 1024):
    x, y = np.meshgrid(np.arange(nx), np.arange(ny), indexing="ij")
    return (0.5 + a * x / 4 + b * y / 4).astype(np.float32)


def check_cycles(shy, orc, h, drops, cycles, kw, flow=None, seed=3, root=None):
    """`cycles` eager cycles against the oracle: fields and statistics."""
    nx, ny = h.shape
    z = np.zeros((nx, ny), np.float32)
    d, mx, my, erfd = z.copy(), z.copy(), z.copy(), z.copy()
    w = shy.World(nx, ny, seed=seed, params=shy.Params(**kw))
    P = orc.Params.default(**kw)
    h = h.copy()
    w.upload("height", h)
    if flow is not None:
        d, mx, my = (f.copy() for f in flow)
        for name, f in (("discharge", d), ("momentumx", mx), ("momentumy", my)):
            w.upload(name, f)
        erfd = w.field("erf_discharge")
    if root is None:
        root = z.copy()
    else:
        w.upload("rootdensity", root)
    for c in range(cycles):
        say(h.shape, drops, kw, "cycle", c)
        w.reset_stats()
        w.erode(drops)
        st = orc.wave_cycle(h, d, mx, my, root, erfd, P, seed, c, drops)
        for name, ref in (("height", h), ("discharge", d), ("momentumx", mx), ("momentumy", my),
                          ("erf_discharge", erfd)):
            assert np.array_equal(bits(w.field(name)), bits(ref)), (name, c)
        assert w.stats() == st.as_dict(), c
    w.close()


@pytest.mark.parametrize("kw,negative", [
    (dict(), False),                           # the short arithmetic
    (dict(gravity=1e-17), False),              # first squared speed below 2^-100: repeated step
    (dict(gravity=3e16), False),               # squared speeds above 2^100: every step repeated
    (dict(momentumTransfer=1e-19), False),     # coupling numerators below 2^-60: repeated
    (dict(momentumTransfer=2e15), False),      # beyond 2^50: the full-sequence walk
    (dict(momentumTransfer=0.0), False),       # zero numerators stay on the short path
    (dict(), True),                            # a negative discharge flags the terrain
])
def test_walk_arithmetic_ranges(shy, orc, kw, negative):
    rng = np.random.default_rng(11)
    nx, ny = 75, 66
    h = plane(nx, ny) + rng.uniform(0, 1e-3, (nx, ny)).astype(np.float32)
    d = rng.uniform(0, 12, (nx, ny)).astype(np.float32)
    if negative:
        d[5, 7] = -0.25
    mx = rng.normal(0, 2, (nx, ny)).astype(np.float32)
    my = rng.normal(0, 2, (nx, ny)).astype(np.float32)
    mx[::3], my[::3] = 0.0, 0.0  # cells without momentum: no coupling
    check_cycles(shy, orc, h, 300, 2, kw, flow=(d, mx, my))


def test_flat_cells(shy, orc):
    """Zero gravity terms and no momentum: drops stand still for 501 steps."""
    h = np.full((33, 70), 0.5, np.float32)
    check_cycles(shy, orc, h, 130, 2, dict())
