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


def check_cycles(shy, orc, h, drops, cycles, kw, flow=None, seed=3, root=None, block=256):
    """`cycles` eager cycles against the oracle: fields and statistics.  A
    walk block other than 256 keeps one lane per drop for few drops too."""
    nx, ny = h.shape
    z = np.zeros((nx, ny), np.float32)
    d, mx, my, erfd = z.copy(), z.copy(), z.copy(), z.copy()
    w = shy.World(nx, ny, seed=seed, params=shy.Params(**kw))
    w.set_tuning(walk_block=block)
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
@pytest.mark.parametrize("block", [256, 128])  # one wave, one lane per drop
def test_walk_arithmetic_ranges(shy, orc, kw, negative, block):
    rng = np.random.default_rng(11)
    nx, ny = 75, 66
    h = plane(nx, ny) + rng.uniform(0, 1e-3, (nx, ny)).astype(np.float32)
    d = rng.uniform(0, 12, (nx, ny)).astype(np.float32)
    if negative:
        d[5, 7] = -0.25
    mx = rng.normal(0, 2, (nx, ny)).astype(np.float32)
    my = rng.normal(0, 2, (nx, ny)).astype(np.float32)
    mx[::3], my[::3] = 0.0, 0.0  # cells without momentum: no coupling
    check_cycles(shy, orc, h, 300, 2, kw, flow=(d, mx, my), block=block)


@pytest.mark.parametrize("block", [256, 128])
def test_flat_cells(shy, orc, block):
    """Zero gravity terms and no momentum: drops stand still for 501 steps."""
    h = np.full((33, 70), 0.5, np.float32)
    check_cycles(shy, orc, h, 130, 2, dict(), block=block)


@pytest.mark.parametrize("nx,ny,drops,kw", [
    (1, 1, 64, dict()),                        # every step leaves the map
    (2, 300, 65, dict()),                      # windows clamped on both sides of an axis
    (64, 64, 256, dict()),
    (130, 67, 6144, dict()),                   # the most drops of one wave each
    (130, 67, 6145, dict()),                   # the first that are not
    (300, 220, 2560, dict()),                  # the same on a map of over 65536 cells
    (300, 220, 2561, dict()),
    (96, 80, 200, dict(maxAge=0.0)),           # one step
    (96, 80, 200, dict(maxAge=62.0)),          # 63 steps: a batch less one
    (96, 80, 200, dict(maxAge=63.0)),          # 64: a whole batch
    (96, 80, 200, dict(maxAge=64.0)),          # 65: one step into the next
    (96, 80, 200, dict(maxAge=700.0)),
    (96, 80, 200, dict(minVol=0.9)),           # ends by volume
    (96, 80, 200, dict(evapRate=-0.01, maxAge=100.0)),  # volumes above 1: full sequences
])
def test_few_drops(shy, orc, nx, ny, drops, kw):
    """Cycles of few drops run one wave per drop: batches of 64 steps, an 8x8
    window of records, commits by atomics."""
    rng = np.random.default_rng(nx + drops)
    h = orc.fbm(5, max(nx, 8), max(ny, 8))[:nx, :ny].copy()
    d, mx, my = (rng.uniform(0, 2, (nx, ny)).astype(np.float32) for _ in range(3))
    root = rng.uniform(0, 1.2, (nx, ny)).astype(np.float32)
    check_cycles(shy, orc, h, drops, 3, kw, flow=(d, mx - 1, my - 1), root=root)


def test_few_and_many_drops_alternate(shy, orc):
    """Both commit paths on one context: each leaves what the other expects."""
    n, seed = 96, 9
    h = orc.fbm(seed, n, n)
    z = np.zeros((n, n), np.float32)
    d, mx, my, root, erfd = z.copy(), z.copy(), z.copy(), z.copy(), z.copy()
    w = shy.World(n, n, seed=seed)
    w.upload("height", h)
    P = orc.Params.default()
    for c, (drops, graph) in enumerate([(300, False), (7000, False), (300, True), (300, True),
                                        (6200, True), (6200, True), (128, False)]):
        w.erode_cycles(1, drops, graph=graph)
        orc.wave_cycle(h, d, mx, my, root, erfd, P, seed, c, drops)
        for name, ref in (("height", h), ("discharge", d), ("momentumx", mx), ("momentumy", my)):
            assert np.array_equal(bits(w.field(name)), bits(ref)), (name, c)
    w.close()


def test_few_drops_ensemble(shy, orc):
    """Small terrains of uneven sides and parameters, one wave per drop, graph
    replays; each equals its own oracle cycles."""
    specs = [dict(nx=40, ny=33, drops=70, seed=3, kw=dict(evapRate=0.002)),
             dict(nx=64, ny=64, drops=256, seed=4, kw=dict(depositionRate=0.2)),
             dict(nx=17, ny=90, drops=5, seed=5, kw=dict(maxAge=130.0)),
             dict(nx=8, ny=8, drops=0, seed=6, kw=dict())]
    e = shy.Ensemble([dict(nx=s["nx"], ny=s["ny"], drops=s["drops"], seed=s["seed"],
                           params=shy.Params(**s["kw"])) for s in specs])
    state = []
    for i, s in enumerate(specs):
        n = max(s["nx"], s["ny"])
        h = orc.fbm(s["seed"], n, n)[:s["nx"], :s["ny"]].copy()
        e.upload(i, "height", h)
        z = np.zeros_like(h)
        state.append([h] + [z.copy() for _ in range(5)])
    e.erode(5, graph=True)
    for i, s in enumerate(specs):
        P = orc.Params.default(**s["kw"])
        steps = 0
        for c in range(5):
            h, d, mx, my, root, erfd = state[i]
            steps += orc.wave_cycle(h, d, mx, my, root, erfd, P, s["seed"], c, s["drops"],
                                    terrain=i).steps
        for name, ref in zip(("height", "discharge", "momentumx", "momentumy"), state[i]):
            assert np.array_equal(bits(e.field(i, name)), bits(ref)), (i, name)
        assert e.terrain_steps()[i] == steps, i
    e.close()


@pytest.mark.parametrize("nx,ny,drops,kw", [
    (64, 64, 6200, dict()),                   # every step in one tile: all parts are its
    (70, 64, 6200, dict(maxAge=3.0)),         # two tiles, fewer entries than one part's least
    (200, 136, 6200, dict(maxAge=120.0)),     # tiles of one part beside tiles of several
    (4400, 1000, 4500, dict(maxAge=30.0)),    # more tiles than the block listing them has threads
])
def test_tile_parts(shy, orc, nx, ny, drops, kw):
    """The tile kernels' work is cut by entries: tiles of one part, of
    several, and the sums of a tile's parts."""
    x, y = np.meshgrid(np.arange(nx), np.arange(ny), indexing="ij")
    # valleys, so that some tiles hold most of the steps
    h = (0.5 + 2e-4 * (np.abs(x % 97 - 48) + np.abs(y % 89 - 44))).astype(np.float32)
    check_cycles(shy, orc, h, drops, 2, kw)


@pytest.mark.parametrize("drops", [16384, 16385, 32768, 32769])
def test_walk_block_widths(shy, orc, drops):
    """Blocks of 64 threads up to 16384 drops, of 128 up to 32768, then 256."""
    h = orc.fbm(8, 200, 144)
    check_cycles(shy, orc, h, drops, 2, dict(maxAge=60.0))


@pytest.mark.parametrize("nx,ny,drops", [
    (60, 70, 1), (60, 70, 1023), (60, 70, 1025),  # blocks of 1024 drops
    (300, 9, 65536), (90, 130, 65537),            # one chunk and one drop more
    (1, 4097, 5000),                              # all bins along one axis
])
def test_drop_order_chunks(shy, nx, ny, drops):
    """The drop order is a permutation: no field and no count depends on it."""
    got = []
    for on in (True, False):
        w = shy.World(nx, ny, seed=4, params=shy.Params(maxAge=40.0))
        w.upload("height", plane(nx, ny))
        w.set_drop_order(on)
        say("order", on, nx, ny, drops)
        w.erode(drops)
        w.erode_cycles(4, drops)
        got.append([bits(w.field(f)) for f in ("height", "discharge", "momentumx", "momentumy")] +
                   [w.stats()])
        w.close()
    assert all(np.array_equal(a, b) for a, b in zip(got[0][:4], got[1][:4]))
    assert got[0][4] == got[1][4]
