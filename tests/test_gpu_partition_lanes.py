"""GPU: the step-log partition where cycles of few drops would not reach it, bit
for bit against the oracle.

Cycles of up to 6144 drops on small maps run one wave per drop and need no
partition; here they keep a lane per drop (a walk block other than the default),
or have more drops.  Rounds of 8192 slots serve terrains of up to 1024 tiles and
rounds of 4096 larger ones; both read the drops' step counts from memory where a
partition block has more than 4096 drops, which takes more than 512 x 4096 drops in
a walk that does not count."""
import numpy as np
import pytest

import test_gpu_partition as part

pytestmark = pytest.mark.gpu


def test_empty_and_parameter_change(shy, orc):
    P1, P2, P3 = (orc.Params.default() for _ in range(3))
    P2.evapRate, P2.maxAge = 0.0023, 300.0
    P3.maxAge = 700.0  # more log rows than the buffers held
    part.run_pair(shy, orc, 256, 9, [(4096, P1), (0, None), (4096, None), (4096, P2),
                                     (4096, None), (4096, P3), (4096, None)], walk_block=128)


# blocks of 128 on request; blocks of 64 and of 256 (in drop order) by the number of
# drops
@pytest.mark.parametrize("times,tuning", [(1, dict(walk_block=128, walk_grid=0, tile=0)),
                                          (1, dict(walk_block=64, walk_grid=0, tile=0)),
                                          (6, None), (40, None)])
def test_ensemble_shared_and_empty_terrains(shy, orc, times, tuning):
    specs = [dict(nx=nx, ny=ny, drops=dr * times, seed=300 + i)
             for i, (nx, ny, dr) in enumerate(part.MIXED)]
    part.ensemble_vs_oracle(shy, orc, specs, 2, tuning)


@pytest.mark.parametrize("n", [200, 2100])  # 16 (of at most 1024) and 1089 tiles
def test_block_steps_read_from_memory(shy, orc, n):
    drops, seed = 512 * 4096 + 1, 8
    P = orc.Params.default(maxAge=2.0)
    w = shy.World(n, n, seed=seed, params=shy.Params(maxAge=2.0))
    w.set_tuning(walk_block=256, walk_grid=700)
    w.generate_fbm(seed, 8)
    h = orc.fbm(seed, n, n)
    z = np.zeros_like(h)
    d, mx, my, root, erfd = z.copy(), z.copy(), z.copy(), z.copy(), z.copy()
    for c in range(2):
        print("steps from memory", n, "cycle", c, flush=True)
        w.reset_stats()
        w.erode(drops)
        st = orc.wave_cycle(h, d, mx, my, root, erfd, P, seed, c, drops)
        for name, ref in (("height", h), ("discharge", d), ("momentumx", mx), ("momentumy", my)):
            assert np.array_equal(part.bits(w.field(name)), part.bits(ref)), (n, c, name)
        assert w.stats() == st.as_dict()
    w.close()
