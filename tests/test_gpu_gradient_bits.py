"""GPU: the network's gradients keep their bits, and are sums of what they claim.

tests/golden/gradient_hashes.json holds digests of the gradients of single layers
and of the first steps of two training runs (make_gradient_hashes.py beside it
says with which kernels and why the bits count).  The second test compares every
gradient of one ragged step with float64 sums over the BF16 tensors that the
step itself used.
"""
import importlib.util
import json
import os

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden")
_spec = importlib.util.spec_from_file_location("make_gradient_hashes",
                                               os.path.join(HERE, "make_gradient_hashes.py"))
make = importlib.util.module_from_spec(_spec)
_spec.loader.exec_module(make)


@pytest.fixture(scope="module")
def golden():
    with open(os.path.join(HERE, "gradient_hashes.json")) as f:
        return json.load(f)


@pytest.fixture(scope="module")
def sg(shy):
    from simplehydrology_amd import surrogate
    return surrogate


@pytest.mark.parametrize("dims", make.LAYERS)
def test_layer_gradient_bits(sg, golden, dims):
    print("layer", dims, flush=True)
    assert make.layer(sg, *dims) == golden["layers"][make.key(*dims)]


@pytest.mark.parametrize("dims", make.RUNS)
def test_training_run_bits(sg, golden, dims):
    print("run", dims, flush=True)
    want = golden["runs"][make.key(*dims)]
    for k, (got, ref) in enumerate(zip(make.run(sg, *dims), want)):
        assert got == ref, k


def test_ragged_step_gradients_are_the_float64_sums(sg):
    """3 x 104 x 152: 13 x 19 pixels at the lowest level.  A product passes at
    most 32 additions inside its MFMA, 4 MFMAs per tile of 16 x 8 pixels of its
    range (5 of 390 tiles in 92 ranges on the largest level, 12 in one range on
    the lowest), and ranges / 8 + 8 additions of the partials: at most 32 + 48 + 9.
    The first and last layer sum 17 x 32 pixels in 92 ranges, 32 + 17 + 20.  A bias
    term passes at most 12 rows and twice 10 folds and an addition between.  So
    under 96 roundings, each of half an ulp (2^-24) of a partial sum that the sum
    of the magnitudes bounds."""
    n, h, w = 3, 104, 152
    gen = torch.Generator().manual_seed(5)
    net = sg.UNet(seed=2, device="cuda:0")
    seen = []
    for c in net.convs():
        def rec(x, g, *a, _c=c, _f=c.backward, **kw):
            seen.append((_c, x, g))
            return _f(x, g, *a, **kw)
        c.backward = rec
    x = torch.randn(n, h, w, 8, generator=gen).to(torch.bfloat16).cuda()
    y = net.forward(x)
    _, gy = sg.mse_loss_and_grad(y, torch.randn(n, h, w, 3, generator=gen).cuda())
    net.backward(gy)
    assert len(seen) == 22
    for c, x, g in seen:
        if isinstance(x, tuple):
            x = torch.cat([x[0].repeat_interleave(2, 1).repeat_interleave(2, 2), x[1]], -1)
        hh, ww = x.shape[1:3]
        x, g = x.double(), g.double()
        if c.taps == 9:
            xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
            cols = [xp[:, t // 3:t // 3 + hh, t % 3:t % 3 + ww] for t in range(9)]
        else:
            cols = [x]
        g2 = g.reshape(-1, c.cout)
        ref = torch.cat([g2.t() @ v.reshape(-1, c.cin) for v in cols], 1)
        mag = torch.cat([g2.t().abs() @ v.reshape(-1, c.cin).abs() for v in cols], 1)
        print("gradient", c.cin, c.cout, hh, ww, flush=True)
        assert bool(((c.dw.double() - ref).abs() <= 96 * 2.0 ** -24 * mag).all())
        assert bool(((c.db.double() - g2.sum(0)).abs() <= 96 * 2.0 ** -24 * g2.abs().sum(0)).all())
