"""GPU: the network's routes give one another's bits: inference in one library
call, inference layer by layer (a layer replaced or wrapped by the program),
training with the fused passes between stages, training by separate passes."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def sg(shy):
    from simplehydrology_amd import surrogate
    return surrogate


def batch(n, h, w):
    gen = torch.Generator().manual_seed(h + w)
    x = torch.randn(n, h, w, 8, generator=gen).to(torch.bfloat16).cuda()
    return x, torch.randn(n, h, w, 3, generator=gen).cuda()


def step(sg, net, x, t):
    """One training step's output, gradients and weights."""
    y = net.forward(x)
    _, gy = sg.mse_loss_and_grad(y, t)
    net.backward(gy)
    net.step(2e-4)
    return [y] + [v.clone() for c in net.convs() for v in (c.dw, c.db, c.w)]


def same(a, b):
    return all(torch.equal(u, v) for u, v in zip(a, b))


# 8 pixels at the lowest level; ragged tiles on every level; tiles of 16 x 8 and (the
# last, 300 tiles of 16 x 16) of 16 x 16 pixels
@pytest.mark.parametrize("n,h,w", [(1, 8, 64), (1, 64, 64), (3, 104, 152), (2, 72, 200),
                                   (20, 48, 80)])
def test_inference_routes(sg, n, h, w):
    print("inference", n, h, w, flush=True)
    net = sg.UNet(seed=n)
    for c in net.convs():
        c.b.normal_()
    x, _ = batch(n, h, w)
    kept = net.forward(x)
    one = net.forward(x, keep=False)
    assert net._one_call() is not None
    assert torch.equal(one, kept) and torch.equal(net.forward(x, keep=False), kept)
    net.e[1].b.forward = net.e[1].b.forward  # a layer of the program's own
    assert net._one_call() is None
    assert torch.equal(net.forward(x, keep=False), kept)


@pytest.mark.parametrize("where", ["conv", "stage", "class"])
def test_wrapped_layer_takes_part_in_inference(sg, monkeypatch, where):
    print("wrapped", where, flush=True)
    net = sg.UNet(seed=4)
    x, _ = batch(2, 32, 48)
    want = net.forward(x, keep=False)
    calls = []

    def wrap(f, at):
        def g(*a, **kw):
            calls.append(at)
            return f(*a, **kw)
        return g

    if where == "conv":
        net.d[1].a.forward_upcat = wrap(net.d[1].a.forward_upcat, 0)
    elif where == "stage":
        net.e[3].forward = wrap(net.e[3].forward, 0)
    else:
        monkeypatch.setattr(sg.Conv, "forward_pool", wrap(sg.Conv.forward_pool, 0))
    assert torch.equal(net.forward(x, keep=False), want)
    assert len(calls) == (3 if where == "class" else 1)


def test_training_routes(sg):
    print("training", flush=True)
    x, t = batch(2, 40, 72)
    a, b = sg.UNet(seed=7), sg.UNet(seed=7)
    for s in b.e + b.d:
        # a program's own stage: forward and backward with their first arguments
        f, g = s.forward, s.backward
        s.forward = lambda x, shape, pool=False, head=None, _f=f: _f(x, shape, pool=pool, head=head)
        s.backward = lambda g, shape, scratch, need_dx=True, _g=g: _g(g, shape, scratch, need_dx)
    for _ in range(2):
        ra, rb = step(sg, a, x, t), step(sg, b, x, t)
        assert a.fused and not b.fused
        assert same(ra, rb)


def test_channels_of_other_networks(sg):
    class Wide(sg.UNet):
        CH = (64, 64, 96, 128)

    class Narrow(sg.UNet):
        CH = (32, 64, 96, 40)

    x, _ = batch(1, 16, 24)
    wide, narrow = Wide(seed=1), Narrow(seed=1)
    print("other channels", flush=True)
    for keep in (True, False):
        with pytest.raises(AssertionError):  # the fused head reads 32 channels
            wide.forward(x, keep=keep)
    # a lowest level that is no multiple of 32: its decoder's input is built
    narrow.forward(x)
    low, skip = narrow.e[3].saved[3], narrow.e[2].saved[3]
    assert torch.equal(narrow.d[2].saved[0], torch.cat(
        [low.repeat_interleave(2, 1).repeat_interleave(2, 2), skip], -1))
