"""GPU: convolutions of rows beyond the tile loop's 31-bit offsets run on the
one-tile kernel, with the fused head too, and need no output of their own for it
(64 channels: from 838861 pixels on).

A convolution of one row of pixels equals the one of any part of it away from the
part's ends: the sums of a pixel run over its neighbours alone, in an order that
does not depend on where it lies, so parts computed by the tile loop give the
same bits."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
np = pytest.importorskip("numpy")


@pytest.mark.parametrize("cin,W", [(64, 838860), (64, 838861), (32, 838900)])
@pytest.mark.parametrize("with_y", [False, True])
def test_head_of_a_long_row(shy, cin, W, with_y):
    from simplehydrology_amd import surrogate as sg
    print("head", cin, W, with_y, flush=True)
    gen = torch.Generator().manual_seed(W)
    conv = sg.Conv(cin, 32, 9, np.random.default_rng(0), "cuda:0")
    head = sg.Conv(32, 8, 1, np.random.default_rng(1), "cuda:0")
    conv.b.copy_(torch.randn(32, generator=gen))
    head.b.copy_(torch.randn(8, generator=gen))
    x = torch.randn(1, 1, W, cin, generator=gen).to(torch.bfloat16).cuda()
    res = torch.randn(1, 1, W, 32, generator=gen).to(torch.bfloat16).cuda()
    y, out = conv.forward_head(x, (1, 1, W), head, res=res, keep=with_y)
    assert with_y == (y is not None)
    part = 4096
    for a in (0, 400000, W - part):
        xs, rs = x[:, :, a:a + part].contiguous(), res[:, :, a:a + part].contiguous()
        yp, op = conv.forward_head(xs, (1, 1, part), head, res=rs)
        lo, hi = (0 if a == 0 else 1), (part if a + part == W else part - 1)
        assert torch.equal(out[:, :, a + lo:a + hi], op[:, :, lo:hi]), a
        if with_y:
            assert torch.equal(y[:, :, a + lo:a + hi], yp[:, :, lo:hi]), a
