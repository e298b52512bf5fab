"""GPU: the gradients of a convolution of [up2(xh), skip] where memory holds one
partial only, or the gradient lies unaligned: the bits of the ones of the
concatenated input."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
np = pytest.importorskip("numpy")

N, H, W, C1, C2, COUT = 2, 18, 34, 64, 32, 32


@pytest.fixture(scope="module")
def data(shy):
    gen = torch.Generator().manual_seed(3)
    xh, sk, g = (torch.randn(*s, generator=gen).to(torch.bfloat16).cuda()
                 for s in ((N, H // 2, W // 2, C1), (N, H, W, C2), (N, H, W, COUT)))
    x = torch.cat([xh.repeat_interleave(2, 1).repeat_interleave(2, 2), sk], -1).contiguous()
    return xh, sk, x, g


@pytest.mark.parametrize("partials", [1, 2, 3])
def test_small_scratch(data, partials):
    from simplehydrology_amd import surrogate as sg
    xh, sk, x, g = data
    conv = sg.Conv(C1 + C2, COUT, 9, np.random.default_rng(0), "cuda:0")
    scratch = sg.Scratch("cuda:0", max_floats=partials * conv.w.numel())
    print("partials", partials, flush=True)
    got = []
    for inp in (x, (xh, sk)):
        conv.dw.fill_(float("nan"))
        conv.db.fill_(float("nan"))
        conv.backward(inp, g, (N, H, W), scratch, need_dx=False)
        got.append((conv.dw.clone(), conv.db.clone()))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    # the call that keeps the bias sums' partials in the same memory
    L = sg.nn()
    dw, db = torch.full_like(conv.dw, float("nan")), torch.full_like(conv.db, float("nan"))
    assert L.shy_nn_conv_wgrad_bias_upcat(
        xh.data_ptr(), sk.data_ptr(), g.data_ptr(), dw.data_ptr(), db.data_ptr(),
        scratch.part.data_ptr(), partials, N, H, W, C1, C2, COUT, sg._stream()) == 0
    ref = torch.empty_like(conv.dw)
    assert L.shy_nn_conv_wgrad(x.data_ptr(), g.data_ptr(), ref.data_ptr(), scratch.part.data_ptr(),
                               partials, N, H, W, C1 + C2, COUT, 9, sg._stream()) == 0
    assert torch.equal(dw, ref) and torch.equal(db, got[0][1])


def test_unaligned_gradient(data):
    from simplehydrology_amd import surrogate as sg
    xh, sk, x, g = data
    off = torch.empty(g.numel() + 1, dtype=torch.bfloat16, device="cuda")
    gu = off[1:].view(g.shape)
    gu.copy_(g)
    conv = sg.Conv(C1 + C2, COUT, 9, np.random.default_rng(0), "cuda:0")
    scratch = sg.Scratch("cuda:0")
    print("unaligned", gu.data_ptr() % 16, flush=True)
    conv.backward(x, gu, (N, H, W), scratch, need_dx=False)
    dw, db = conv.dw.clone(), conv.db.clone()
    conv.dw.fill_(float("nan"))
    conv.db.fill_(float("nan"))
    conv.backward((xh, sk), gu, (N, H, W), scratch, need_dx=False)
    assert torch.equal(conv.dw, dw) and torch.equal(conv.db, db)
