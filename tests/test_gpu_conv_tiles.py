"""GPU: the persistent tile loop of the 3x3 convolutions at the edges of its
16 x 16 tiles (one pixel less, one tile, one more, left and right edge in one
tile), with each epilogue, against float64.

FP32 sums of at most 9 x 96 exact products: 1e-5 relative in norm is beyond
100 times their rounding.  BF16 results add at most half an ulp, 2^-9, per
value (two roundings where a residual follows the first)."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SIZES = [(260, 15, 16), (260, 16, 1), (70, 17, 33), (24, 47, 65), (300, 1, 15)]


def rand(*shape, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(*shape, generator=g).to(torch.bfloat16)


def conv64(x, w):
    """x [N,H,W,C] f64, w [Cout][9 Cin] tap-major -> [N,H,W,Cout]."""
    n, h, wd, c = x.shape
    xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1))
    w = w.reshape(-1, 9, c)
    return sum(xp[:, t // 3:t // 3 + h, t % 3:t % 3 + wd] @ w[:, t].T for t in range(9))


def close(y, ref, tol):
    assert float((y.double().cpu() - ref).norm()) <= tol * float(ref.norm())


@pytest.mark.parametrize("N,H,W", SIZES)
@pytest.mark.parametrize("cin,cout", [(32, 32), (64, 96)])
def test_forward_epilogues(shy, N, H, W, cin, cout):
    from simplehydrology_amd import surrogate as sg
    print("tiles", N, H, W, cin, cout, flush=True)
    L, s = sg.nn(), torch.cuda.current_stream().cuda_stream
    x, w, res = rand(N, H, W, cin, seed=1), rand(cout, 9 * cin, seed=2), rand(N, H, W, cout, seed=3)
    b = torch.randn(cout, generator=torch.Generator().manual_seed(4))
    xd, wd, rd, bd = (t.cuda().contiguous() for t in (x, w, res, b))
    ref = conv64(x.double(), w.double())
    yf = torch.full((N, H, W, cout), float("nan"), device="cuda")
    assert L.shy_nn_conv_fwd(xd.data_ptr(), wd.data_ptr(), bd.data_ptr(), None, None,
                             yf.data_ptr(), N, H, W, cin, cout, 9, 0, s) == 0
    close(yf, ref + b.double(), 1e-5)
    # BF16 with bias, residual and ReLU; guard rows behind the output
    y = torch.full((N * H * W + 64, cout), 7.0, dtype=torch.bfloat16, device="cuda")
    assert L.shy_nn_conv_fwd(xd.data_ptr(), wd.data_ptr(), bd.data_ptr(), rd.data_ptr(),
                             y.data_ptr(), None, N, H, W, cin, cout, 9, 1, s) == 0
    close(y[:N * H * W].view(N, H, W, cout), (ref + b.double() + res.double()).relu(), 2 ** -8)
    assert bool((y[N * H * W:] == 7.0).all())
    # the backward pass's residual and mask: the separate passes' bits
    plain = torch.empty(N, H, W, cout, dtype=torch.bfloat16, device="cuda")
    assert L.shy_nn_conv_fwd(xd.data_ptr(), wd.data_ptr(), None, None, plain.data_ptr(), None, N, H,
                             W, cin, cout, 9, 0, s) == 0
    close(plain, ref, 2 ** -8)
    mask = rand(N, H, W, cout, seed=5).cuda()
    for gres, mk in ((rd, mask), (None, mask), (rd, None)):
        got = torch.empty_like(plain)
        assert L.shy_nn_conv_dgrad(xd.data_ptr(), wd.data_ptr(), gres.data_ptr() if gres is not None
                                   else None, mk.data_ptr() if mk is not None else None,
                                   got.data_ptr(), N, H, W, cout, cin, 9, s) == 0
        want = plain if gres is None else (plain.float() + gres.float()).to(torch.bfloat16)
        if mk is not None:
            want = torch.where(mk > 0, want, torch.zeros_like(want))
        assert torch.equal(got, want)


@pytest.mark.parametrize("N,H,W,c1,c2,cout", [(70, 18, 34, 64, 32, 32), (260, 14, 16, 32, 64, 64),
                                              (130, 2, 32, 64, 32, 32)])
def test_upsampled_input(shy, N, H, W, c1, c2, cout):
    from simplehydrology_amd import surrogate as sg
    print("upcat", N, H, W, c1, c2, cout, flush=True)
    L, s = sg.nn(), torch.cuda.current_stream().cuda_stream
    xh, sk = rand(N, H // 2, W // 2, c1, seed=1), rand(N, H, W, c2, seed=2)
    w, res = rand(cout, 9 * (c1 + c2), seed=3), rand(N, H, W, cout, seed=4)
    d = [t.cuda().contiguous() for t in (xh, sk, w, res)]
    up = xh.double().repeat_interleave(2, 1).repeat_interleave(2, 2)
    ref = conv64(torch.cat([up, sk.double()], -1), w.double())
    for r in (None, d[3]):
        y = torch.empty(N, H, W, cout, dtype=torch.bfloat16, device="cuda")
        assert L.shy_nn_conv_fwd_upcat(d[0].data_ptr(), d[1].data_ptr(), d[2].data_ptr(), None,
                                       r.data_ptr() if r is not None else None, y.data_ptr(), None,
                                       N, H, W, c1, c2, cout, 0, s) == 0
        close(y, ref if r is None else ref + res.double(), 2 ** -8)


@pytest.mark.parametrize("X,Y,tile,halo,batch", [(64, 64, 64, 8, 4), (65, 97, 64, 8, 3),
                                                 (40, 300, 32, 4, 40), (33, 32, 32, 4, 16)])
def test_tiled_inference_passes(shy, X, Y, tile, halo, batch):
    """Features, windows, crops and decoding of the tiled inference against
    the element-wise passes, on strided maps with values below zero.  The math
    library's log1p and expm1 differ by at most 2 ulp each, which BF16 inputs
    pass on as half an ulp of theirs at most: the network's output moves by
    less than 2^-8 of its norm."""
    from simplehydrology_amd import surrogate as sg
    print("tiled", X, Y, tile, flush=True)
    g = torch.Generator().manual_seed(X)
    a = torch.randn(X, Y, 4, generator=g).cuda()
    a[..., 1:] *= 30.0
    h, d, mx, my = (a[..., k] for k in range(4))
    net = sg.UNet(seed=1)
    got = sg.predict_tiled(net, h, d, mx, my, tile=tile, halo=halo, batch=batch)
    # float64 maps take the element-wise passes; features() keeps float32
    want = sg.predict_tiled(net, h.double(), d, mx, my, tile=tile, halo=halo, batch=batch)
    for u, v in zip(got, want):
        assert u.shape == v.shape and u.dtype == torch.float32 and u.is_contiguous()
        assert float((u - v).norm()) <= 2 ** -8 * float(v.norm())
