"""GPU: weight and bias gradients at the edges of the 32 x 4 pixel tiles (one
pixel less, exactly one tile, one more), of the output channels per block
(32 or 64) and of the partials (one split, one tile each).

FP32 sums of exact bf16 products: against float64 the relative error of a sum
of P products is at most P ulp/2 and about sqrt(P) ulp/2 for these random
ones; 1e-5 is beyond 100 times that for the largest P here (3 x 11 x 70)."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
np = pytest.importorskip("numpy")


@pytest.mark.parametrize("N,H,W,cin,cout", [
    (1, 1, 1, 32, 32), (1, 3, 31, 32, 64), (1, 4, 32, 64, 32), (2, 5, 33, 32, 96),
    (1, 8, 64, 64, 64), (3, 11, 70, 96, 128), (1, 2, 200, 32, 32), (1, 60, 3, 32, 64),
])
@pytest.mark.parametrize("splits", [1, 2, 512])
def test_wgrad_and_bias_at_tile_edges(shy, N, H, W, cin, cout, splits):
    from simplehydrology_amd import surrogate as sg
    print("wgrad", N, H, W, cin, cout, splits, flush=True)
    gen = torch.Generator().manual_seed(H * W + cout)
    x = torch.randn(N, H, W, cin, generator=gen).to(torch.bfloat16)
    g = torch.randn(N, H, W, cout, generator=gen).to(torch.bfloat16)
    xd, gd = x.cuda().contiguous(), g.cuda().contiguous()
    dw = torch.full((cout, 9 * cin), float("nan"), device="cuda")
    db = torch.full((cout,), float("nan"), device="cuda")
    part = torch.full((splits * cout * 9 * cin,), float("nan"), device="cuda")
    bpart = torch.empty(1024 * cout, device="cuda")
    L, s = sg.nn(), torch.cuda.current_stream().cuda_stream
    rc = L.shy_nn_conv_wgrad_bias(xd.data_ptr(), gd.data_ptr(), dw.data_ptr(), db.data_ptr(),
                                  part.data_ptr(), splits, bpart.data_ptr(), 1024, N, H, W, cin,
                                  cout, 9, s)
    assert rc == 0, L.shy_nn_last_error()
    torch.cuda.synchronize()
    xr = torch.nn.functional.pad(x.double(), (0, 0, 1, 1, 1, 1))
    ref = torch.stack([torch.einsum("nhwo,nhwi->oi", g.double(), xr[:, dy:dy + H, dx:dx + W])
                       for dy in range(3) for dx in range(3)], 1).reshape(cout, 9 * cin)
    assert float((dw.cpu().double() - ref).norm()) <= 1e-5 * float(ref.norm())
    bref = g.double().sum((0, 1, 2))
    assert float((db.cpu().double() - bref).norm()) <= 1e-5 * float(bref.norm())
    # the weight gradient alone: the same tiles
    dw2 = torch.full_like(dw, float("nan"))
    rc = L.shy_nn_conv_wgrad(xd.data_ptr(), gd.data_ptr(), dw2.data_ptr(), part.data_ptr(), splits,
                             N, H, W, cin, cout, 9, s)
    assert rc == 0, L.shy_nn_last_error()
    assert float((dw2.cpu().double() - ref).norm()) <= 1e-5 * float(ref.norm())


@pytest.mark.parametrize("N,H,W,c1,c2,cout", [(1, 2, 2, 32, 32, 32), (2, 6, 34, 64, 32, 32),
                                              (1, 18, 64, 32, 64, 64)])
def test_wgrad_of_upsampled_input(shy, N, H, W, c1, c2, cout):
    """The gradients of a convolution of [up2(xh), skip], read from the two
    tensors: the bits of the ones from the concatenated input."""
    from simplehydrology_amd import surrogate as sg
    print("wgrad upcat", N, H, W, c1, c2, cout, flush=True)
    gen = torch.Generator().manual_seed(H * W + cout)
    xh, sk, g = (torch.randn(*s, generator=gen).to(torch.bfloat16).cuda()
                 for s in ((N, H // 2, W // 2, c1), (N, H, W, c2), (N, H, W, cout)))
    x = torch.cat([xh.repeat_interleave(2, 1).repeat_interleave(2, 2), sk], -1).contiguous()
    conv = sg.Conv(c1 + c2, cout, 9, np.random.default_rng(0), "cuda:0")
    scratch = sg.Scratch("cuda:0")
    got = []
    for inp in (x, (xh, sk)):
        conv.dw.fill_(float("nan"))
        conv.db.fill_(float("nan"))
        conv.backward(inp, g, (N, H, W), scratch, need_dx=False)
        got.append((conv.dw.clone(), conv.db.clone()))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("N,H,W,c,cu,off", [(1, 2, 2, 8, 8, 0), (2, 6, 10, 32, 96, 64),
                                            (3, 14, 6, 64, 160, 96)])
def test_fused_skip_gradients(shy, N, H, W, c, cu, off):
    """The passes between two stages of the backward in one kernel each: the
    separate passes' bits."""
    from simplehydrology_amd import surrogate as sg
    print("skip", N, H, W, c, cu, off, flush=True)
    L, s = sg.nn(), torch.cuda.current_stream().cuda_stream
    gen = torch.Generator().manual_seed(c)
    gp, gu, y = (torch.randn(*d, generator=gen).to(torch.bfloat16).cuda()
                 for d in ((N, H // 2, W // 2, c), (N, H, W, cu), (N, H, W, c)))
    spread, share, out = (torch.empty_like(y) for _ in range(3))
    assert L.shy_nn_pool2(gp.data_ptr(), spread.data_ptr(), N, H, W, c, 1, s) == 0
    assert L.shy_nn_channels(gu.data_ptr(), share.data_ptr(), N * H * W, c, cu, off, 1, s) == 0
    assert L.shy_nn_skip_bwd(gp.data_ptr(), gu.data_ptr(), y.data_ptr(), out.data_ptr(), N, H, W, c,
                             cu, off, s) == 0
    assert torch.equal(out, sg._relu_bwd(y, sg._add(spread, share)))
    down, gated = torch.empty_like(gp), torch.empty_like(gp)
    yh = torch.randn(N, H // 2, W // 2, c, generator=gen).to(torch.bfloat16).cuda()
    assert L.shy_nn_up2(gu.data_ptr(), down.data_ptr(), N, H // 2, W // 2, c, cu, off, 1, s) == 0
    assert L.shy_nn_up2_bwd_relu(gu.data_ptr(), yh.data_ptr(), gated.data_ptr(), N, H // 2, W // 2,
                                 c, cu, off, s) == 0
    assert torch.equal(gated, sg._relu_bwd(yh, down))
