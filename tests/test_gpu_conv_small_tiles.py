"""GPU: the 16 x 8 tiles of the 3x3 convolutions (layers whose 16 x 8 tiles all run
at once: 768 blocks of 32 output channels on 256 CUs; maps of up to 8 rows) at
their edges, with each epilogue, against float64, and the layers on both sides of
the lines: the last of 16 x 8 tiles and the first of 16 x 16 ones, and wide layers
of one tile per block.

Tolerances as in test_gpu_conv_tiles; a head output is an FP32 sum of 32 products
of the rounded values (1e-6 is beyond 10 times its rounding), a pooled value is
stated to the bit."""
import pytest

import test_gpu_conv_tiles as tiles

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

SIZES = [(1, 1, 1), (1, 7, 15), (2, 8, 16), (1, 9, 17), (3, 17, 33), (1, 24, 64), (5, 47, 65)]


@pytest.mark.parametrize("N,H,W", SIZES)
@pytest.mark.parametrize("cin,cout", [(32, 32), (64, 96)])
def test_forward_epilogues(shy, N, H, W, cin, cout):
    tiles.test_forward_epilogues(shy, N, H, W, cin, cout)


@pytest.mark.parametrize("N,H,W,cin,cout", [
    (384, 16, 16, 32, 32), (385, 16, 16, 32, 32),  # 768 and 770 tiles of 16 x 8
    (128, 16, 16, 64, 96), (129, 16, 16, 64, 96),  # 256 and 258, three channel blocks each
    (770, 8, 15, 32, 32),                          # more than run at once, of 8 rows
    (97, 15, 16, 160, 256),                        # 97 tiles of 16 x 16 on 96 blocks: one each
])
def test_lines_between_the_variants(shy, N, H, W, cin, cout):
    tiles.test_forward_epilogues(shy, N, H, W, cin, cout)


@pytest.mark.parametrize("N,H,W,c1,c2,cout", [(1, 2, 2, 32, 32, 32), (1, 8, 16, 64, 32, 32),
                                              (2, 10, 18, 32, 64, 64), (3, 26, 34, 64, 32, 96),
                                              (1, 6, 250, 96, 64, 32)])
def test_upsampled_input(shy, N, H, W, c1, c2, cout):
    tiles.test_upsampled_input(shy, N, H, W, c1, c2, cout)


def operands(N, H, W, cin, cout):
    x, w = tiles.rand(N, H, W, cin, seed=1), tiles.rand(cout, 9 * cin, seed=2)
    res = tiles.rand(N, H, W, cout, seed=3)
    b = torch.randn(cout, generator=torch.Generator().manual_seed(4))
    ref = (tiles.conv64(x.double(), w.double()) + b.double() + res.double()).relu()
    return [t.cuda().contiguous() for t in (x, w, res, b)], ref


@pytest.mark.parametrize("N,H,W", [(1, 1, 1), (1, 7, 15), (1, 9, 17), (5, 47, 65), (260, 15, 16)])
@pytest.mark.parametrize("cin,hc", [(32, 8), (64, 16)])
def test_head(shy, N, H, W, cin, hc):
    from simplehydrology_amd import surrogate as sg
    print("head", N, H, W, cin, hc, flush=True)
    (x, w, res, b), ref = operands(N, H, W, cin, 32)
    hw = tiles.rand(hc, 32, seed=5).cuda()
    hb = torch.randn(hc, generator=torch.Generator().manual_seed(6)).cuda()
    y = torch.empty(N, H, W, 32, dtype=torch.bfloat16, device="cuda")
    out = torch.full((N, H, W, hc), float("nan"), device="cuda")
    assert sg.nn().shy_nn_conv_fwd_head(x.data_ptr(), w.data_ptr(), b.data_ptr(), res.data_ptr(),
                                        y.data_ptr(), hw.data_ptr(), hb.data_ptr(), out.data_ptr(),
                                        N, H, W, cin, hc, 1, sg._stream()) == 0
    tiles.close(y, ref, 2 ** -8)
    tiles.close(out, (y.double() @ hw.double().t() + hb.double()).cpu(), 1e-6)


@pytest.mark.parametrize("N,H,W", [(1, 2, 2), (1, 8, 16), (1, 10, 18), (5, 46, 66), (260, 14, 16)])
@pytest.mark.parametrize("cin,cout", [(32, 32), (64, 96)])
def test_pool(shy, N, H, W, cin, cout):
    from simplehydrology_amd import surrogate as sg
    print("pool", N, H, W, cin, cout, flush=True)
    (x, w, res, b), ref = operands(N, H, W, cin, cout)
    y = torch.empty(N, H, W, cout, dtype=torch.bfloat16, device="cuda")
    p = torch.full((N, H // 2, W // 2, cout), float("nan"), dtype=torch.bfloat16, device="cuda")
    assert sg.nn().shy_nn_conv_fwd_pool(x.data_ptr(), w.data_ptr(), b.data_ptr(), res.data_ptr(),
                                        y.data_ptr(), p.data_ptr(), N, H, W, cin, cout, 1,
                                        sg._stream()) == 0
    tiles.close(y, ref, 2 ** -8)
    q = y.float().view(N, H // 2, 2, W // 2, 2, cout)
    want = 0.25 * (q[:, :, 0, :, 0] + q[:, :, 0, :, 1] + q[:, :, 1, :, 0] + q[:, :, 1, :, 1])
    assert torch.equal(p, want.to(torch.bfloat16))
