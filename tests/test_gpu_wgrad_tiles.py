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
