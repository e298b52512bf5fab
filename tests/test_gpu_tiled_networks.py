"""GPU: tiled inference with a network of the program's own, whose output is not
the library network's [n, tile, tile, 8] in float32, against the element-wise
route (float64 maps take it)."""
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


class Own:
    """A network whose output has other channels, another type or strides."""

    def __init__(self, form):
        self.form = form

    def forward(self, x, keep=True):
        y = x.float() * 0.5
        return {"three": y[..., :3].contiguous(), "sixteen": torch.cat([y, y], -1),
                "half": y.to(torch.bfloat16), "strided": torch.cat([y, y], -1)[..., :8],
                "planar": y.permute(0, 3, 1, 2).contiguous().permute(0, 2, 3, 1),
                "library": y}[self.form]


@pytest.mark.parametrize("form", ["three", "sixteen", "half", "strided", "planar", "library"])
def test_output_forms(shy, form):
    from simplehydrology_amd import surrogate as sg
    print("tiled", form, flush=True)
    gen = torch.Generator().manual_seed(2)
    a = torch.randn(60, 70, 4, generator=gen).cuda()
    h, d, mx, my = (a[..., k] for k in range(4))
    net = Own(form)
    kw = dict(tile=32, halo=4, batch=5)
    got = sg.predict_tiled(net, h, d, mx, my, **kw)
    want = sg.predict_tiled(net, h.double(), d, mx, my, **kw)
    for u, v in zip(got, want):
        # log1p and expm1 of two libraries, at most 2 ulp each, and a BF16 input
        # that rounds the other way by an ulp of its own (2^-8)
        assert float((u - v).norm()) <= 2 ** -8 * float(v.norm())
        assert torch.isfinite(u).all()
