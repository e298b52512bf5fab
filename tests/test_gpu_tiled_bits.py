"""GPU: the fused features, windows and decoding of the tiled inference give the
element-wise functions' bits: for 2^24 floats spread over all of them (zeros,
infinities and NaN among them), and for windows of a map."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

N = 4096


@pytest.fixture(scope="module")
def sg(shy):
    from simplehydrology_amd import surrogate
    return surrogate


def floats():
    """Every 257th pattern (257 is odd, so signs, exponents and fractions mix),
    and the special values."""
    v = (torch.arange(N * N, dtype=torch.int64, device="cuda") * 257) % 2 ** 32
    v = torch.where(v >= 2 ** 31, v - 2 ** 32, v).to(torch.int32).view(torch.float32).clone()
    v[:8] = torch.tensor([0.0, -0.0, float("inf"), -float("inf"), float("nan"), -1.0, 2.0 ** -149,
                          -2.0 ** -126])
    return v.reshape(N, N)


def same(a, b):
    a, b = a.contiguous(), b.contiguous()
    return bool(((a.view(torch.int32) == b.view(torch.int32)) | (a.isnan() & b.isnan())).all())


def test_encoding(sg):
    v = floats()
    h = torch.zeros_like(v)
    f = torch.empty(N, N, 8, device="cuda")
    print("encoding", flush=True)
    strides = (C.c_longlong * 8)(*([N, 1] * 4))
    assert sg.nn().shy_nn_flow_features(h.data_ptr(), v.data_ptr(), v.data_ptr(), v.data_ptr(),
                                        strides, f.data_ptr(), N, N, sg.SLOPE_SCALE,
                                        1.0 / sg.D_SCALE, sg._stream()) == 0
    assert same(f[..., 3:6], sg.encode_flow(v, v, v))


def test_decoding(sg):
    y = floats()[..., None].expand(N, N, 8).contiguous()
    out = [torch.empty(N, N, device="cuda") for _ in range(3)]
    print("decoding", flush=True)
    assert sg.nn().shy_nn_window_output(y.data_ptr(), (C.c_int * 6)(0, 0, N, 0, 0, N), 1,
                                        *(o.data_ptr() for o in out), N, N, N, sg.D_SCALE,
                                        sg._stream()) == 0
    for a, b in zip(out, sg.decode_flow(y)):
        assert same(a, b)


def test_features_and_windows(sg):
    gen = torch.Generator().manual_seed(1)
    a = torch.randn(50, 61, 4, generator=gen).cuda()
    h, d, mx, my = (a[..., k] for k in range(4))
    want = sg.features(h, d, mx, my)
    f = torch.empty_like(want)
    strides = (C.c_longlong * 8)(*(s for t in (h, d, mx, my) for s in t.stride()))
    print("features", flush=True)
    L, s, tile = sg.nn(), sg._stream(), 24
    assert L.shy_nn_flow_features(h.data_ptr(), d.data_ptr(), mx.data_ptr(), my.data_ptr(), strides,
                                  f.data_ptr(), 50, 61, sg.SLOPE_SCALE, 1.0 / sg.D_SCALE, s) == 0
    assert same(f, want)
    at = [(0, 0), (26, 37), (3, 11)]
    xs = torch.empty(3, tile, tile, 8, device="cuda")
    x = torch.empty(3, tile, tile, 8, dtype=torch.bfloat16, device="cuda")
    jobs = (C.c_int * 18)(*(v for i, j in at for v in (i, i, tile, j, j, tile)))
    assert L.shy_nn_window_copy(f.data_ptr(), jobs, 3, xs.data_ptr(), 50, 61, tile, s) == 0
    mean = xs[..., 0].mean(dim=(1, 2))
    assert L.shy_nn_window_input(xs.data_ptr(), mean.data_ptr(), x.data_ptr(), 3, tile, sg.H_SCALE,
                                 s) == 0
    assert torch.equal(x.view(torch.int16), sg.window_batch(want, at, tile).view(torch.int16))
