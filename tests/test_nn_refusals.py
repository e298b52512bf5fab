"""CPU: what the network's one-call inference refuses, it refuses before its
first launch (no GPU is needed to see it)."""
import ctypes as C

import pytest

CH = (32, 64, 96, 128)


@pytest.fixture(scope="module")
def nn():
    from simplehydrology_amd import surrogate
    return surrogate.nn()


def table(v):
    return (C.c_int * 4)(*v)


def forward(nn, ch=CH, cin=8, head_c=8, n=1, h=16, w=24, work=None):
    """The call with memory that is never read: every refusal comes first."""
    p = C.c_void_p(4096)
    t = (C.c_void_p * 22)(*([4096] * 22))
    if work is None:
        work = nn.shy_nn_unet_work_bytes(table(CH), 1, 16, 24)
    return nn.shy_nn_unet_forward(p, t, t, table(ch), cin, head_c, p, work, p, n, h, w, None)


@pytest.mark.parametrize("ch", [(64, 64, 96, 128), (96, 64, 96, 128), (0, 64, 96, 128),
                                (32, 48, 96, 128), (32, 64, 16, 128), (32, 64, 96, -32)])
def test_channels(nn, ch):
    """The last convolution and the head read 32 channels; the others come in
    multiples of 32."""
    assert nn.shy_nn_unet_work_bytes(table(ch), 1, 16, 24) == -1
    assert forward(nn, ch=ch, work=1 << 40) != 0
    assert b"ch[0] = 32" in nn.shy_nn_last_error()


@pytest.mark.parametrize("kw", [dict(cin=12), dict(cin=0), dict(head_c=6), dict(head_c=20)])
def test_first_and_last_layer(nn, kw):
    assert forward(nn, **kw) != 0
    assert b"cin a multiple of 8" in nn.shy_nn_last_error()


@pytest.mark.parametrize("h,w", [(12, 24), (16, 20), (0, 24), (16, 4)])
def test_sides(nn, h, w):
    assert nn.shy_nn_unet_work_bytes(table(CH), 1, h, w) == -1
    assert forward(nn, h=h, w=w, work=1 << 40) != 0
    assert b"multiples of 8" in nn.shy_nn_last_error()


def test_work_memory(nn):
    need = nn.shy_nn_unet_work_bytes(table(CH), 1, 16, 24)
    assert need > 0
    assert forward(nn, work=need - 1) != 0
    assert b"work memory too small" in nn.shy_nn_last_error()
