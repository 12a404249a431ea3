"""GPU parity: the int8 tile kernel on the strip-linear copy for K an odd multiple of 64 (the last stage has one half),
every tile shape and a split of K, against exact integers and the zero-padded route, bit for bit."""

import pytest
import torch

from keras_amd import ops as kops
from tests.helpers import c_gemm_i8

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,K,N", [
    (17, 64, 48), (9, 192, 1003), (130, 960, 260), (64, 1600, 6400), (1000, 1600, 640), (33, 14400, 256),
    (1024, 2624, 4096),   # the ring of four stages
    (3600, 192, 4096), (3700, 320, 4100),  # the 256 x 256 tile
])
def test_half_tail(dev, M, K, N):
    g = torch.Generator().manual_seed(K + M)
    a = torch.randint(-128, 128, (M, K), generator=g, dtype=torch.int8)
    w = torch.randint(-128, 128, (K, N), generator=g, dtype=torch.int8)
    ad, wd = a.to(dev), w.to(dev)
    strip, pre = kops.int8_strip_copy(wd), kops.prepack_int8_kernel(wd)
    for dtype in (torch.float32, torch.bfloat16):
        sa = (torch.rand(M, generator=g) + 0.5).to(dtype).to(dev)
        sb = (torch.rand(N, generator=g) + 0.5).to(dtype).to(dev)
        bias = torch.randn(N, generator=g).to(dtype).to(dev)
        args = dict(a_scale=sa, kernel_scale=sb, bias=bias, out_dtype=dtype, exact_epilogue=True)
        y = kops.int8_matmul(ad, wd, strip=strip, **args)
        assert torch.equal(y, kops.int8_matmul(ad, wd, prepacked=pre, **args))
    acc = kops.int8_matmul(ad, wd, strip=strip, want_acc=True, want_y=False)
    acc = acc[1] if isinstance(acc, tuple) else acc
    assert torch.equal(acc.cpu(), c_gemm_i8(a, w))


def test_half_tail_layer_with_unaligned_bias(dev):
    """Scales and bias that do not start on 16 bytes (views) are taken as before."""
    from keras_amd.layers import Dense

    g = torch.Generator().manual_seed(0)
    layer = Dense(256, device="cuda:0")
    layer.build((None, 192))
    layer.quantize("int8")
    x = torch.randn(40, 192, generator=g).to(dev)
    b = torch.randn(257, generator=g).to(dev)
    layer.bias.assign(b[1:])
    y = layer(x)
    layer.bias.assign(b[1:].clone())
    assert torch.equal(y, layer(x))


@pytest.mark.parametrize("K", [192, 256])
def test_rows_that_do_not_start_on_16_bytes(dev, K):
    """Quantised rows that are a view into a larger buffer, with the strip-linear copy at hand."""
    g = torch.Generator().manual_seed(K)
    w = torch.randint(-128, 128, (K, 96), generator=g, dtype=torch.int8).to(dev)
    flat = torch.randint(-128, 128, (40 * K + 3,), generator=g, dtype=torch.int8).to(dev)
    a = flat[3:].view(40, K)
    acc = kops.int8_matmul(a, w, strip=kops.int8_strip_copy(w), want_acc=True, want_y=False)
    assert torch.equal(acc.cpu(), c_gemm_i8(a.cpu(), w.cpu()))
