"""GPU parity: the int8 forward as one call of the C ABI (k3q_dense_i8) -- float32 rows quantised inside the product's
workgroups, other rows ahead of it -- against quantizer and product called one by one, bit for bit."""

import pytest
import torch

from keras_amd import _lib, ops as kops, quantizers
from keras_amd.layers import Dense, EinsumDense
from keras_amd.layers.together import shared_input_rows

pytestmark = pytest.mark.gpu


def operands(M, K, N, dtype, dev, bias):
    g = torch.Generator().manual_seed(M * 31 + K + N)
    x = torch.randn(M, K, generator=g)
    x[0] *= 1e-30 if M % 2 else 3e4
    if M > 1:
        x[-1] = 0
    if M > 2:
        x[1, K // 2], x[1, 3] = float("inf"), float("nan")
    w = torch.randint(-127, 128, (K, N), generator=g, dtype=torch.int8)
    ks = (torch.rand(N, generator=g) * 900 + 100).to(dtype)
    b = None if not bias else torch.randn((M, N) if bias == "rows" else (N,), generator=g).to(dtype)
    return x.to(dtype).to(dev), w.to(dev), ks.to(dev), None if b is None else b.to(dev)


def same(a, b):
    return torch.equal(a.view(torch.int16 if a.dtype == torch.bfloat16 else torch.int32),
                       b.view(torch.int16 if b.dtype == torch.bfloat16 else torch.int32))


# (M K up to 16384 values, 3072 columns and more: quantised inside; one, four and eight pieces a thread; strips one
# or two a wave, a ring of two or four units; just past the limit: a launch ahead)
@pytest.mark.parametrize("M,K,N,bias", [
    (1, 1024, 3072, "one"), (2, 1024, 8192, None), (8, 1024, 3088, "rows"), (16, 1024, 8208, "one"), (1, 4096, 4096, "one"),
    (3, 4096, 8192, "rows"), (4, 4096, 3072, None), (1, 16384, 3072, "one"), (5, 3072, 4112, "one"),
    (5, 4096, 4096, "one"), (16, 1600, 6400, "rows"), (3, 64, 5, "one"),
])
@pytest.mark.parametrize("value_range", [(-127, 127), (-128, 100), (-100.5, 90.25)])
def test_decode_rows(dev, M, K, N, bias, value_range):
    x, w, ks, b = operands(M, K, N, torch.float32, dev, bias)
    strip = kops.int8_strip_copy(w)
    kops._workspace(dev, 4 << 20).fill_(0xFF)
    got = kops.int8_dense_strip(x, strip, N, ks, bias=b, value_range=value_range)
    want = kops.int8_dense_strip(x, strip, N, ks, bias=b, value_range=value_range, quantize=lambda rows:
                                 quantizers.abs_max_quantize(rows, axis=-1, value_range=value_range))
    assert same(got, want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,K,N,bias", [(17, 64, 1, "one"), (33, 192, 130, None), (100, 1600, 6400, "one"),
                                        (129, 960, 1003, "one"), (300, 4096, 512, None), (1000, 256, 2048, "one")])
def test_more_rows(dev, M, K, N, bias, dtype):
    x, w, ks, b = operands(M, K, N, dtype, dev, bias)
    strip = kops.int8_strip_copy(w)
    kops._workspace(dev, 64 << 20).fill_(0xFF)
    q, s = quantizers.abs_max_quantize(x, axis=-1)
    want = kops.int8_matmul(q, w, a_scale=s, kernel_scale=ks, bias=b, out_dtype=dtype, exact_epilogue=True, strip=strip)
    assert same(kops.int8_dense_rows(x, strip, N, ks, bias=b), want)
    # operands that start anywhere, rows that lie apart
    off = lambda t: None if t is None else torch.cat((t[:1], t))[1:]
    apart = torch.cat((x, x), dim=1)[:, :K]
    assert same(kops.int8_dense_rows(apart, strip, N, off(ks), bias=off(b)), want)


def test_what_is_refused(dev):
    x, w, ks, _ = operands(20, 128, 64, torch.float32, dev, None)
    strip, lib, y = kops.int8_strip_copy(w), _lib.load(), torch.empty(20, 64, device=dev)
    ws = torch.empty(1 << 16, dtype=torch.uint8, device=dev)

    def call(dtype=_lib.K3Q_F32, M=20, K=128, stride=0, lo=-127.0, hi=127.0, ws_bytes=1 << 16):
        return lib.k3q_dense_i8(_lib.ptr(x), dtype, M, K, 64, _lib.ptr(strip), _lib.ptr(ks), None, stride, 1e-7, lo, hi,
                                _lib.ptr(y), _lib.ptr(ws), ws_bytes, _lib.stream_ptr(dev))

    assert call() == 0 and call(M=0) == 0
    assert 0 not in (call(dtype=7), call(K=96), call(stride=64), call(lo=-129.0), call(hi=128.0), call(lo=5.0, hi=4.0),
                     call(ws_bytes=64), call(M=-1))
    with pytest.raises(ValueError):
        kops.int8_dense_rows(x, strip, 64, ks[:-1])
    with pytest.raises(TypeError):
        kops.int8_dense_rows(x, strip, 64, ks.to(torch.bfloat16))
    with pytest.raises(ValueError):
        kops.int8_dense_rows(x, strip[:-16], 64, ks)


@pytest.mark.parametrize("policy", ["float32", "mixed_bfloat16"])
@pytest.mark.parametrize("rows", [1, 4, 16, 17, 200])
def test_layers_share_rows_or_not(dev, policy, rows):
    """Inside `shared_input_rows` the rows are quantised once and handed on; outside, in the layer's own call: the same bits."""
    layers = [Dense(3072, dtype=policy, device="cuda:0"), EinsumDense("bd,dnh->bnh", (24, 128), dtype=policy, device="cuda:0")]
    for layer in layers:
        layer.build((None, 1024))
        layer.quantize("int8")
    x = torch.randn(rows, 1024, generator=torch.Generator().manual_seed(rows)).to(dev)
    alone = [layer(x) for layer in layers]
    with shared_input_rows():
        shared = [layer(x) for layer in layers]
    assert all(same(a, b) for a, b in zip(alone, shared))
