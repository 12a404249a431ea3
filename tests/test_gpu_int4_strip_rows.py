"""GPU parity: the general form of the strip-linear int4 decode kernel (k3q_gemv_w4s_rows: float32 or
bfloat16 rows, any K % 8, any N) against the float64 value of the same stored operands."""

import pytest
import torch

from keras_amd import ops as kops, quantizers
from tests.helpers import c_w4_matmul_f64
from tests.test_gpu_int4_matmul import make_layer

pytestmark = pytest.mark.gpu


def magnitude(x, packed, scale, zero, block_size, N):
    """sum_k |x| (|w - zero| + 48) scale: what a rounding error of the sums is relative to (the kernel adds
    24 to every weight and takes it out again)."""
    w = quantizers.unpack_int4(packed, N, axis=-1).cpu().double()
    K = w.shape[0]
    if block_size:
        g = torch.arange(K) // block_size
        w = ((w - zero.double()[g]).abs() + 48) * scale.double()[g].abs()
    else:
        w = (w.abs() + 48) / scale.double().abs()
    return x.double().abs() @ w


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,K,N,block_size", [
    (1, 16, 1, None), (3, 24, 17, 128), (16, 136, 5, None), (5, 128, 16, 128), (6, 1600, 6400, 128),
    (8, 4096, 4096, 128), (9, 2048, 5247, 128), (16, 2048, 5247, None), (2, 960, 1003, 128), (16, 768, 768, 128),
    (7, 4544, 2100, None), (8, 8192, 8208, 128), (16, 4096, 14336, 128), (11, 8192, 4096, None),
    (2, 14336, 1024, 128), (3, 1000, 20001, 128), (4, 2056, 9000, None),
])
def test_rows_shapes(dev, dtype, M, K, N, block_size):
    qk, bias = make_layer(K, N, block_size, seed=M + K, with_bias=(M % 2 == 1))
    g = torch.Generator().manual_seed(K)
    x = torch.randn(M, K, generator=g).to(dtype)
    scale, kernel = qk["kernel_scale"].to(dtype), qk["kernel"].to(dev)
    zero = qk["kernel_zero"] if block_size else None
    assert kops.int4_strip_rows_launches(dtype, M, K, N, block_size) > 0
    per_row = M == 9  # a bias row per row of x
    b = None if bias is None else bias.to(dtype)
    if per_row:
        b = torch.randn(M, N, generator=g).to(dtype)
    got = kops.int4_matmul_strip_rows(
        x.to(dev), kops.int4_strip_copy(kernel, N), N, kernel_scale=None if block_size else scale.to(dev),
        gparams=kops.int4_strip_rows_params(scale.to(dev), zero.to(dev), K, N, block_size) if block_size else None,
        block_size=block_size, bias=None if b is None else b.to(dev))
    torch.cuda.synchronize()
    assert got.dtype == dtype and tuple(got.shape) == (M, N)
    exact = c_w4_matmul_f64(x, qk["kernel"], scale, zero, block_size, None if per_row else b, N)
    if per_row:
        exact = exact + b.double()
    mag = magnitude(x, kernel, scale, zero, block_size, N)
    err = (got.double().cpu() - exact).abs()
    if dtype == torch.float32:
        # two parts leave 2^-17 of a value, three nothing; float32 sums of K terms: 2^-24 sqrt(K) of the magnitudes,
        # four times that (plus the result's own roundings)
        split = 2.0 ** -17 if N % 8 == 0 and K % 16 == 0 else 0.0
        bound = mag * (split + 4 * 2.0 ** -24 * K ** 0.5) + exact.abs() * 2.0 ** -22
    else:  # sum, quotient and biased result are each rounded to bfloat16: half an ulp is up to 2^-8 of the value
        size = exact.abs() + (0 if b is None else 2 * b.double().abs())
        bound = mag * 4 * 2.0 ** -24 * K ** 0.5 + size * 3.05 * 2.0 ** -8
    assert bool((err <= bound).all()), float((err / bound).max())


def test_rows_layer_routes(dev):
    """Layers whose shapes only this form takes agree with the kernel on the stored weights."""
    from keras_amd.layers import Dense, EinsumDense

    g = torch.Generator().manual_seed(3)
    for policy, dt in (("float32", torch.float32), ("mixed_bfloat16", torch.bfloat16)):
        layer = Dense(1003, dtype=policy, device="cuda:0")
        layer.build((None, 1600))
        layer.quantize("int4")
        x = torch.randn(2, 3, 1600, generator=g).to(dt).to(dev)
        y = layer(x)
        assert "w4s" in layer._cache and tuple(y.shape) == (2, 3, 1003)
        other = kops.int4_matmul(x, layer._kernel.value, layer.kernel_scale.value.to(dt), 1003,
                                 kernel_zero=layer.kernel_zero.value, block_size=128,
                                 bias=layer.bias.value.to(dt))
        tol = 1e-5 if dt == torch.float32 else 1e-2
        assert float((y - other).abs().max()) <= tol * float(other.abs().max())
        # assigned weights reach the copies, in place
        shadow = layer._cache["w4s"][2].data_ptr()
        layer._kernel.assign(torch.zeros_like(layer._kernel.value))
        layer.kernel_zero.assign(torch.zeros_like(layer.kernel_zero.value))
        # (the offset of 24 is taken out of float32 sums: 2^-24 sqrt(K) of 24 sum |x| scale, below 1e-4 here)
        assert float((layer(x).float() - layer.bias.value.to(dt).float()).abs().max()) < 1e-4
        assert layer._cache["w4s"][2].data_ptr() == shadow
        ein = EinsumDense("btd,dnh->btnh", (None, 4, 64), dtype=policy, device="cuda:0")
        ein.build((None, None, 192))
        ein.quantize("int4")
        assert tuple(ein(torch.randn(2, 2, 192, generator=g).to(dt).to(dev)).shape) == (2, 2, 4, 64)
        assert "w4s" in ein._cache


@pytest.mark.parametrize("dtype,M,K,widths,block_size", [
    (torch.float32, 4, 256, (1003, 1001, 777), 128),          # three parts, weights without an offset
    (torch.float32, 8, 1024, (96, 64, 48), 128),              # two parts
    (torch.float32, 3, 512, (3200, 3200, 40), None),          # more strip groups than workgroups
    (torch.float32, 8, 4096, (8192, 8208), 128),              # ... and room for one reduction buffer
    (torch.bfloat16, 16, 1000, (1003, 9, 5247), 128),
    (torch.bfloat16, 5, 1600, (6400, 6400, 1600, 1600, 1600), None),  # more kernels than a launch takes
    (torch.float32, 2, 384, (1003, 96, 9000, 1000), 128),     # plans that differ
    (torch.bfloat16, 2, 384, (1003, 96, 9000, 1000), 128),
    (torch.float32, 16, 256, (96, 104), 128),                 # more rows than a launch takes
])
def test_shared_launch_has_the_bits_of_the_separate_calls(dev, dtype, M, K, widths, block_size):
    g = torch.Generator(device=dev).manual_seed(K + M)
    rand = lambda *s: torch.rand(*s, generator=g, device=dev)
    kernels = []
    for i, N in enumerate(widths):
        packed = torch.randint(-128, 128, (K, (N + 1) // 2), generator=g, device=dev, dtype=torch.int8)
        kernel = dict(units=N, shadow=kops.int4_strip_copy(packed, N),
                      bias=rand(N).to(dtype) if i % 2 else None)
        if block_size:
            groups = -(-K // block_size)
            zero = torch.randint(-8, 8, (groups, N), generator=g, device=dev, dtype=torch.int8)
            kernel["gparams"] = kops.int4_strip_rows_params((rand(groups, N) + 1).to(dtype), zero, K, N, block_size)
        else:
            kernel["kernel_scale"] = (rand(N) + 1).to(dtype)
        kernels.append(kernel)
    x = torch.randn(M, K, generator=g, device=dev).to(dtype)
    together = kops.int4_matmul_strip_rows_multi(x, kernels, block_size=block_size)
    for y, kernel in zip(together, kernels):
        assert torch.equal(y, kops.int4_matmul_strip_rows(x, block_size=block_size, **kernel))
