"""GPU parity: the int4 tile kernel for any K % 8, any N, float32 or bfloat16 rows (k3q_gemm_w4_rows) against
the float64 value of the same stored operands."""

import pytest
import torch

from keras_amd import ops as kops
from keras_amd.layers import Dense, EinsumDense
from keras_amd.layers.dense import TILE_ROWS_MAX_F32
from tests.helpers import c_w4_matmul_f64
from tests.test_gpu_int4_matmul import make_layer
from tests.test_gpu_int4_strip_rows import magnitude

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,K,N,block_size", [
    (1, 16, 1, None), (17, 24, 33, 128), (31, 136, 5, 128), (32, 1600, 6400, 128), (33, 960, 1003, 128),
    (64, 128, 128, None), (65, 2048, 5247, 128), (128, 768, 2094, None), (129, 4544, 3200, 128), (300, 1600, 6400, 128),
    (342, 1000, 777, 128), (513, 320, 1028, 128), (1025, 192, 100, None), (2050, 448, 260, 128), (64, 4096, 14336, 128),
])
def test_tiles_rows(dev, dtype, M, K, N, block_size):
    qk, bias = make_layer(K, N, block_size, seed=M + K, with_bias=(M % 2 == 1))
    g = torch.Generator().manual_seed(K)
    x = torch.randn(M, K, generator=g).to(dtype)
    scale, kernel = qk["kernel_scale"].to(dtype), qk["kernel"].to(dev)
    zero = qk["kernel_zero"] if block_size else None
    b = None if bias is None else bias.to(dtype)
    per_row = M == 33
    if per_row:
        b = torch.randn(M, N, generator=g).to(dtype)
    # poisoned scratch: a partial or a row that is read before it is written shows
    kops._workspace(dev, 64 << 20).fill_(0xFF)
    got = kops.int4_matmul_tiles_rows(
        x.to(dev), kops.int4_strip_copy(kernel, N), N,
        kops.int4_tile_columns(scale.to(dev), N) if block_size else scale.to(dev),
        kernel_zero=kops.int4_tile_columns(zero.to(dev), N) if block_size else None,
        block_size=block_size, bias=None if b is None else b.to(dev))
    torch.cuda.synchronize()
    assert got.dtype == dtype and tuple(got.shape) == (M, N)
    exact = c_w4_matmul_f64(x, qk["kernel"], scale, zero, block_size, None if per_row else b, N)
    if per_row:
        exact = exact + b.double()
    mag = magnitude(x, kernel, scale, zero, block_size, N)
    err = (got.double().cpu() - exact).abs()
    if dtype == torch.float32:  # (as in test_rows_shapes)
        split = 2.0 ** -17 if N % 8 == 0 and K % 16 == 0 else 0.0
        bound = mag * (split + 4 * 2.0 ** -24 * K ** 0.5) + exact.abs() * 2.0 ** -22
    else:  # sum, quotient and biased result are each rounded to bfloat16: half an ulp is up to 2^-8 of the value
        size = exact.abs() + (0 if b is None else 2 * b.double().abs())
        bound = mag * 4 * 2.0 ** -24 * K ** 0.5 + size * 3.05 * 2.0 ** -8
    assert bool((err <= bound).all()), float((err / bound).max())


def test_layer_with_parameters_that_start_anywhere(dev):
    """Scales and zero points assigned from views into larger buffers, which the kernels on the stored weights take."""
    layer = Dense(96, device="cuda:0")
    layer.build((None, 256))
    layer.quantize("int4")
    x = torch.randn(40, 256, generator=torch.Generator().manual_seed(0)).to(dev)
    want = layer(x)
    for var in (layer.kernel_scale, layer.kernel_zero):
        buffer = torch.empty(var.value.numel() + 1, dtype=var.value.dtype, device=dev)
        buffer[1:] = var.value.flatten()
        var.assign(buffer[1:].view(var.shape))
    assert torch.equal(layer(x), want)


def check_layer(layer, x, units):
    """A layer's output against the float64 value of its variables, with the bounds above.  Without a strip-linear copy the
    call went to the de-quantised kernel: its weights are two bfloat16 parts (2^-16 of each is lost) for float32 rows,
    one for bfloat16 rows (2^-8)."""
    scale, zero = layer.kernel_scale.value, layer.kernel_zero.value
    y = layer(x).reshape(-1, units)
    x2 = x.reshape(y.shape[0], -1).cpu()
    args = (layer._kernel.value, scale.to(x.dtype), zero, 128, units)
    exact = c_w4_matmul_f64(x2, args[0].cpu(), args[1].cpu(), zero.cpu(), 128, None, units)
    mag = magnitude(x2, args[0], args[1].cpu(), zero.cpu(), 128, units)
    err, K = (y.double().cpu() - exact).abs(), x2.shape[1]
    if x.dtype == torch.float32:
        bound = mag * (2.0 ** -16 + 4 * 2.0 ** -24 * K ** 0.5) + exact.abs() * 2.0 ** -22
    else:
        weights = 0.0 if "w4s" in layer._cache else 2.0 ** -8
        bound = mag * (weights + 4 * 2.0 ** -24 * K ** 0.5) + exact.abs() * 1.02 * 2.0 ** -8
    assert bool((err <= bound).all()), float((err / bound).max())


@pytest.mark.parametrize("policy", ["float32", "mixed_bfloat16"])
@pytest.mark.parametrize("kind,K,units,rows,copy", [
    ("dense", 1000, 1003, 40, True), ("dense", 320, 1028, 600, True), ("dense", 192, 101, 1000, True),
    ("dense", 256, 128, TILE_ROWS_MAX_F32, None), ("dense", 256, 128, TILE_ROWS_MAX_F32 + 1, False),
    ("einsum", 192, 105, 40, True), ("einsum", 136, 105, 900, True), ("einsum", 256, 192, 300, None),
])
def test_layer_routes(dev, policy, kind, K, units, rows, copy):
    """Ragged layers and float32 rows on both sides of the line to the de-quantised kernel; copy: whether the call reads the
    strip-linear copy (None: float32 rows do)."""
    dtype = torch.float32 if policy == "float32" else torch.bfloat16
    if kind == "dense":
        layer = Dense(units, dtype=policy, device="cuda:0", use_bias=False)
        layer.build((None, K))
    else:
        layer = EinsumDense("btd,dnh->btnh", (None, 3, units // 3), dtype=policy, device="cuda:0")
        layer.build((None, None, K))
    layer.quantize("int4")
    x = torch.randn(2, rows // 2, K, generator=torch.Generator().manual_seed(rows)).to(dtype).to(dev)
    x = x if rows % 2 == 0 else torch.cat((x.flatten(0, 1), x[0, :1])).unsqueeze(0)
    check_layer(layer, x, units)
    expected = copy if copy is not None else dtype == torch.float32 or rows <= 512
    assert ("w4s" in layer._cache) == expected
    # (scales and zero points padded to whole strips are rebuilt with the variables)
    layer.kernel_scale.assign(layer.kernel_scale.value * 2)
    layer.kernel_zero.assign(-layer.kernel_zero.value)
    check_layer(layer, x, units)
