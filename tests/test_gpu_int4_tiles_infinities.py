"""GPU: rows with infinities and NaN in bfloat16 int4 calls of aligned shapes on both sides of the line between the int4 tiles
and the GEMM on the de-quantised kernel: the NaN and the infinities of the float product."""

import math

import pytest
import torch

from keras_amd.layers import Dense, EinsumDense
from keras_amd.layers.dense import int4_tile_rows_route
from keras_amd.quantization_config import Int4QuantizationConfig
from keras_amd.quantizers import unpack_int4

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("group", [128, -1])
@pytest.mark.parametrize("rows,K,N,tiles", [(513, 2048, 1024, True), (700, 1152, 1088, True), (1024, 4096, 1024, True),
                                            (1025, 4096, 1024, False), (600, 1024, 256, False)])
@pytest.mark.parametrize("kind", ["dense", "einsum"])
def test_infinite_rows(dev, rows, K, N, tiles, group, kind):
    assert bool(int4_tile_rows_route(torch.bfloat16, rows, K, N, group if group > 0 else None)) == tiles
    if kind == "dense":
        layer = Dense(N, dtype="mixed_bfloat16", device="cuda:0", use_bias=False)
        layer.build((None, K))
    else:
        layer = EinsumDense("btd,dn->btn", (None, N), dtype="mixed_bfloat16", device="cuda:0")
        layer.build((None, None, K))
    layer.quantize("int4", config=Int4QuantizationConfig(block_size=group))
    q = unpack_int4(layer._kernel.value, N, axis=-1).double()
    scale = layer.kernel_scale.value.to(torch.bfloat16).double()
    if group > 0:
        g = torch.arange(K, device=dev) // group
        w = (q - layer.kernel_zero.value.double()[g]) * scale.reshape(-1, N)[g]
    else:
        w = q / scale.reshape(-1)
    assert bool((w == 0).any())
    x = torch.randn(rows, K, generator=torch.Generator().manual_seed(rows)).to(torch.bfloat16)
    x[3, 5], x[rows // 2, K - 1], x[rows - 1, 70] = math.inf, -math.inf, math.nan
    x[7, 0] = x[7, 1] = math.inf
    x = x.to(dev)
    got = layer(x if kind == "dense" else x[None]).reshape(rows, N).double()
    odd = [3, 7, rows // 2, rows - 1]
    want = x[odd].double() @ w
    assert torch.equal(got[odd].isnan(), want.isnan()) and torch.equal(got[odd].isinf(), want.isinf())
    assert torch.equal(got[odd][want.isinf()], want[want.isinf()])
    rest = torch.ones(rows, dtype=torch.bool, device=dev)
    rest[odd] = False
    assert bool(got[rest].isfinite().all())
