"""GPU: what the int8 attention projections keep beside their variables, and that an assignment leaves the assigned
tensors alone."""

import pytest
import torch

from keras_amd import _lib
from keras_amd.layers import EinsumDense

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("policy", ["float32", "bfloat16"])
@pytest.mark.parametrize("equation,output,row", [
    ("btd,dnh->btnh", (None, 8, 64), (512,)), ("btnh,nhd->btd", (None, 512), (8, 64))])
def test_projection_keeps_one_copy_of_its_kernel(dev, policy, equation, output, row):
    layer = EinsumDense(equation, output, dtype=policy, device="cuda:0")
    layer.build((None, None) + row)
    layer.quantize("int8")
    dtype = torch.float32 if policy == "float32" else torch.bfloat16
    inputs = [torch.randn(2, t, *row, device=dev).to(dtype) for t in (1, 4, 20)]
    first = [layer(x) for x in inputs]
    a = layer._kernel.value
    before = a.clone()
    layer._kernel.assign(-a)
    for x, y in zip(inputs, first):
        assert torch.equal(layer(x), -y)
    assert torch.equal(a, before)
    layer._kernel.assign(a)
    for x, y in zip(inputs, first):
        assert torch.equal(layer(x), y)
    copy = _lib.load().k3q_w8s_shadow_bytes(512, 512)
    assert layer.resident_bytes()["derived"] <= copy + 4 * 512  # (and the scales, in the compute type)
