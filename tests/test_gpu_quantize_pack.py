"""GPU: grouped weight quantisation and int4 packing in one launch against the two calls, bit for bit."""

import pytest
import torch

from keras_amd import quantizers

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("K,N,block", [(1, 4, 128), (129, 252, 128), (100, 260, 32), (300, 1028, 64), (257, 516, 7),
                                       (4096, 4096, 128), (64, 30, 32), (64, 4, 256)])
def test_quantize_and_pack_is_the_two_calls(dev, dtype, K, N, block):
    g = torch.Generator(device=dev).manual_seed(K)
    x = torch.randn(K, N, generator=g, device=dev).to(dtype)
    x[:, 1] = 0.0  # a column without a range: epsilon alone
    x[0, 0] = 65504.0
    if K > 64:  # multiples of half a step: quotients on the rounding boundary
        x[:, 2] = (torch.arange(K, device=dev) % 31).to(dtype) * 0.5
    q, scale, zero = quantizers.abs_max_quantize_grouped_with_zero_point(x, block_size=block, to_numpy=True)
    want = quantizers.pack_int4(q, axis=-1)[0]
    got, s2, z2 = quantizers.quantize_and_pack_grouped(x, block, x.device)
    assert torch.equal(got, want) and torch.equal(s2, scale) and torch.equal(z2, zero)
