"""GPU: the float32 sums of the bfloat16 tile GEMM with four stages are sums of parts of K, as those of a K split are."""

import pytest
import torch

from keras_amd import ops as kops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,parts", [(1024, 4096, 2), (1100, 1920, 3), (129, 16512, 1)])
def test_parts_of_k_are_summed_on_their_own(dev, M, N, parts):
    """A large value at the start of K and its negative at the end of it: what lies between is lost against it within its part
    (2^24 + 2^-5 is 2^24 in float32), and kept in the parts that hold neither.  (A part that holds the negative at its end
    sums its small values first.)  parts: of 14336 values, in whole stages of 64.  Where the large values meet the small sums,
    half a unit of 2^24, which is 1, is lost; the result's own rounding to bfloat16 is up to 1, too."""
    K = 14336
    x = torch.full((M, K), 2.0 ** -5, dtype=torch.bfloat16, device=dev)
    x[:, 0], x[:, -1] = 2.0 ** 24, -2.0 ** 24
    packed = torch.full((K, N // 2), 0x11, dtype=torch.int8, device=dev)  # every weight 1
    y = kops.int4_matmul(x, packed, torch.ones(N, dtype=torch.bfloat16, device=dev), N)
    first = -(-K // 64 // parts) * 64
    want = (K - first - 1) * 2.0 ** -5 if parts > 1 else 0.0
    assert float((y.float() - want).abs().max()) <= (2.0 if parts > 1 else 0.0)
