"""GPU: the abs-max weight quantizer over the lengths of its chunks of rows (256 down to 32, by how many workgroups there
are), with a last chunk of one row and rows that its steps of 32 do not divide; the bits of the oracle."""

import pytest
import torch

from keras_amd import quantizers as kq
from oracle import keras_cpu_path as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("K,N", [(1, 4), (33, 260), (97, 7), (769, 768), (4097, 1600), (1025, 8196), (4100, 16388),
                                 (2049, 1001)])
def test_chunks(dev, K, N, dtype):
    g = torch.Generator().manual_seed(K * 3 + N)
    w = (torch.randn(K, N, generator=g) * 0.02).to(dtype)
    w[K - 1, 0] = 3.0   # the largest of a column in the last row
    w[:, N - 1] = 0.0
    for axis_first in (w, w[None].expand(2, K, N).contiguous()) if K * N < 1 << 20 else (w,):
        axis = axis_first.dim() - 2
        want_q, want_s = ref.abs_max_quantize(axis_first, axis, to_numpy=True)
        q, s = kq.abs_max_quantize(axis_first.to(dev), axis, to_numpy=True)
        assert torch.equal(q.cpu(), want_q) and torch.equal(s.cpu(), want_s)
