"""GPU: the grouped weight quantizer on both sides of the group sizes at which a thread holds 2, 4, 8 or 16 rows: the bits of the
oracle."""

import numpy as np
import pytest
import torch

from keras_amd import quantizers
from oracle import keras_cpu_path as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("block", [1, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128])
@pytest.mark.parametrize("groups,short", [(3, 0), (300, 1)])
def test_edges_of_rows_held(dev, block, groups, short, dtype):
    """groups * 2 column tiles: fewer items than workgroups, and two a workgroup with a short last group."""
    K, N = groups * block - (short if block > 1 else 0), 260
    g = torch.Generator().manual_seed(block + groups)
    w = (torch.randn(K, N, generator=g) * 0.02).to(dtype)
    want_q, want_s, want_z = ref.abs_max_quantize_grouped_with_zero_point(w, block)
    q, s, z = quantizers.abs_max_quantize_grouped_with_zero_point(w.to(dev), block_size=block, to_numpy=True)
    packed, s2, z2 = quantizers.quantize_and_pack_grouped(w.to(dev), block, dev)
    assert torch.equal(packed, quantizers.pack_int4(q, axis=-1)[0]) and torch.equal(s, s2) and torch.equal(z, z2)
    for got, want in ((q, want_q), (s, want_s), (z, want_z)):
        np.testing.assert_array_equal(got.float().cpu().numpy(), torch.as_tensor(want).float().numpy().reshape(got.shape))
