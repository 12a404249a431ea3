"""GPU: the grouped weight quantizer where a workgroup walks several work items (groups of rows x 256 columns, 512 at a
time): one, two and three of them, a last group that is short, a last column tile that is; the bits of the oracle."""

import numpy as np
import pytest
import torch

from keras_amd import quantizers
from oracle import keras_cpu_path as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("K,N,block", [
    (128, 131072, 128),   # 512 items of whole groups: one each
    (2560, 6660, 128),    # 540: some workgroups two, the last tile 4 columns wide
    (4096, 8448, 128),    # 1056: two and three
    (2565, 6660, 128),    # 567: the last group holds 5 rows
    (1030, 8192, 64),     # 544: groups of half the registers, the last of 6 rows
    (1000, 6148, 37),     # 700: groups that no thread's rows divide
])
def test_several_items_per_workgroup(dev, K, N, block, dtype):
    g = torch.Generator().manual_seed(K + N)
    w = (torch.randn(K, N, generator=g) * 0.02).to(dtype)
    w[:, N - 1] = 0.0  # a column without a range
    want_q, want_s, want_z = ref.abs_max_quantize_grouped_with_zero_point(w, block)
    q, s, z = quantizers.abs_max_quantize_grouped_with_zero_point(w.to(dev), block_size=block, to_numpy=True)
    packed, s2, z2 = quantizers.quantize_and_pack_grouped(w.to(dev), block, dev)
    assert torch.equal(packed, quantizers.pack_int4(q, axis=-1)[0]) and torch.equal(s, s2) and torch.equal(z, z2)
    for got, want in ((q, want_q), (s, want_s), (z, want_z)):
        np.testing.assert_array_equal(got.float().cpu().numpy(), torch.as_tensor(want).float().numpy().reshape(got.shape))
