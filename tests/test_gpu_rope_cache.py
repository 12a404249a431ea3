"""GPU: the prompt's rotation and cache update in one launch against the torch ops it replaces."""

import pytest
import torch

from keras_amd import ops as kops
from keras_amd.decoder_harness import apply_rope, rope_tables

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,H,max_len,first", [(1, 1, 1, 8, 3), (2, 5, 3, 64, 59), (8, 128, 32, 256, 0),
                                                 (3, 33, 5, 40, 7)])
def test_rope_cache_is_the_torch_sequence(dev, B, T, H, max_len, first):
    g = torch.Generator().manual_seed(T)
    mk = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).to(dev)
    q, k, v = mk(B, T, H, 128), mk(B, T, H, 128), mk(B, T, H, 128)
    kc, vc = mk(B, H, max_len, 128), mk(B, H, max_len, 128)
    cos_t, sin_t = rope_tables(128, max_len, dev, dtype=torch.bfloat16)
    pos = (torch.randperm(T, generator=g) + first).to(dev)  # any order
    qk = apply_rope(torch.cat((q, k), dim=2), cos_t.index_select(0, pos), sin_t.index_select(0, pos))
    want_k, want_v = kc.clone(), vc.clone()
    want_k.index_copy_(2, pos, qk[:, :, H:].transpose(1, 2))
    want_v.index_copy_(2, pos, v.transpose(1, 2))
    # (k: every second row of a larger tensor: not contiguous)
    wide = torch.empty(B, T, 2 * H, 128, dtype=torch.bfloat16, device=dev)
    wide[:, :, ::2] = k
    got = kops.rope_cache(q, wide[:, :, ::2], v, cos_t, sin_t, pos, kc, vc)
    bits = lambda t: t.contiguous().view(torch.int16)
    assert torch.equal(bits(got), bits(qk[:, :, :H]))
    assert torch.equal(bits(kc), bits(want_k)) and torch.equal(bits(vc), bits(want_v))


def test_rope_cache_position_outside(dev):
    mk = lambda *s: torch.ones(*s, dtype=torch.bfloat16, device=dev)
    kc, vc = mk(1, 2, 8, 128), mk(1, 2, 8, 128)
    cos_t, sin_t = rope_tables(128, 8, dev, dtype=torch.bfloat16)
    flag = torch.zeros(1, dtype=torch.int32, device=dev)
    x = 2 * mk(1, 2, 2, 128)
    kops.rope_cache(x, x, x, cos_t, sin_t, torch.tensor([7, 8], device=dev), kc, vc, oob_flag=flag)
    assert int(flag) == 1 and float(vc[:, :, 7].min()) == 2.0 and float(vc[:, :, :7].max()) == 1.0
