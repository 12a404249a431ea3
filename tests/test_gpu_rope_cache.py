"""GPU: the prompt's rotation and cache update in one launch against the torch ops it replaces."""

import pytest
import torch

from keras_amd import ops as kops
from keras_amd.decoder_harness import DecoderBlock, apply_rope, rope_tables
from keras_amd.layers.layer import as_tensor

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


def test_prompt_keeps_the_gradient_of_the_attention_projections(dev):
    """The launch is none of autograd's: where a gradient is asked for, the torch sequence runs."""
    block = DecoderBlock(256, 2, 512, dtype="bfloat16", device=dev, name="block")
    cos_t, sin_t = rope_tables(128, 16, dev, dtype=torch.bfloat16)
    pos = torch.arange(6, device=dev)
    mask = torch.zeros(6, 16, dtype=torch.bfloat16, device=dev)
    rows = lambda: (cos_t[:6], sin_t[:6], mask)
    x = torch.randn(2, 6, 256, generator=torch.Generator().manual_seed(0)).to(torch.bfloat16).to(dev)

    def run():
        cache = tuple(torch.zeros(2, 2, 16, 128, dtype=torch.bfloat16, device=dev) for _ in range(2))
        return block.forward(x, rows, cache, pos, tables=(cos_t, sin_t))

    assert not run().requires_grad
    for projection in (block.query, block.key, block.value):
        kernel = as_tensor(projection._kernel)
        kernel.requires_grad_()
        assert run().requires_grad
        with torch.no_grad():
            assert not run().requires_grad
        kernel.requires_grad_(False)
