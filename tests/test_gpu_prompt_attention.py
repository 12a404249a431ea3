"""GPU parity: attention of a prompt over the cache (k3q_prompt_attention) against float64, and no further from it than
the library's kernel."""

import math

import pytest
import torch

from keras_amd import ops as kops

pytestmark = pytest.mark.gpu


def attention64(q, k, v, mask):
    s = torch.matmul(q.double().transpose(1, 2), k.double().transpose(2, 3).contiguous()) / math.sqrt(q.shape[-1])
    return torch.matmul(torch.softmax(s + mask.double(), dim=-1), v.double()).transpose(1, 2)


@pytest.mark.parametrize("B,T,H,max_len,kind", [
    (1, 1, 1, 4, "causal"), (2, 17, 3, 20, "causal"), (1, 64, 2, 64, "causal"), (2, 65, 5, 128, "causal"),
    (1, 130, 2, 260, "late"), (3, 33, 2, 192, "gaps"), (2, 70, 2, 256, "bias"), (8, 128, 32, 256, "causal"),
])
def test_against_float64(dev, B, T, H, max_len, kind):
    g = torch.Generator().manual_seed(T + max_len)
    mk = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)
    q, k, v = 2 * mk(B, T, H, 128), mk(B, H, max_len, 128), mk(B, H, max_len, 128)
    keys, rows = torch.arange(max_len)[None, :], torch.arange(T)[:, None]
    if kind == "late":  # a later piece of the sequence: the first positions see many rows
        rows = rows + max_len - T
    mask = torch.zeros(T, max_len).masked_fill(keys > rows, float("-inf"))
    if kind == "gaps":  # blocks of rows that nobody, or only some positions, may attend to; the last row is open to all
        mask = torch.where((keys // 64 == 1) | ((keys + rows) % 3 == 0), float("-inf"), 0.0)
        mask[:, -1] = 0
    if kind == "bias":  # an additive mask that closes nothing
        mask = torch.randn(T, max_len, generator=g)
    mask = mask.to(torch.bfloat16)
    args = [t.to(dev) for t in (q, k, v, mask)]
    assert kops.prompt_attention_supported(*args)
    got = kops.prompt_attention(*args)
    want = attention64(*args)
    # float32 scores and sums, probabilities to 2^-17, one rounding of the result to bfloat16 (eight bits: up to
    # 2^-8 of it)
    size = torch.matmul(torch.softmax(torch.matmul(args[0].double().transpose(1, 2), args[1].double().transpose(2, 3).contiguous())
                                      / math.sqrt(128) + args[3].double(), dim=-1), args[2].double().abs()).transpose(1, 2)
    assert bool(((got.double() - want).abs() <= want.abs() * 2.0 ** -8 + size * 2.0 ** -15).all())
    library = torch.nn.functional.scaled_dot_product_attention(
        args[0].transpose(1, 2), args[1], args[2], attn_mask=args[3][None, None]).transpose(1, 2)
    err = lambda y: float((y.double() - want).norm() / want.norm())
    assert err(got) <= 1.01 * err(library), (err(got), err(library))
    # operands that lie apart or start anywhere
    wide = torch.empty(B, T, 2 * H, 128, dtype=torch.bfloat16, device=dev)
    wide[:, :, ::2] = args[0]
    off = torch.cat((args[3].flatten()[:1], args[3].flatten()))[1:].view(T, max_len)
    assert torch.equal(kops.prompt_attention(wide[:, :, ::2], args[1], args[2], off), got)


def test_closed_rows_are_not_read(dev):
    """What the mask closes for all positions may hold anything."""
    mk = lambda *s: torch.ones(*s, dtype=torch.bfloat16, device=dev)
    q, k, v = mk(1, 3, 1, 128), mk(1, 1, 192, 128), mk(1, 1, 192, 128)
    k[:, :, 64:] = float("nan")
    v[:, :, 64:] = float("nan")
    mask = torch.zeros(3, 192, dtype=torch.bfloat16, device=dev)
    mask[:, 64:] = float("-inf")
    assert torch.equal(kops.prompt_attention(q, k, v, mask), q)


def test_what_keeps_the_library(dev):
    mk = lambda *s, dtype=torch.bfloat16: torch.zeros(*s, dtype=dtype, device=dev)
    q, k, v, mask = mk(1, 2, 3, 128), mk(1, 3, 8, 128), mk(1, 3, 8, 128), mk(2, 8)
    assert kops.prompt_attention_supported(q, k, v, mask)
    assert not kops.prompt_attention_supported(mk(1, 2, 3, 64), mk(1, 3, 8, 64), mk(1, 3, 8, 64), mask)
    assert not kops.prompt_attention_supported(q, mk(1, 3, 6, 128), mk(1, 3, 6, 128), mk(2, 6))
    assert not kops.prompt_attention_supported(q.float(), k.float(), v.float(), mask.float())
    assert not kops.prompt_attention_supported(q, k, v, mask[:1])
    assert not kops.prompt_attention_supported(q.clone().requires_grad_(), k, v, mask)
    with pytest.raises(ValueError):
        kops.prompt_attention(q, k, v, mask[:1])
