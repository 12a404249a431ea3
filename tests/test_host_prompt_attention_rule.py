"""CPU: which prompts the attention kernel is for (measured lines; the reasons stand at the rule)."""

import pytest

from keras_amd import ops as kops


@pytest.mark.parametrize("B,T,H,max_len,pays", [
    (8, 16, 32, 256, True), (8, 128, 32, 256, True), (1, 2, 16, 256, True), (8, 16, 32, 260, False), (8, 33, 32, 512, True),
    (8, 33, 32, 516, False), (1, 512, 32, 4096, False), (16, 64, 32, 256, False), (16, 128, 32, 256, True),
    (64, 512, 32, 512, True),
])
def test_rule(B, T, H, max_len, pays):
    assert kops.prompt_attention_pays(B, T, H, max_len) is pays
