"""Which prompts of f32 weights take the batched prefill and which the token
loop (host arithmetic: no GPU). Times behind the sizes: ms, token loop / batched.
"""
import dataclasses
from ctypes import byref

import pytest

from vvli_amd import _lib
from vvli_amd import config as C

NARROW = C.Config(vocab_size=500, hidden_size=256, intermediate_size=512, num_hidden_layers=2, num_attention_heads=4,
                  num_key_value_heads=2, max_position_embeddings=40000, rope_theta=1e6, rms_norm_eps=1e-6,
                  tie_word_embeddings=True, architecture="qwen2")


def batched(cfg, start, n, kind=C.WEIGHT_F32) -> bool:
    return bool(_lib.lib().vvli_gpu_test_prefill_batched(byref(cfg.to_c(kind)), start, n))


@pytest.mark.parametrize("cfg,start,n,want", [
    (C.NAMED["qwen2.5-0.5b"](), 0, 48, True),
    (C.NAMED["qwen2.5-0.5b"](), 0, 2, True),        # 2.33 / 1.04
    (C.NAMED["qwen2.5-0.5b"](), 4000, 2, True),     # 3.03 / 2.65
    (C.NAMED["qwen2.5-0.5b"](), 16000, 2, False),   # 0.77 / 1.27 (four layers)
    (C.NAMED["qwen2.5-0.5b"](), 16000, 4, True),    # 1.51 / 1.22 (four layers)
    (C.NAMED["qwen2.5-0.5b"](), 32000, 4, False),   # 2.08 / 2.31 (four layers)
    (C.NAMED["qwen2.5-0.5b"](), 32000, 6, True),    # 3.11 / 2.30 (four layers)
    (C.NAMED["qwen2.5-0.5b"](), 32000, 2**31, True),
    (C.NAMED["llama-3.2-1b"](), 0, 1, False),       # 0.36 / 0.38 (four layers)
    (C.NAMED["llama-3.2-1b"](), 2000, 1, False),    # 0.39 / 0.51 (four layers)
    (C.NAMED["llama-3.2-1b"](), 2000, 2, True),     # 0.74 / 0.51 (four layers)
    (C.NAMED["llama-3.2-1b"](), 32000, 3, False),   # 1.75 / 2.50 (four layers)
    (C.NAMED["qwen2.5-7b"](), 0, 1, False),         # 0.44 / 0.51 (two layers)
    (NARROW, 0, 2, True),                           # 0.42 / 0.26 (eight layers)
    (NARROW, 4000, 2, False),                       # 0.56 / 0.76 (eight layers)
    (NARROW, 14000, 4, False),                      # 1.47 / 2.00 (eight layers)
    (NARROW, 24000, 6, False),                      # 2.62 / 3.25 (eight layers)
    (NARROW, 100, 33, True),
])
def test_f32_prompts(cfg, start, n, want):
    assert batched(cfg, start, n) is want


def test_bf16_prompts_and_other_head_sizes():
    assert batched(C.NAMED["llama-3.2-1b"](), 32000, 1, C.WEIGHT_BF16)
    odd = dataclasses.replace(NARROW, num_attention_heads=16, num_key_value_heads=8)  # head_dim 16
    assert not batched(odd, 0, 64) and not batched(odd, 0, 64, C.WEIGHT_BF16)
