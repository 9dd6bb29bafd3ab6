"""GPU parity of the batched prefill for f32 weights (prefill_f32.hip) with the
reference's token loop (src/generator.zig:243-251), restated by the oracle, and
with the library's own token loop.

Bar: 1e-5 max relative error on K/V rows and logits. Everything is f32 on both
sides, so they differ by the order of their sums: a sum of K products in one
f32 chain is off by about sqrt(K) 2^-24 of its size, 4.2e-6 for the longest
here (K = 4864), and the chains of both sides are shorter than that.
"""
import numpy as np
import pytest

from vvli_amd import config as C
from vvli_amd import runtime as R
from vvli_amd._lib import VvliError

pytestmark = pytest.mark.gpu

TOL = 1e-5


def rel_err(got, ref) -> float:
    ref = np.asarray(ref, dtype=np.float64)
    return float(np.max(np.abs(np.asarray(got, dtype=np.float64) - ref)) / max(float(np.max(np.abs(ref))), 1e-30))


def cfg(**kw) -> C.Config:
    base = dict(vocab_size=500, hidden_size=256, intermediate_size=512, num_hidden_layers=2, num_attention_heads=4,
                num_key_value_heads=2, max_position_embeddings=4096, rope_theta=1e6, rms_norm_eps=1e-6,
                tie_word_embeddings=True, architecture="qwen2", qkv_bias=True, rope_layout=C.ROPE_SPLIT_HALF)
    base.update(kw)
    return C.Config(**base)


# name -> (config, rows of one prefill call each, in order)
CASES = {
    # every row-tile count of the products and its neighbours; start > 0, ragged key chunks
    "row_tiles": (cfg(), [1, 15, 16, 17, 33, 48, 49, 64, 65, 2]),
    # K not a multiple of the 16-wide step (hidden 36 x 4 heads of 32 is not one; 100 and 1028 are K of down)
    "k_tail_100": (cfg(hidden_size=64, num_attention_heads=2, num_key_value_heads=1, intermediate_size=100), [37]),
    "k_tail_1028": (cfg(intermediate_size=1028), [70]),
    # the Qwen2.5-0.5B layer: group 7, K splits on o_proj and down
    "qwen05": (cfg(hidden_size=896, intermediate_size=4864, num_attention_heads=14, num_key_value_heads=2), [48, 20]),
    "interleaved_untied": (cfg(hidden_size=512, num_attention_heads=8, num_key_value_heads=8, qkv_bias=False,
                               tie_word_embeddings=False, architecture="llama", rope_layout=C.ROPE_INTERLEAVED,
                               rope_theta=5e5), [40]),
    "hd128": (cfg(hidden_size=896, num_attention_heads=7, num_key_value_heads=1), [29, 30]),
    "hd32": (cfg(hidden_size=128, num_attention_heads=4, num_key_value_heads=4), [131]),
    # more rows than one chunk of 2048
    "two_chunks": (cfg(hidden_size=64, intermediate_size=128, num_attention_heads=2, num_key_value_heads=1), [2100]),
}


@pytest.mark.parametrize("name", list(CASES))
def test_f32_prefill_matches_token_loop(name, oracle_mod, host_threads):
    c, parts = CASES[name]
    total = sum(parts)
    blob = R.synthetic_blob(c, C.WEIGHT_F32, seed=0, stddev=0.05)
    toks = np.random.default_rng(5).integers(0, c.vocab_size, size=total).astype(np.uint32)
    orc = oracle_mod.OracleRunner(c, blob, total + 8, threads=host_threads)
    print(f"case={name} parts={parts}", flush=True)
    with R.Runner(c, blob, total + 8) as gpu, R.Runner(c, blob, total + 8) as loop:
        loop.set_prefill_path("loop")
        start = 0
        for n in parts:
            logits, am = gpu.prefill(toks[start:start + n], start)
            ll, al = loop.prefill(toks[start:start + n], start)
            for i in range(start, start + n):
                ref = orc.forward_token(int(toks[i]), i)
            assert rel_err(logits, ref) <= TOL and rel_err(logits, ll) <= TOL, f"{name} rows [{start}, {start + n})"
            assert am == al == oracle_mod.argmax(ref)
            start += n
        for layer in range(c.num_hidden_layers):
            for pos in sorted({0, 1, total // 2, total - 1}):
                for g, r in zip(gpu.kv_read(layer, pos), orc.kv_read(layer, pos)):
                    assert rel_err(g, r) <= TOL, f"{name} kv layer {layer} pos {pos}"
        nxt = int(toks[0])
        assert rel_err(gpu.forward_token(nxt, total), orc.forward_token(nxt, total)) <= TOL


def test_f32_generation_and_paths(oracle_mod):
    c = cfg()
    blob = R.synthetic_blob(c, C.WEIGHT_F32, seed=1, stddev=0.05)
    prompt = np.arange(3, 30, dtype=np.uint32)
    with R.Runner(c, blob, 64) as gpu:
        with pytest.raises(VvliError):
            gpu.set_prefill_path("batched")  # the bf16 prefill
        a, _ = gpu.generate_greedy_measured(prompt, 12, batched_prefill=True)
        b, _ = gpu.generate_greedy_measured(prompt, 12, batched_prefill=False)
        assert a.tolist() == b.tolist()


def test_f32_prefill_without_room_for_its_buffers():
    """Prompts whose chunk buffers do not fit run the token loop, report no
    error, ask for the memory once, and take the batched prefill when there is
    room again."""
    from ctypes import byref, c_uint32

    from vvli_amd import _lib

    c = cfg()
    blob = R.synthetic_blob(c, C.WEIGHT_F32, seed=2, stddev=0.05)
    prompt = np.arange(5, 45, dtype=np.uint32)
    tries = c_uint32()

    def limit(gpu, n) -> int:
        _lib.check(_lib.lib().vvli_gpu_test_limit_prefill_memory(gpu._h, n, byref(tries)))
        return tries.value

    with R.Runner(c, blob, 64) as gpu, R.Runner(c, blob, 64) as loop:
        loop.set_prefill_path("loop")
        want = loop.prefill(prompt)[0].copy()
        limit(gpu, 1000)
        for _ in range(3):
            assert np.array_equal(gpu.prefill(prompt)[0], want)  # the same token loop
        assert limit(gpu, 2**63) == 1
        assert rel_err(gpu.prefill(prompt)[0], want) <= TOL
        gpu.prefill(prompt)
        assert limit(gpu, 2**63) == 2


@pytest.mark.parametrize("hd,heads,kv", [(64, 4, 2), (32, 7, 1), (128, 2, 2)])
def test_f32_prefill_rows_before_a_nan_row(hd, heads, kv):
    """A row that is NaN (its embedding is) leaves the rows before it as the
    token loop does: hidden keys have no weight, whatever their values."""
    c = cfg(hidden_size=hd * heads, num_attention_heads=heads, num_key_value_heads=kv)
    blob = R.synthetic_blob(c, C.WEIGHT_F32, seed=4, stddev=0.05)
    bad, at, n = 77, 25, 37  # (not the first row of a block of 16 query vectors)
    blob[bad * c.hidden_size] = np.nan  # (the embedding comes first)
    toks = np.arange(100, 100 + n, dtype=np.uint32)
    toks[at] = bad
    with R.Runner(c, blob, 64) as gpu, R.Runner(c, blob, 64) as loop:
        loop.set_prefill_path("loop")
        for r in (gpu, loop):
            r.prefill(toks[:5], 0)
            r.prefill(toks[5:], 5)
        for layer in range(c.num_hidden_layers):
            for pos in range(n):
                for g, r in zip(gpu.kv_read(layer, pos), loop.kv_read(layer, pos)):
                    assert np.array_equal(np.isnan(g), np.isnan(r)), f"layer {layer} pos {pos}"
                    assert bool(np.isnan(r).all()) == (pos == at or (pos > at and layer > 0))
                    if pos < at:
                        assert rel_err(g, r) <= TOL
