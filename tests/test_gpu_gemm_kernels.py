"""The GEMM kernels behind linear and the batched prefill, at the sizes where
their tiles, K steps and dispatch rules end.

linear is compared with f64. Bound, per output element: the bf16 weights are
exact, each f32 activation keeps at least 16 bits as two bf16 halves (relative
2^-17 per product) and K products are summed in f32 in some order (at most
K * 2^-24 relative to the sum of their sizes), so
|y - ref| <= (2^-16 + K * 2^-24) * sum_k |w x|.
"""
import numpy as np
import pytest

from vvli_amd import config as C
from vvli_amd import runtime as R

pytestmark = pytest.mark.gpu


def check_linear(M, N, K, bias):
    import torch

    g = torch.Generator(device="cuda").manual_seed(M * 31 + N * 7 + K)
    w = (torch.randn(N, K, device="cuda", generator=g) * 0.02).bfloat16()
    x = torch.randn(M, K, device="cuda", generator=g)
    b = torch.randn(N, device="cuda", generator=g).bfloat16() if bias else None
    y = torch.full((M + 1, N), 7.0, device="cuda")  # one row more: must stay as it is
    print(f"linear M={M} N={N} K={K} bias={bias}", flush=True)
    R.linear(w.data_ptr(), x.data_ptr(), y.data_ptr(), M, N, K, None if b is None else b.data_ptr(),
             torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    ref = x.double() @ w.double().t()
    size = x.double().abs() @ w.double().abs().t()
    if bias:
        ref, size = ref + b.double(), size + b.double().abs()
    worst = float(((y[:M].double() - ref).abs() / size).max())
    assert worst <= 2.0**-16 + K * 2.0**-24, f"{worst:.3e}"
    assert bool((y[M] == 7).all())


# The 256 x 256 tile (two rounds of 128 x 256 tiles in one of these): 1 to 5 K
# steps with and without a tail, ragged rows and columns.
@pytest.mark.parametrize("M,N,K,bias", [(512, 32768, 8, False), (511, 32741, 40, True), (385, 32760, 96, False),
                                        (500, 32513, 136, True), (2048, 8192, 256, False)])
def test_wide_tile(M, N, K, bias):
    check_linear(M, N, K, bias)


def rel_err(got, ref):
    return float(np.max(np.abs(got.astype(np.float64) - ref)) / np.max(np.abs(ref)))


def check_prefill(cfg, parts, tol=2e-3):
    """Batched prefill against the token loop (bar of the prefill tests: 2e-3)."""
    total = sum(parts)
    blob = R.synthetic_blob(cfg, C.WEIGHT_BF16, seed=0, stddev=0.02)
    toks = np.random.default_rng(3).integers(0, cfg.vocab_size, size=total).astype(np.uint32)
    with R.Runner(cfg, blob, total + 8) as gpu:
        got = {}
        for path in ("loop", "batched"):
            gpu.kv_clear()
            gpu.set_prefill_path(path)
            at = 0
            for n in parts:
                print(f"prefill {path} [{at}, {at + n})", flush=True)
                lg, _ = gpu.prefill(toks[at:at + n], at)
                at += n
            rows = [gpu.kv_read(l, p) for l in range(cfg.num_hidden_layers) for p in (0, total // 2, total - 1)]
            got[path] = (lg.copy(), rows)
    assert rel_err(got["batched"][0], got["loop"][0]) <= tol
    for (k, v), (rk, rv) in zip(got["batched"][1], got["loop"][1]):
        assert rel_err(k, rk) <= tol and rel_err(v, rv) <= tol


def test_wide_tile_prefill():
    """q|k|v with bias, gate/up (4624 interleaved columns), the residual
    projections (down with a K tail) all on the 256 x 256 tile: 2000 rows of
    width 4608 are two rounds of the smaller tile."""
    check_prefill(C.Config(vocab_size=300, hidden_size=4608, intermediate_size=2312, num_hidden_layers=2,
                           num_attention_heads=72, num_key_value_heads=8, max_position_embeddings=4096,
                           rope_theta=1e6, rms_norm_eps=1e-6, tie_word_embeddings=True, architecture="qwen2",
                           qkv_bias=True), [2000])
