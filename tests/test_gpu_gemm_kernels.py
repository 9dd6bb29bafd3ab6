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


def check_linear(M, N, K, bias, gemm_kernel):
    import torch

    route = R.linear_route(M, N, K)
    assert R.GEMM_KERNELS[route.gemm_kernel] == gemm_kernel  # the sizes still reach what they are here for
    assert R.LINEAR_KERNELS[route.kernel] == ("few_rows" if gemm_kernel == "few_rows" else "tiles")
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
    check_linear(M, N, K, bias, "256x256")


# The 128 x 256 tile: unsplit, K split three ways (summed by a pass of their
# own) and 32 ways (added atomically), ragged rows and columns.
@pytest.mark.parametrize("M,N,K,bias", [(129, 18900, 64, True), (129, 9000, 2048, False), (130, 100, 8192, True)])
def test_tile(M, N, K, bias):
    check_linear(M, N, K, bias, "128x256")


# The few-row GEMM: each row tile (16, 32, 64, 128 rows) with ragged rows and
# columns, K chunks with a tail, K splits and their sum, several items a block,
# f32 rows at an address that the copies cannot take.
@pytest.mark.parametrize("M,N,K,bias", [(7, 2049, 8192, True), (16, 20000, 2056, False), (17, 2100, 4104, True),
                                        (31, 1000, 2056, True), (48, 777, 2040, False), (64, 300, 1000, True),
                                        (65, 200, 40, False), (100, 8200, 520, True), (128, 130, 72, True),
                                        (128, 2048, 8, False)])
def test_few_rows(M, N, K, bias):
    check_linear(M, N, K, bias, "few_rows")


def test_few_rows_unaligned_and_repeated():
    import torch

    M, N, K = 33, 2048, 2048
    w = (torch.randn(N, K, device="cuda") * 0.02).bfloat16()
    pool = torch.randn(M * K + 1, device="cuda")
    x = pool[1:].view(M, K)  # 4-byte aligned only
    y, y2 = torch.empty(M, N, device="cuda"), torch.empty(M, N, device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    R.linear(w.data_ptr(), x.data_ptr(), y.data_ptr(), M, N, K, None, s)
    ref = x.double() @ w.double().t()
    size = x.double().abs() @ w.double().abs().t()
    assert float(((y.double() - ref).abs() / size).max()) <= 2.0**-16 + K * 2.0**-24
    x = x.clone()
    R.linear(w.data_ptr(), x.data_ptr(), y.data_ptr(), M, N, K, None, s)
    R.linear(w.data_ptr(), x.data_ptr(), y2.data_ptr(), M, N, K, None, s)
    torch.cuda.synchronize()
    assert torch.equal(y, y2)  # the splits are added in a fixed order


@pytest.mark.parametrize("M,N,K", [(65, 200, 40), (100, 2048, 2048), (130, 300, 4104)])
def test_unaligned_weights(M, N, K):
    """W at an 8-byte address: 64 rows a launch, one of them short, with and without K splits."""
    import torch

    pool = (torch.randn(N * K + 4, device="cuda") * 0.02).bfloat16()
    w = pool[4:].view(N, K)
    assert w.data_ptr() % 16 == 8
    x, b = torch.randn(M, K, device="cuda"), torch.randn(N, device="cuda").bfloat16()
    y = torch.full((M + 1, N), 7.0, device="cuda")
    R.linear(w.data_ptr(), x.data_ptr(), y.data_ptr(), M, N, K, b.data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    ref = x.double() @ w.double().t() + b.double()
    size = x.double().abs() @ w.double().abs().t() + b.double().abs()
    assert float(((y[:M].double() - ref).abs() / size).max()) <= 2.0**-16 + K * 2.0**-24
    assert bool((y[M] == 7).all())


def linear_call(w, x, y, stream):
    R.linear(w.data_ptr(), x.data_ptr(), y.data_ptr(), x.shape[0], w.shape[0], w.shape[1], None, stream.cuda_stream)


def replays(graph, y, e, exact, between):
    """Three replays, eager work and a synchronization between them, each against the eager result."""
    import torch

    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        if exact:
            assert torch.equal(y, e)
        else:
            assert float((y - e).norm() / e.norm()) <= 1e-5  # sum orders of the same 16-bit products
        between()


def test_few_rows_under_capture():
    """A call that the few-row GEMM runs with scratch and the skinny kernel
    without takes the latter under capture: on a fresh stream, and with no
    address of the stream's scratch in the graph."""
    import torch

    M, N, K = 33, 2048, 2048
    eager, cap = R.linear_route(M, N, K), R.linear_route(M, N, K, captured=True)
    assert R.LINEAR_KERNELS[eager.kernel] == "few_rows" and eager.scratch_bytes > 0
    assert R.LINEAR_KERNELS[cap.kernel] == "skinny" and cap.scratch_bytes == 0
    w = (torch.randn(N, K, device="cuda") * 0.02).bfloat16()
    x = torch.randn(M, K, device="cuda")
    y, e = torch.empty(M, N, device="cuda"), torch.empty(M, N, device="cuda")
    linear_call(w, x, e, torch.cuda.current_stream())
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        linear_call(w, x, y, torch.cuda.current_stream())
    replays(g, y, e, False, lambda: x.add_(0))


# Calls that keep scratch under capture: K-split partials of the few-row GEMM
# and of the skinny kernel, split planes with partials and without.
CAPTURED = [(16, 2048, 8192), (5, 16, 8192), (512, 2048, 2048), (300, 9000, 512)]


@pytest.mark.parametrize("M,N,K", CAPTURED)
def test_captured_scratch_outlives_growth(M, N, K):
    """The usual order: a warm-up call, the capture, then larger eager calls on
    that stream, which free and replace the scratch of its eager calls, and the
    replays on another stream beside them."""
    import torch

    assert R.linear_route(M, N, K, captured=True).scratch_bytes > 0
    w = (torch.randn(N, K, device="cuda") * 0.02).bfloat16()
    x = torch.randn(M, K, device="cuda")
    y, e = torch.empty(M, N, device="cuda"), torch.empty(M, N, device="cuda")
    wl = (torch.randn(256, 8192, device="cuda") * 0.02).bfloat16()
    xl = torch.randn(1500, 8192, device="cuda")
    yl = torch.empty(1500, 256, device="cuda")
    ref = xl[:2].double() @ wl.double().t()
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    linear_call(w, x, e, st)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        linear_call(w, x, y, torch.cuda.current_stream())
    rows = [500]

    def larger():  # one row more each time: its scratch grows again
        linear_call(wl, xl[: rows[0]], yl[: rows[0]], st)
        rows[0] += 500
        st.synchronize()
        assert float((yl[:2].double() - ref).norm() / ref.norm()) <= 1e-4

    larger()
    replays(g, y, e, True, larger)


@pytest.mark.parametrize("M,N,K", CAPTURED)
def test_first_call_of_a_stream_under_capture(M, N, K):
    """The capture's scratch is not the stream's: an eager call before the
    first replay, and one after the graph is gone, have their own."""
    import torch

    w = (torch.randn(N, K, device="cuda") * 0.02).bfloat16()
    x = torch.randn(M, K, device="cuda")
    y, y2, e = (torch.zeros(M, N, device="cuda") for _ in range(3))
    linear_call(w, x, e, torch.cuda.current_stream())
    st = torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        linear_call(w, x, y, torch.cuda.current_stream())
    linear_call(w, x, y2, st)
    torch.cuda.synchronize()
    assert torch.equal(y2, e) and not bool(y.any())
    replays(g, y, e, True, lambda: linear_call(w, x, y2, st))
    del g
    y2.zero_()
    linear_call(w, x, y2, st)
    torch.cuda.synchronize()
    assert torch.equal(y2, e)


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


def test_few_row_prefill():
    """Prompt parts on each row tile of the few-row GEMM and just past it,
    behind cached rows: q|k|v with bias, gate/up, o and down with K splits and
    K tails (width 448, 1000)."""
    check_prefill(C.Config(vocab_size=300, hidden_size=448, intermediate_size=1000, num_hidden_layers=2,
                           num_attention_heads=7, num_key_value_heads=1, max_position_embeddings=4096, rope_theta=1e6,
                           rms_norm_eps=1e-6, tie_word_embeddings=True, architecture="qwen2", qkv_bias=True),
                  [1, 16, 17, 32, 33, 64, 65, 100, 128, 129])


# The 128 x 128 tile: fewer than its three stages of 64 and an odd and even
# number of them, K tails of 8 to 56, ragged rows and columns, one block, a
# full round, K splits that are summed by a pass of their own.
@pytest.mark.parametrize("M,N,K,bias", [(129, 100, 8, True), (250, 300, 72, False), (200, 5000, 200, True),
                                        (512, 8192, 136, False), (512, 8190, 504, True), (300, 1000, 2056, True),
                                        (131, 1001, 4024, False), (700, 513, 8192, True)])
def test_square_tile(M, N, K, bias):
    check_linear(M, N, K, bias, "128x128")


def test_square_tile_prefill():
    """q|k|v with bias, gate/up, o and down with K splits and K tails (width
    448, 1000) behind cached rows, at the row counts around its tiles."""
    check_prefill(C.Config(vocab_size=300, hidden_size=448, intermediate_size=1000, num_hidden_layers=2,
                           num_attention_heads=7, num_key_value_heads=1, max_position_embeddings=4096, rope_theta=1e6,
                           rms_norm_eps=1e-6, tie_word_embeddings=True, architecture="qwen2", qkv_bias=True),
                  [140, 256, 257, 520])


def test_square_tile_under_capture():
    """A K-split call captured after a smaller one on that stream, whose scratch
    would not hold its partial sums."""
    import torch

    K = 2048
    w = (torch.randn(2048, K, device="cuda") * 0.02).bfloat16()
    x = torch.randn(512, K, device="cuda")
    y, e = torch.empty(512, 2048, device="cuda"), torch.empty(512, 2048, device="cuda")
    st = torch.cuda.Stream()
    R.linear(w.data_ptr(), x.data_ptr(), e.data_ptr(), 512, 2048, K, None, torch.cuda.current_stream().cuda_stream)
    st.wait_stream(torch.cuda.current_stream())
    R.linear(w.data_ptr(), x.data_ptr(), y.data_ptr(), 512, 16, K, None, st.cuda_stream)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st):
        R.linear(w.data_ptr(), x.data_ptr(), y.data_ptr(), 512, 2048, K, None, torch.cuda.current_stream().cuda_stream)
    for _ in range(3):
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert float((y - e).norm() / e.norm()) <= 1e-5  # sum orders of the same 16-bit products
        x += 0  # eager work between the replays
