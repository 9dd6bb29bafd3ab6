"""Which kernel vvli_gpu_linear runs, from the sizes and the device's compute
units alone (host arithmetic: no GPU)."""
import pytest

from vvli_amd import runtime as R

SIZES = [(2048, 2048), (8192, 2048), (16384, 2048), (4096, 2048), (2048, 8192), (3584, 18944), (18944, 3584),
         (128256, 2048), (130, 72), (200, 40), (2048, 8)]
ROWS = [1, 2, 3, 4, 5, 16, 17, 33, 64, 65, 96, 100, 127, 128, 129, 512]


def kernel(route) -> str:
    return R.LINEAR_KERNELS[route.kernel]


@pytest.mark.parametrize("cus", [32, 64, 128, 192, 256, 304])
def test_few_rows_only_where_the_gemm_takes_it(cus):
    """A call that is planned without split planes runs the few-row kernel, and
    the others above 64 rows have room for their planes: whatever the number
    of compute units (a partitioned device, a mask), the GEMM's own plan is the
    one that decides."""
    for M in ROWS:
        for N, K in SIZES:
            r = R.linear_route(M, N, K, cus)
            if kernel(r) == "few_rows":
                assert R.GEMM_KERNELS[r.gemm_kernel] == "few_rows" and M <= 128, (M, N, K, cus)
            elif M > 64:
                assert kernel(r) == "tiles" and r.scratch_bytes >= 4 * M * K, (M, N, K, cus)
                assert R.GEMM_KERNELS[r.gemm_kernel] != "few_rows", (M, N, K, cus)


def test_few_rows_past_one_round_of_a_small_device():
    # 256 and 64 items of 64 rows of W: one round of 256 CUs, more than one of 128 and of 32.
    assert kernel(R.linear_route(128, 16384, 2048, 256)) == "few_rows"
    assert kernel(R.linear_route(128, 16384, 2048, 128)) == "tiles"
    assert kernel(R.linear_route(100, 4096, 2048, 32)) == "tiles"


def test_captured_calls_that_can_do_without_scratch_do():
    """Up to 64 rows a captured call either runs a kernel without scratch, or
    one that needs it eager too; larger ones run as eager ones do."""
    seen = 0
    for M in ROWS:
        for N, K in SIZES + [(2048, 4096), (3584, 3584), (512, 4096), (1152, 896)]:
            e, c = R.linear_route(M, N, K), R.linear_route(M, N, K, captured=True)
            if M > 64 or e.scratch_bytes == 0:
                assert c.scratch_bytes == e.scratch_bytes, (M, N, K)
            if M > 64:
                assert (c.kernel, c.splits) == (e.kernel, e.splits), (M, N, K)
            if c.scratch_bytes == 0 and e.scratch_bytes > 0:
                assert kernel(e) == "few_rows" and kernel(c) == "skinny" and c.splits == 1
                seen += 1
    assert seen > 0
    # 33 x 2048 x 2048: K splits of the few-row GEMM, or the unsplit skinny kernel
    assert R.linear_route(33, 2048, 2048).scratch_bytes > 0
    assert R.linear_route(33, 2048, 2048, captured=True).scratch_bytes == 0
    # 16 x 2048 x 8192: the skinny kernel would split K too
    assert R.linear_route(16, 2048, 8192, captured=True).scratch_bytes > 0


def test_without_memory_for_partial_sums():
    """What runs when the scratch of a call cannot be had: no more than the
    skinny kernel's own (M <= 64) or the split planes need."""
    for M in ROWS:
        for N, K in SIZES + [(2048, 4096), (3584, 3584), (512, 4096), (1152, 896)]:
            e, l = R.linear_route(M, N, K), R.linear_route(M, N, K, lean=True)
            assert kernel(l) != "few_rows"
            if M > 64:
                assert kernel(l) == "tiles" and l.scratch_bytes == 64 * 1024 + 4 * M * (-(-K // 32) * 32)
            elif kernel(l) == "skinny" and l.splits == 1 or kernel(l) == "gemv":
                assert l.scratch_bytes == 0
            if kernel(e) == kernel(l):
                assert l.scratch_bytes <= e.scratch_bytes


def test_unaligned_weights_stay_off_the_copies():
    """No kernel that copies W into LDS in 16-byte units gets a W at another address."""
    for M in ROWS:
        for N, K in SIZES:
            r = R.linear_route(M, N, K, unaligned=True)
            assert kernel(r) in ("gemv", "skinny"), (M, N, K)
            assert r.scratch_bytes <= 64 * 1024 + 8 * 64 * N * 4


# Timed on both sides (us: skinny or tiles / few-row GEMM): well away from the
# lines between the kernels.
@pytest.mark.parametrize("M,N,K,want", [
    (64, 5000, 520, "skinny"),     # 8.6 / 11.6: short rows of X that don't start on cache lines
    (64, 1927, 1136, "skinny"),    # 9.0 / 10.8
    (5, 2048, 2048, "skinny"),     # 6.0 / 8.2
    (16, 2048, 8192, "few_rows"),  # 22.9 / 11.6
    (16, 9000, 3000, "few_rows"),  # 31.8 / 19.6
    (5, 50304, 2048, "few_rows"),  # 57.6 / 40.4
    (64, 512, 2048, "few_rows"),   # 18.4 / 9.2
    (65, 3584, 18944, "tiles"),    # 54.4 / 68.1: 74 K chunks a block
    (100, 11008, 4096, "tiles"),   # 43.4 / 58.7
    (128, 18944, 3584, "tiles"),   # 61.2 / 101.8: two rounds
    (65, 2048, 16384, "few_rows"), # 39.4 / 35.0: 32 chunks
    (128, 8192, 2048, "few_rows"), # 29.2 / 25.3
])
def test_the_faster_kernel(M, N, K, want):
    assert kernel(R.linear_route(M, N, K)) == want
