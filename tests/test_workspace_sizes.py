"""The workspace sizes that the library names cover every path a call of that size can take. CPU only."""

import pytest

from vybforge_amd import _lib, ops

ALL = [2, 8, 12, 13, 14, 22]


def gemm_size(ty, M, N, K):
    return _lib.lib.vybdq_gemm_workspace_size(ty, M, N, K)


@pytest.mark.parametrize("ty", [2, 8, 12, 13])
@pytest.mark.parametrize("N,K", [(1040, 5120), (5136, 17408), (1088, 5120), (5120, 28672), (64, 53248), (64, 256)])
def test_gemm_64_rows_hold_the_scaled_copy_of_x(ty, N, K):
    """From 64 rows the register bodies convert X into the workspace, row by row scaled; which body a call takes also
    depends on what the query does not see (the alignment of W), so there is room for the copy at every shape."""
    for M in (64, 65):
        assert gemm_size(ty, M, N, K) >= M * K * 2 + M * 4


@pytest.mark.parametrize("ty", ALL)
@pytest.mark.parametrize("N,K", [(2560, 9728), (5120, 17408), (17408, 5120), (1024, 5120), (320, 768), (64, 256),
                                 (4096, 53248), (9728, 2560)])
def test_gemm_few_rows_size_covers_smaller_batches(ty, N, K):
    """One workspace for the largest batch serves every smaller one: up to 64 rows the size never falls as rows are
    added, and a longer call's holds that of 64 rows."""
    sizes = [gemm_size(ty, M, N, K) for M in range(1, 65)]
    assert sizes[0] > 0 or N * K > 1 << 26
    assert sizes == sorted(sizes)
    assert all(gemm_size(ty, M, N, K) >= sizes[62] for M in (64, 65, 96, 200, 512))


@pytest.mark.parametrize("ty", ALL)
@pytest.mark.parametrize("plan", ["9,1", "40,1", "99,3", "0,1", "x"])
def test_gemm_few_rows_override_that_does_not_fit(monkeypatch, ty, plan):
    """A tuning override whose K range does not fit LDS (or that is none) leaves the planner's choice."""
    own = gemm_size(ty, 64, 512, 53248)
    own21 = gemm_size(ty, 21, 896, 12800)
    monkeypatch.setenv("VYBDQ_ROWS_PLAN", plan)
    assert gemm_size(ty, 64, 512, 53248) == own
    assert gemm_size(ty, 21, 896, 12800) == own21 > 0


def test_exl3_size_covers_smaller_batches():
    """vybdq_exl3_gemm refuses a workspace below its need: the size for a batch holds every smaller one's."""
    f = _lib.lib.vybdq_exl3_workspace_size
    for K in (128, 256, 384, 1152, 1920, 2048, 4096, 5120, 17408):
        for N in (128, 256, 768, 1024, 5120, 14848, 17408, 26624, 131072):
            sizes = [f(B, K, N) for B in range(1, 17)]
            assert sizes == sorted(sizes), (K, N)


def test_moe_exl3_size_covers_fewer_tokens():
    """vybdq_moe_forward_exl3 refuses a workspace below its need: the size for T tokens holds that of fewer."""
    f = _lib.lib.vybdq_moe_exl3_workspace_size
    Ts = list(range(1, 34)) + [48, 63, 64, 65, 100, 128, 200, 256, 512, 1024]
    for H, I in ((256, 256), (256, 1536), (512, 2048), (1024, 512), (2560, 1024), (4096, 2048)):
        for E in (8, 12, 96, 288):
            for k in (1, 4, 8):
                sizes = [f(T, H, I, E, k) for T in Ts]
                assert sizes == sorted(sizes), (H, I, E, k)


@pytest.mark.parametrize("B", [1, 2, 4, 16])
def test_exl3_splits_feed_every_wave(B):
    """Four waves of a workgroup take 64 k at a time: from K = 512 no split is planned that leaves some idle."""
    for K in (512, 1024, 1536, 1920, 2048, 4096, 5120):
        for N in (768, 1536, 2048, 5120, 9728, 14848, 17408):
            arrivals = (N // 128 * 4 + 255) // 256 * 256
            rotated = 0 if B <= 2 else (B * K * 2 + 255) // 256 * 256
            size = _lib.lib.vybdq_exl3_workspace_size(B, K, N)
            own = [s for s in range(1, 17) if arrivals + rotated + s * B * N * 4 <= size]
            assert max(own) <= -(-K // 256) or B > 2, (K, N)  # (above 2 rows the size covers batches of 2 as well)


@pytest.mark.parametrize("ty,M,N,K,wide", [
    (8, 2000, 25600, 5120, False), (22, 600, 25600, 5120, False), (14, 600, 25600, 5120, False), (8, 4096, 5120, 17408, False),
    (2, 3000, 17408, 5120, False), (2, 1700, 25600, 5120, False), (14, 512, 9728, 2560, False), (14, 300, 5120, 17408, False),
    (12, 1999, 17408, 5120, True), (14, 1999, 5120, 17408, True), (8, 2000, 17408, 5120, True), (22, 1400, 5120, 17408, True),
    (13, 3000, 5120, 17408, True), (14, 1024, 9728, 2560, True)])
def test_wide_gemm_is_taken_where_it_measured_faster(ty, M, N, K, wide):
    """Prompts whose matrix is expanded name 2 N K bytes: the shapes on either side of the rule, as measured (the first six
    ran 4 to 12% slower expanded)."""
    assert (gemm_size(ty, M, N, K) >= 2 * N * K + 2 * M * K) == wide


def test_gemm_workspace_cap():
    """A workspace of a long prompt can be capped at what the fused body uses."""
    M, N, K = 1999, 5120, 17408
    assert ops.GemmWorkspace([(M, N, K)], "cpu", 14).nbytes >= 2 * N * K
    ws = ops.GemmWorkspace([(M, N, K)], "cpu", 14, max_bytes=100 << 20)
    assert ws.nbytes == 100 << 20 and ws.buf.numel() == ws.nbytes + 256
    assert ops.GemmWorkspace([(1, 64, 256)], "cpu", 14, max_bytes=100 << 20).nbytes == gemm_size(14, 1, 64, 256)
