"""GPU parity of the GEMM at a few X rows (M <= 64 with a workspace: X resident in LDS, weights
streamed past it) against the float64 oracle."""

import numpy as np
import pytest
import torch

from oracle import iquants, kquants, matmul
from tests.test_gpu_gguf import gate, to_dev, x_as
from tests.test_gpu_kquant import _x_pattern
from vybforge_amd import ops, synth
from vybforge_amd._lib import call, lib

pytestmark = pytest.mark.gpu

TYPES = [ops.GGML_Q4_0, ops.GGML_Q8_0, ops.GGML_Q4_K, ops.GGML_Q5_K, ops.GGML_Q6_K, ops.GGML_IQ2_S]
# (M, N, K): one row and full row fragments; one super-block; tiles of 64, 128 and 256 weight rows;
# odd super-block counts (Q6_K / IQ2_S rows at every 2-byte alignment within 16); K ranges split
SHAPES = [(1, 64, 256), (9, 192, 768), (16, 256, 512), (17, 384, 1280), (32, 512, 2304), (33, 128, 5120),
          (48, 640, 1024), (63, 320, 768), (64, 256, 17408)]


def weights(ty, rng, N, K):
    if ty == ops.GGML_Q4_0:
        raw = synth.q4_0_weights(rng, N, K)
        return raw, matmul.q4_0_matrix(raw, N, K)
    if ty == ops.GGML_Q8_0:
        raw = synth.q8_0_weights(rng, N, K)
        return raw, matmul.q8_0_matrix(raw, N, K)
    raw = synth.kquant_weights(rng, ty, N, K)
    return raw, (iquants.matrix_iq2_s if ty == ops.GGML_IQ2_S else lambda r, n, k: kquants.matrix(ty, r, n, k))(raw, N, K)


@pytest.mark.parametrize("ty", TYPES)
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_rows_gemm(dev, ty, M, N, K):
    """Every type at the edges of tiles, row fragments and K ranges; the same call without a workspace (the
    general tiles) agrees within the gate."""
    rng = np.random.default_rng(ty * 1000 + M + N + K)
    raw, w = weights(ty, rng, N, K)
    xd, x64 = x_as(synth.activations(rng, (M, K)), ("bf16", "f16", "f32")[(M + ty) % 3], dev)
    xd = xd.reshape(M, K)
    Wd = to_dev(raw, dev)
    ws = ops.GemmWorkspace([(M, N, K)], dev, ty)
    assert ws.nbytes > 0
    ref = matmul.gemm_rows_f64(x64.reshape(M, K), w)
    assert matmul.rel_maxnorm(ops.gemm(ty, Wd, xd, N, K, workspace=ws).cpu().numpy(), ref) < matmul.TOL
    assert matmul.rel_maxnorm(ops.gemm(ty, Wd, xd, N, K).cpu().numpy(), ref) < matmul.TOL


@pytest.mark.parametrize("ty", TYPES)
@pytest.mark.parametrize("plan,K,splits", [("1,1", 1792, 7), ("2,3", 1792, 4), ("3,2", 1792, 3), ("9,1", 1024, 1),
                                           ("1,2,2", 1792, 7), ("3,1,2", 1792, 3), ("2,2,1", 768, 2), ("9,9,2", 1024, 1)])
def test_rows_gemm_plans(dev, monkeypatch, ty, plan, K, splits):
    """Forced K ranges and workgroups per range: several tiles per workgroup (the LDS stages run on across
    tiles), a ragged last range, one range (a K whose X fits LDS for every type), rows in groups of 16 and all in one
    workgroup; f64 output with a residual and a wider row stride."""
    monkeypatch.setenv("VYBDQ_TUNING", "1")
    monkeypatch.setenv("VYBDQ_ROWS_PLAN", plan)
    M, N, ldy = 21, 896, 1000
    rng = np.random.default_rng(ty + len(plan))
    raw, w = weights(ty, rng, N, K)
    x = synth.activations(rng, (M, K)).astype(np.float16)
    rs = synth.activations(rng, (M, ldy)).astype(np.float64)
    Wd, Xd, y = to_dev(raw, dev), to_dev(x, dev), to_dev(rs, dev)
    ws = ops.GemmWorkspace([(M, N, K)], dev, ty)
    assert ws.nbytes == (splits * M * N * 4 if splits > 1 else 256)  # the forced plan
    call("vybdq_gemm_ws", ty, Wd.data_ptr(), Xd.data_ptr(), y.data_ptr(), M, N, K, ops.F16, ops._dt(torch.float64), ldy,
         y.data_ptr(), ws.ptr, ws.nbytes, torch.cuda.current_stream().cuda_stream)
    got = y.cpu().numpy()
    assert matmul.rel_maxnorm(got[:, :N], matmul.gemm_rows_f64(x.astype(np.float64), w, rs[:, :N])) < matmul.TOL
    np.testing.assert_array_equal(got[:, N:], rs[:, N:])


@pytest.mark.parametrize("ty", TYPES)
@pytest.mark.parametrize("xdt", ["f16", "bf16", "f32"])
def test_rows_gemm_ranges(dev, ty, xdt):
    """Rows of very different magnitude, an outlier channel, an all-zero row and blocks: every row against its
    own largest output (the power-of-two scales of X are per row and super-block)."""
    M, N, K = 13, 256, 768
    rng = np.random.default_rng(ty + len(xdt))
    raw, w = weights(ty, rng, N, K)
    x = rng.standard_normal((M, K))
    big = 6e4 if xdt == "f16" else 1e30
    x *= np.array([1.0, big / 8, 1e-3, 1.0, 100.0, 1e-2, 1.0, 1.0, 0.0, 1.0, 1.0, 1.0, 10.0])[:, None]
    x[3, 300] = big
    x[6, 256:512] = 0
    x[7] += 1000.0
    xd, x64 = x_as(x.astype(np.float32), xdt, dev)
    ws = ops.GemmWorkspace([(M, N, K)], dev, ty)
    y = ops.gemm(ty, to_dev(raw, dev), xd.reshape(M, K), N, K, y_dtype=torch.float64, workspace=ws).cpu().numpy()
    ref = matmul.gemm_rows_f64(x64.reshape(M, K), w)
    assert not y[8].any()
    for m in range(M):
        if m != 8:
            assert gate(y[m:m + 1], ref[m:m + 1], torch.float64) < matmul.TOL, m


@pytest.mark.parametrize("ty", [ops.GGML_Q4_K, ops.GGML_Q6_K])
def test_rows_gemm_falls_back(dev, ty):
    """Weights at a 4-byte address take the general tiles; a workspace too small for the planned partials takes a plan
    with fewer K ranges."""
    M, N, K = 24, 256, 1024
    rng = np.random.default_rng(ty)
    raw, w = weights(ty, rng, N, K)
    x = synth.activations(rng, (M, K)).astype(np.float16)
    ref = matmul.gemm_rows_f64(x.astype(np.float64), w)
    off = torch.zeros(raw.size + 4, dtype=torch.uint8, device=dev)
    off[4:] = to_dev(raw, dev)
    Wd, Xd = to_dev(raw, dev), to_dev(x, dev)
    ws = ops.GemmWorkspace([(M, N, K)], dev, ty)
    assert matmul.rel_maxnorm(ops.gemm(ty, off[4:], Xd, N, K, workspace=ws).cpu().numpy(), ref) < matmul.TOL
    y = torch.empty((M, N), dtype=torch.float32, device=dev)
    call("vybdq_gemm_ws", ty, Wd.data_ptr(), Xd.data_ptr(), y.data_ptr(), M, N, K, ops.F16, ops.F32, 0, 0, ws.ptr, 256,
         torch.cuda.current_stream().cuda_stream)
    assert matmul.rel_maxnorm(y.cpu().numpy(), ref) < matmul.TOL
    assert lib.vybdq_gemm_workspace_size(ty, M, N, K) == ws.nbytes


@pytest.mark.parametrize("ty", TYPES)
@pytest.mark.parametrize("N,K,Mmax", [(256, 4352, 64), (320, 1280, 33), (128, 2560, 300)])
def test_rows_gemm_one_workspace(dev, ty, N, K, Mmax):
    """One workspace sized for the largest row count serves the smaller ones on k_rows_mm, and so does half of it
    (fewer K ranges): bf16 activations past fp16's range, which the general tiles would convert as they are, match."""
    rng = np.random.default_rng(ty + N + Mmax)
    raw, w = weights(ty, rng, N, K)
    xd, x64 = x_as((rng.standard_normal((Mmax, K)) * 1e6).astype(np.float32), "bf16", dev)
    Wd, x64 = to_dev(raw, dev), x64.reshape(Mmax, K)
    ws = ops.GemmWorkspace([(Mmax, N, K)], dev, ty)
    ref = matmul.gemm_rows_f64(x64, w)
    for M in (1, 9, 16, 17, 24, 31, 32, 33, 48, 63, 64):
        if M > Mmax:
            continue
        for part in (1, 2):
            y = torch.zeros((M, N), dtype=torch.float32, device=dev)
            call("vybdq_gemm_ws", ty, Wd.data_ptr(), xd.data_ptr(), y.data_ptr(), M, N, K, ops.BF16, ops.F32, 0, 0,
                 ws.ptr, ws.nbytes // part, torch.cuda.current_stream().cuda_stream)
            assert matmul.rel_maxnorm(y.cpu().numpy(), ref[:M]) < matmul.TOL, (M, part)


@pytest.mark.parametrize("kind", ["fp16_limit", "tiny", "huge"])
@pytest.mark.parametrize("xdt", ["bf16", "f32"])
@pytest.mark.parametrize("ty,N,K,at", [(ops.GGML_Q4_0, 208, 768, 0), (ops.GGML_Q8_0, 1040, 256, 0),
                                       (ops.GGML_Q8_0, 64, 53248, 0), (ops.GGML_Q4_K, 128, 1024, 4),
                                       (ops.GGML_Q5_K, 192, 512, 4), (ops.GGML_Q8_0, 256, 512, 4)])
def test_gemm_64_rows_off_the_rows_path(dev, ty, N, K, at, xdt, kind):
    """64 rows that k_rows_mm does not take (N % 64, no plan for the K, weights at a 4-byte address) keep the row
    scales of X: activations of any magnitude neither overflow nor flush to zero."""
    M = 64
    rng = np.random.default_rng(ty + N + at + len(kind))
    raw, w = weights(ty, rng, N, K)
    xd, x64 = x_as(_x_pattern(kind, rng, M, K), xdt, dev)
    W = torch.zeros(raw.size + 16, dtype=torch.uint8, device=dev)[at:at + raw.size]
    W[:] = to_dev(raw, dev)
    ws = ops.GemmWorkspace([(M, N, K)], dev, ty)
    y = ops.gemm(ty, W, xd.reshape(M, K), N, K, workspace=ws).cpu().numpy()
    assert np.all(np.isfinite(y))
    assert matmul.rel_maxnorm(y, matmul.gemm_rows_f64(x64.reshape(M, K), w)) < matmul.TOL


@pytest.mark.parametrize("ty", TYPES)
@pytest.mark.parametrize("xdt", ["bf16", "f16", "f32"])
@pytest.mark.parametrize("M,N,K", [(11, 64, 512), (30, 256, 1792), (64, 128, 1280)])
def test_rows_gemm_non_finite(dev, ty, xdt, M, N, K):
    """Infinities and NaNs of X: one, several of one sign and of both, in one super-block and in two, beside a NaN.
    Every output is what the sum over k gives (the infinity's sign, or NaN), and the other rows stay as they are."""
    rng = np.random.default_rng(ty + M + len(xdt))
    raw, w = weights(ty, rng, N, K)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[0, 5] = np.inf
    x[1, 300] = -np.inf
    x[2, [64, 70, 200]] = np.inf
    x[4, [31, 32]] = np.inf, -np.inf
    x[5, [100, K - 1]] = np.inf
    x[6, [8, 264]] = -np.inf, np.inf
    x[7, 17] = np.nan
    x[8, [40, 41]] = np.inf, np.nan
    x[M - 1, K - 256] = np.inf
    xd, x64 = x_as(x, xdt, dev)
    ws = ops.GemmWorkspace([(M, N, K)], dev, ty)
    y = ops.gemm(ty, to_dev(raw, dev), xd.reshape(M, K), N, K, workspace=ws).cpu().numpy()
    with np.errstate(invalid="ignore"):
        terms = x64.reshape(M, 1, K) * np.asarray(w, dtype=np.float64)[None]
        ref = terms.sum(-1)
    bad = [0, 1, 2, 4, 5, 6, 7, 8, M - 1]
    np.testing.assert_array_equal(y[bad], ref[bad].astype(np.float32))
    assert not np.isfinite(y[bad]).any()
    good = [m for m in range(M) if m not in bad]
    assert matmul.rel_maxnorm(y[good], ref[good]) < matmul.TOL


@pytest.mark.parametrize("ty", TYPES)
@pytest.mark.parametrize("M", [3, 20, 37, 50, 63])
@pytest.mark.parametrize("plan,splits", [("2,2", 1), ("1,3", 2)])
def test_rows_gemm_non_finite_in_place(dev, ty, M, plan, splits, monkeypatch):
    """Non-finite rows of X where a workgroup walks several tiles and Y is its own residual with a row stride: the
    residual is read once, columns past N stay."""
    monkeypatch.setenv("VYBDQ_TUNING", "1")
    monkeypatch.setenv("VYBDQ_ROWS_PLAN", plan)
    N, K, ldy = 896, 512, 1000
    rng = np.random.default_rng(ty + M)
    raw, w = weights(ty, rng, N, K)
    x = rng.standard_normal((M, K)).astype(np.float16)
    x[0, 5] = np.inf
    x[1, [200, 300]] = -np.inf, np.inf
    x[M - 1, K - 1] = np.nan
    rs = synth.activations(rng, (M, ldy)).astype(np.float64)
    Wd, Xd, y = to_dev(raw, dev), to_dev(x, dev), to_dev(rs, dev)
    ws = ops.GemmWorkspace([(M, N, K)], dev, ty)
    assert ws.nbytes == (splits * M * N * 4 if splits > 1 else 256)  # the forced plan
    call("vybdq_gemm_ws", ty, Wd.data_ptr(), Xd.data_ptr(), y.data_ptr(), M, N, K, ops.F16, ops._dt(torch.float64), ldy,
         y.data_ptr(), ws.ptr, ws.nbytes, torch.cuda.current_stream().cuda_stream)
    got = y.cpu().numpy()
    with np.errstate(invalid="ignore"):
        ref = rs[:, :N] + (x.astype(np.float64).reshape(M, 1, K) * np.asarray(w, dtype=np.float64)[None]).sum(-1)
    bad = [0, 1, M - 1]
    np.testing.assert_array_equal(got[bad, :N], ref[bad])
    good = [m for m in range(M) if m not in bad]
    if good:
        assert matmul.rel_maxnorm(got[good, :N], ref[good]) < matmul.TOL
    np.testing.assert_array_equal(got[:, N:], rs[:, N:])


@pytest.mark.parametrize("ty", TYPES)
@pytest.mark.parametrize("xdt", ["bf16", "f32"])
def test_gemm_one_workspace_above_64_rows(dev, ty, xdt):
    """A workspace sized for 257 rows of a short matrix holds less than the K splits of 129 rows and their scaled copy
    of X: the copy is kept, and activations of any magnitude match at every smaller count."""
    N, K, Mmax = 192, 1024, 257
    rng = np.random.default_rng(ty)
    raw, w = weights(ty, rng, N, K)
    xd, x64 = x_as(_x_pattern("huge", rng, Mmax, K), xdt, dev)
    Wd, x64 = to_dev(raw, dev), x64.reshape(Mmax, K)
    ws = ops.GemmWorkspace([(Mmax, N, K)], dev, ty)
    ref = matmul.gemm_rows_f64(x64, w)
    for M in (65, 96, 128, 129, 200, 256, 257):
        if M < 96 and ty in (ops.GGML_Q6_K, ops.GGML_IQ2_S):
            continue  # the 64-row tiles, which take X as it is
        y = ops.gemm(ty, Wd, xd.reshape(Mmax, K)[:M], N, K, workspace=ws).cpu().numpy()
        assert np.all(np.isfinite(y)) and matmul.rel_maxnorm(y, ref[:M]) < matmul.TOL, M
