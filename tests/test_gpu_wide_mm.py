"""GPU parity of the prefill GEMM that expands the packed matrix to fp16 in the workspace (many X rows)
against the float64 oracle; the tile height is forced (the rule takes it at large sizes only)."""

import numpy as np
import pytest
import torch

from oracle import matmul
from tests.test_gpu_gguf import gate, to_dev, x_as
from tests.test_gpu_rows_mm import TYPES, weights
from vybforge_amd import ops, synth
from vybforge_amd._lib import call

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ty", TYPES)
@pytest.mark.parametrize("mf,M,N,K", [(2, 129, 64, 256), (3, 200, 320, 768), (4, 300, 576, 512), (3, 385, 256, 1280)])
def test_wide_gemm(dev, monkeypatch, ty, mf, M, N, K):
    """Every type and tile height: partial row tiles, N that ends inside a tile, odd super-block counts."""
    monkeypatch.setenv("VYBDQ_TUNING", "1")
    monkeypatch.setenv("VYBDQ_WIDE", str(mf))
    rng = np.random.default_rng(ty * 100 + M + N)
    raw, w = weights(ty, rng, N, K)
    xd, x64 = x_as(synth.activations(rng, (M, K)), ("bf16", "f16", "f32")[(mf + ty) % 3], dev)
    ws = ops.GemmWorkspace([(M, N, K)], dev, ty)
    assert ws.nbytes >= 2 * N * K
    y = ops.gemm(ty, to_dev(raw, dev), xd.reshape(M, K), N, K, workspace=ws).cpu().numpy()
    assert matmul.rel_maxnorm(y, matmul.gemm_rows_f64(x64.reshape(M, K), w)) < matmul.TOL


@pytest.mark.parametrize("ydt", [torch.float64, torch.bfloat16])
def test_wide_gemm_residual_ldy(dev, monkeypatch, ydt):
    """A residual of the output's type and a wider row stride; rows of very different magnitude."""
    monkeypatch.setenv("VYBDQ_TUNING", "1")
    monkeypatch.setenv("VYBDQ_WIDE", "2")
    ty, M, N, K, ldy = ops.GGML_Q6_K, 150, 320, 512, 400
    rng = np.random.default_rng(3)
    raw, w = weights(ty, rng, N, K)
    x = (rng.standard_normal((M, K)) * np.where(np.arange(M) % 2, 1e-9, 1e9)[:, None]).astype(np.float32)
    rs = torch.from_numpy(synth.activations(rng, (M, ldy)).astype(np.float64)).to(ydt)
    Wd, Xd, y = to_dev(raw, dev), to_dev(x, dev), rs.clone().to(dev)
    ws = ops.GemmWorkspace([(M, N, K)], dev, ty)
    call("vybdq_gemm_ws", ty, Wd.data_ptr(), Xd.data_ptr(), y.data_ptr(), M, N, K, ops.F32, ops._dt(ydt), ldy,
         y.data_ptr(), ws.ptr, ws.nbytes, torch.cuda.current_stream().cuda_stream)
    got, r64 = y.to(torch.float64).cpu().numpy(), rs.to(torch.float64).numpy()
    ref = matmul.gemm_rows_f64(x.astype(np.float64), w, r64[:, :N])
    for m in (0, 1, 148, 149):
        assert gate(got[m:m + 1, :N], ref[m:m + 1], ydt) < matmul.TOL, m
    np.testing.assert_array_equal(got[:, N:], r64[:, N:])


def test_wide_gemm_rule(dev):
    """The rule: a long prompt of a large matrix expands it, a short one does not, and a workspace sized for the
    fused body, or capped below the expanded matrix, still serves the long one."""
    M, N, K = 1024, 9728, 2560
    ty = ops.GGML_Q6_K
    assert ops.GemmWorkspace([(M, N, K)], "cpu", ty).nbytes >= 2 * N * K
    assert ops.GemmWorkspace([(160, N, K)], "cpu", ty).nbytes < 2 * N * K
    rng = np.random.default_rng(1)
    raw, w = weights(ty, rng, N, K)
    x = torch.from_numpy(synth.activations(rng, (M, K))).to(torch.bfloat16)
    ref = matmul.gemm_rows_f64(x[::97].to(torch.float64).numpy(), w)
    Wd, Xd = to_dev(raw, dev), x.to(dev)
    capped = ops.GemmWorkspace([(M, N, K)], dev, ty, max_bytes=2 * N * K)
    assert capped.nbytes == 2 * N * K
    for ws in (ops.GemmWorkspace([(M, N, K)], dev, ty), ops.GemmWorkspace([(160, N, K)], dev, ty), capped):
        y = ops.gemm(ty, Wd, Xd, N, K, workspace=ws).cpu().numpy()
        assert matmul.rel_maxnorm(y[::97], ref) < matmul.TOL
