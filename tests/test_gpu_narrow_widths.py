"""Widths of 4 to 8 columns, where the lane groups of SpMM and SDDMM are cut differently (4 and 8: one and two lanes of 16-byte
pieces; 5 to 7: four lanes, SDDMM on blocks eight lanes of one float), against the oracle; rows of every length around a chunk."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

FMTS = ["csr", "csr_split", "bcsr", "bcsr_split"]


@pytest.fixture(scope="module", params=[(0, 1), (3, 40), (700, 901)])
def matrix(oracle, request):
    """rows of lengths lo .. hi in turn: empty and single entries, around a chunk, longer than a wavefront's share"""
    from gpu_util import Formats

    lo, hi = request.param
    n = 1203
    rng = np.random.default_rng(hi)
    deg = np.array([lo + i % (hi - lo + 1) for i in range(n)]) if hi < 100 else np.where(np.arange(n) % 97 == 5, lo, 2)
    rowPtr = np.zeros(n + 1, np.int32)
    rowPtr[1:] = np.cumsum(deg)
    colIdx = np.concatenate([np.sort(rng.choice(n, d, replace=False)) for d in deg]).astype(np.int32)
    return Formats(oracle, rowPtr, colIdx, rng.uniform(0.1, 1.0, colIdx.size).astype(np.float32))


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("N", [4, 5, 6, 7, 8])
def test_spmm(oracle, matrix, fmt, N):
    from gpu_util import assert_close, spmm_abs_scale, spmm_capi, spmm_oracle

    X = np.random.default_rng(N).standard_normal((matrix.n + 1, N)).astype(np.float32)
    want = spmm_oracle(oracle, fmt, matrix, X)
    for CF, bw in ((1, 4), (1, 8), (2, 4)):
        print("case", fmt, N, CF, bw, flush=True)
        got = spmm_capi(fmt, matrix, torch.from_numpy(X).cuda(), CF, bw)
        torch.cuda.synchronize()
        assert_close(got, want, what="%s N=%d CF=%d" % (fmt, N, CF), scale=spmm_abs_scale(oracle, matrix, X, want.shape[0]))


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("K", [4, 5, 6, 7, 8])
def test_sddmm(oracle, matrix, fmt, K):
    from gpu_util import assert_close, sddmm_capi, sddmm_oracle

    rng = np.random.default_rng(K)
    A, B = (rng.standard_normal((matrix.n + 1, K)).astype(np.float32) for _ in range(2))
    A /= np.linalg.norm(A, axis=1, keepdims=True)
    B /= np.linalg.norm(B, axis=1, keepdims=True)
    want = sddmm_oracle(oracle, fmt, matrix, A, B[: matrix.n])
    for bw in (4, 8, 4 | 0x100):
        print("case", fmt, K, bw, flush=True)
        got = sddmm_capi(fmt, matrix, torch.from_numpy(A).cuda(), torch.from_numpy(B[: matrix.n]).cuda(), bw)
        torch.cuda.synchronize()
        assert_close(got, want, what="%s K=%d bw=%#x" % (fmt, K, bw))


def test_the_plan_keeps_four_entries_in_flight():
    from paramspmm_ae_amd import _capi

    for N in (5, 6, 7):
        p = _capi.spmm_plan(N, 1, 4)
        assert (p["lanes_per_row"], p["unroll"], p["col_tiles"]) == (4, 4, 1)
    assert [_capi.spmm_plan(N, 1, 4)["lanes_per_row"] for N in (4, 8, 9)] == [1, 2, 4]
