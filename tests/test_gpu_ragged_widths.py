"""Widths that are no multiple of four: the last 16-byte piece of a feature row is moved back to end with the row and
repeats up to three columns of the piece in front of it.  Checked at the edges of the pieces and of the column tiles, with
guard values behind the outputs; the rows several wavefronts add to (row-split layouts) must count a repeated column once."""
import numpy as np
import pytest
import torch

from conftest import random_csr

pytestmark = pytest.mark.gpu

FMTS = ["csr", "csr_split", "bcsr", "bcsr_split"]


@pytest.fixture(scope="module")
def small(oracle):
    from gpu_util import Formats

    rowPtr, colIdx, val = random_csr(1501, 12, 21, empty_frac=0.1, hub=(7, 800), values="uniform")
    return Formats(oracle, rowPtr, colIdx, val)


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("N", [4, 5, 7, 9, 15, 17, 31, 33, 47, 63, 65, 127, 129, 255])
def test_spmm_ragged_widths(oracle, small, fmt, N):
    from gpu_util import assert_close, spmm_abs_scale, spmm_capi, spmm_oracle
    from paramspmm_ae_amd import _capi

    F = small
    X = np.random.default_rng(N).standard_normal((F.n + 1, N)).astype(np.float32)
    want = spmm_oracle(oracle, fmt, F, X)
    scale = spmm_abs_scale(oracle, F, X, want.shape[0])
    Xd = torch.from_numpy(X).cuda()
    for CF in (1, 2, 8, _capi.pack_cf(1, 16, 4), _capi.pack_cf(2, 4, 2, even_split=True), _capi.pack_cf(4, 4, 1, even_split=True)):
        print("case", fmt, N, CF, flush=True)
        got = spmm_capi(fmt, F, Xd, CF, 4)
        torch.cuda.synchronize()
        assert_close(got, want, what="%s N=%d CF=%#x" % (fmt, N, CF), scale=scale)


@pytest.mark.parametrize("N", [5, 47, 130])
def test_spmm_ragged_widths_write_inside_the_output(oracle, small, N):
    from gpu_util import stream
    from paramspmm_ae_amd import _capi

    F, p = small, _capi.ptr
    X = torch.randn(F.n, N, device="cuda")
    flat = torch.full((F.n * N + 8,), 7.0, device="cuda")
    Y = flat[4:4 + F.n * N]  # rows start at odd multiples of four bytes
    _capi.check(_capi.lib.psp_spmm_csr_f32(p(F.d["rowPtr"]), p(F.d["colIdx"]), p(F.d["val"]), p(X), p(Y), F.n, N, F.n, 1, 4, stream()))
    torch.cuda.synchronize()
    assert bool((flat[:4] == 7).all()) and bool((flat[-4:] == 7).all())


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("K", [4, 5, 9, 31, 33, 47, 65, 127, 255, 1023])
def test_sddmm_ragged_widths(oracle, small, fmt, K):
    from gpu_util import assert_close, sddmm_capi, sddmm_oracle

    F = small
    rng = np.random.default_rng(K)
    A = rng.standard_normal((F.n + 1, K)).astype(np.float32)
    B = rng.standard_normal((F.n, K)).astype(np.float32)
    A /= np.linalg.norm(A, axis=1, keepdims=True)
    B /= np.linalg.norm(B, axis=1, keepdims=True)
    want = sddmm_oracle(oracle, fmt, F, A, B)
    for bw in (4, 8 | 0x100):
        print("case", fmt, K, bw, flush=True)
        got = sddmm_capi(fmt, F, torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda(), bw)
        torch.cuda.synchronize()
        assert_close(got, want, what="%s K=%d bw=%#x" % (fmt, K, bw))
