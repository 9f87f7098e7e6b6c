"""The SDDMM walk changes its A row between any two entries of a step: row lengths from 0 to past every chunk, in an order that puts
row ends at every position of a step and a chunk, one row over several windows, for each group width; row maxima with them."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [4, 8, 13, 32, 64, 100, 192, 256, 300, 700])
@pytest.mark.parametrize("layout", ["plain", "balanced", "split"])
def test_sddmm_row_ends_everywhere(K, layout):
    from paramspmm_ae_amd import _capi

    lib, p = _capi.lib, _capi.ptr
    rng = np.random.default_rng(K)
    lengths = np.concatenate([rng.permutation(np.tile(np.arange(0, 36), 8)), [700], np.ones(90, int), rng.integers(0, 4, 200), [65, 64, 63, 0]])
    M, n = len(lengths), 257
    rowPtr = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    colIdx = rng.integers(0, n, rowPtr[-1]).astype(np.int32)
    row = np.repeat(np.arange(M), lengths)
    A, B = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((n, K)).astype(np.float32)
    scale = rng.standard_normal(rowPtr[-1]).astype(np.float32)
    dot = np.einsum("pk,pk->p", A[row].astype(np.float64), B[colIdx].astype(np.float64))
    tol = 1e-5 * np.einsum("pk,pk->p", np.abs(A[row]), np.abs(B[colIdx])) + 1e-6
    dev = {k: torch.from_numpy(v).cuda() for k, v in dict(rowPtr=rowPtr, colIdx=colIdx, A=A, B=B, scale=scale).items()}
    bw, S = 4, M
    if layout == "balanced":
        bw |= 0x100
    if layout == "split":
        pieces = [(r, min(b + 8, rowPtr[r + 1])) for r in range(M) for b in range(rowPtr[r], rowPtr[r + 1], 8)]
        S = len(pieces)
        dev["target"] = torch.tensor([r for r, _ in pieces], dtype=torch.int32, device="cuda")
        dev["rowPtr"] = torch.tensor([0] + [e for _, e in pieces], dtype=torch.int32, device="cuda")
    target = [p(dev["target"])] if layout == "split" else []
    form = "_split" if layout == "split" else ""
    stream = torch.cuda.current_stream().cuda_stream
    for scaled in (False, True):
        print("case", layout, K, scaled, flush=True)
        out = torch.full((len(colIdx),), float("nan"), device="cuda")
        sc = p(dev["scale"]) if scaled else None
        _capi.check(getattr(lib, "psp_sddmm_csr%s_f32" % form)(p(dev["rowPtr"]), p(dev["colIdx"]), *target, p(dev["A"]), p(dev["B"]), sc, p(out), S, K,
                                                               bw, stream))
        want = dot * scale if scaled else dot
        assert (np.abs(out.cpu().numpy() - want) <= tol * (np.abs(scale) if scaled else 1) + 1e-6).all()
        again, top = torch.full_like(out, float("nan")), torch.full((M,), float("nan"), device="cuda")
        rows = [M] if layout == "split" else []
        _capi.check(getattr(lib, "psp_sddmm_csr%s_rowmax_f32" % form)(p(dev["rowPtr"]), p(dev["colIdx"]), *target, p(dev["A"]), p(dev["B"]), sc, p(again),
                                                                      p(top), S, *rows, K, bw, stream))
        assert torch.equal(again, out)
        want_top = np.full(M, np.finfo(np.float32).min, np.float32)
        np.maximum.at(want_top, row, out.cpu().numpy())
        assert np.array_equal(top.cpu().numpy(), want_top)
