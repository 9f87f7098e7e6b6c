"""psp_spmm_window_grad_f32: the weight gradient f(Z)^T (A G) formed inside the windowed product, with (A G) W^T masked by Z, with
A G stored or with neither, against float64 products; row counts around the 64-row blocks and over several workgroups."""
import numpy as np
import pytest
import scipy.sparse as sp
import torch

from test_gpu_window import banded_csr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,KZ", [(16, 16), (16, 32), (32, 32)])
@pytest.mark.parametrize("M", [1, 17, 63, 64, 65, 129, 40003])
def test_weight_gradient_in_the_windowed_product(M, N, KZ):
    from paramspmm_ae_amd import _capi
    import ParamSpMM

    rowPtr, colIdx, val = banded_csr(M, 9, 40, M + N, far=0.1, empty_frac=0.05, hub=(M // 2, min(M, 300)))
    dev = [torch.from_numpy(x).cuda() for x in (rowPtr, colIdx, val)]
    rp, ci, v = ParamSpMM.window_build(*dev)
    A = sp.csr_matrix((val.astype(np.float64), colIdx, rowPtr), shape=(M, M))
    rng = np.random.default_rng(KZ)
    rows = M + 1  # one row past the matrix
    G, Z, W = (rng.standard_normal(s).astype(np.float32) for s in ((rows, N), (rows, KZ), (KZ, N)))
    Gd, Zd, Wd = (torch.from_numpy(x).cuda() for x in (G, Z, W))
    AG, magnitude = A @ G[:M].astype(np.float64), abs(A) @ np.abs(G[:M]).astype(np.float64)
    p, L, st = _capi.ptr, _capi.lib, torch.cuda.current_stream().cuda_stream
    for dense, relu, keep in ((True, 1, True), (False, 1, True), (False, 0, True), (False, 0, False)):
        if not L.psp_spmm_window_grad_supported(N, KZ, int(dense)):
            assert dense and KZ != N
            continue
        print("case", M, N, KZ, dense, relu, keep, flush=True)
        floats = L.psp_spmm_window_grad_workspace_floats(M, N, KZ, int(dense))
        ws = torch.full((floats,), float("nan"), device="cuda")
        dW, Y = torch.full((KZ, N), float("nan"), device="cuda"), torch.full((rows, N), float("nan"), device="cuda")

        def run():
            _capi.check(L.psp_spmm_window_grad_f32(p(rp), p(ci), p(v), p(Gd), p(Zd), KZ, relu, p(Wd) if dense else None, p(Y) if keep else None, p(dW),
                                                   p(ws), floats, M, int(ci.numel()), N, rows, st))
            return dW.clone(), Y.clone()

        got_w, got_y = run()
        f = np.maximum(Z[:M], 0) if relu else Z[:M]
        assert (np.abs(got_w.cpu().numpy() - f.T.astype(np.float64) @ AG) <= 1e-5 * (np.abs(f).T.astype(np.float64) @ magnitude) + 1e-6).all()
        if keep:
            want, scale = (AG @ W.T.astype(np.float64), magnitude @ np.abs(W.T)) if dense else (AG, magnitude)
            if dense:
                want = np.where(Z[:M] > 0, want, 0)
            y = got_y.cpu().numpy()
            assert (np.abs(y[:M] - want) <= 1e-5 * scale + 1e-6).all() and (y[M:] == 0).all()
            assert not dense or (y[:M][Z[:M] <= 0] == 0).all()
        assert torch.equal(run()[0], got_w)
