"""The attention layer's sparse work on the PCSR formats, one launch per direction (psp_attn_*_f32), against float64
restatements of the separate operators: att[p] = alpha <X_i, X_j>, Y_i = sum att[p] X_j; G_i = sum att[p] dY_j and the sum of
<dY_i, dY_j> times the columns.  Widths at the edges of the lane groups and of the 16-byte pieces."""
import numpy as np
import pytest
import torch

from conftest import random_csr

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def graph():
    from paramspmm_ae_amd.graph_input import graph_input

    rowPtr, colIdx, val = random_csr(1502, 9, 33, empty_frac=0.1, hub=(6, 900), values="uniform")
    g = graph_input("t", "")
    g.verbose = False
    return g.load_from_csr(rowPtr, colIdx, val, manual_granularity=16, if_mask=True)


@pytest.mark.parametrize("vec,split", [(1, False), (1, True), (2, False), (2, True)])
@pytest.mark.parametrize("K", [4, 16, 17, 32, 33, 47, 64, 65, 100, 128])
def test_attention_forward_backward(graph, vec, split, K):
    from paramspmm_ae_amd.gnn_conv import _slot_columns
    from paramspmm_ae_amd.PCSR import pcsr_spmm

    import ParamSpCONV as SpCONV

    g, n = graph, graph.mtx_nodes
    op = pcsr_spmm(g, vec_size=vec, if_split=split)
    gen = torch.Generator(device="cuda").manual_seed(K)
    X = torch.nn.functional.normalize(torch.randn(n, K, device="cuda", generator=gen), dim=1)
    dY = torch.randn(n, K, device="cuda", generator=gen)
    alpha = torch.tensor([1.7], device="cuda")
    fmt = op.fmt_code
    for bw in (4, 8):
        print("case", vec, split, K, bw, flush=True)
        att, Y = SpCONV.attn_forward(fmt, X, op.rowPtr, op.colIdx, op.val, op.target_row, alpha, bw)
        csr = att if vec == 1 else att.view(-1)[op.mask]
        # entries in the order of csr: CSR entries, or the slots of the mask
        rows = torch.repeat_interleave(torch.arange(n, device="cuda"), g.csr_data.row_nnz.cuda().long())
        if vec == 1:
            cols = op.colIdx.long()
        else:
            cols = op.colIdx.long()[op.mask // 2]
            assert int(torch.count_nonzero(att[op.val == 0])) == 0
        Xd, dYd = X.double().cpu(), dY.double().cpu()
        r, c = rows.cpu(), cols.cpu()
        want = 1.7 * (Xd[r] * Xd[c]).sum(1)
        np.testing.assert_allclose(csr.cpu().numpy(), want.numpy(), rtol=1e-5, atol=2e-6)
        scale = torch.zeros(n, K, dtype=torch.float64).index_add_(0, r, want.abs()[:, None] * Xd[c].abs())
        Yw = torch.zeros(n, K, dtype=torch.float64).index_add_(0, r, want[:, None] * Xd[c])
        assert bool(((Y.double().cpu() - Yw).abs() <= 4e-6 + 1e-5 * scale).all())
        slots = _slot_columns(op, g.csr_data.on_device("colIdx", "cuda"))
        G, wsum = SpCONV.attn_backward(fmt, dY, att, op.rowPtr, op.colIdx, op.target_row, slots, bw)
        Gw = torch.zeros(n, K, dtype=torch.float64).index_add_(0, r, want[:, None] * dYd[c])
        scale = torch.zeros(n, K, dtype=torch.float64).index_add_(0, r, want.abs()[:, None] * dYd[c].abs())
        assert bool(((G.double().cpu() - Gw).abs() <= 2e-5 + 1e-5 * scale).all())
        terms = (dYd[r] * dYd[c]).sum(1) * g.csr_data.colIdx.double()
        assert abs(float(wsum) - float(terms.sum())) <= 1e-5 * float(terms.abs().sum())
