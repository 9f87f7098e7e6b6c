"""An operator whose attributes are replaced between two calls: the layers use what it holds now, and an attention layer multiplies
its weight gradient with the columns that it is given."""
import pytest
import torch

from conftest import random_csr

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def graph():
    from paramspmm_ae_amd.graph_input import graph_input

    rowPtr, colIdx, val = random_csr(1502, 9, 33, empty_frac=0.1, hub=(6, 700), values="uniform")
    g = graph_input("t", "")
    g.verbose = False
    return g.load_from_csr(rowPtr, colIdx, val, manual_granularity=16, if_mask=True)


def test_layers_follow_the_operators_format(graph):
    from paramspmm_ae_amd import gnn_conv as G
    from paramspmm_ae_amd.PCSR import pcsr_spmm

    n, gen = graph.mtx_nodes, torch.Generator(device="cuda").manual_seed(1)
    X, W = torch.randn(n, 32, device="cuda", generator=gen), torch.randn(32, 16, device="cuda", generator=gen)
    plain, split = (pcsr_spmm(graph, vec_size=1, if_split=s) for s in (False, True))
    want = G.GCNFunction.apply(X, W, plain)
    # the row-split format by its arrays and its switch, then back again
    own = plain.rowPtr, plain.target_row, plain.if_split
    for arrays in ((split.rowPtr, split.target_row, True), own):
        was = G._native(plain)
        plain.rowPtr, plain.target_row, plain.if_split = arrays
        now = G._native(plain)
        assert now is not was and G._native(plain) is now
        assert torch.allclose(G.GCNFunction.apply(X, W, plain), want, rtol=1e-5, atol=1e-5)
    # another row pointer for the SpMM alone
    win = pcsr_spmm(graph, vec_size=1, if_split=False, CF=0, window=True)
    was = G._native(win)
    win.rowPtr_w = win.rowPtr_w.clone()
    assert G._native(win) is not was
    assert torch.allclose(G.GCNFunction.apply(X, W, win), want, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("width", [16, 144])  # one launch per direction; separate operators
@pytest.mark.parametrize("config", [(1, False), (1, True), (2, False), (2, True)])
def test_attention_weight_gradient_uses_the_columns_it_is_given(graph, width, config):
    from paramspmm_ae_amd import gnn_conv as G
    from paramspmm_ae_amd.PCSR import pcsr_spmm

    op, n, c = pcsr_spmm(graph, vec_size=config[0], if_split=config[1]), graph.mtx_nodes, graph.csr_data
    gen = torch.Generator(device="cuda").manual_seed(width)
    X, dY = (torch.randn(n, width, device="cuda", generator=gen) for _ in range(2))
    W, aw = torch.randn(width, width, device="cuda", generator=gen) / width, torch.ones(1, 1, device="cuda").requires_grad_()
    own = c.on_device("colIdx", "cuda")
    d = dY.cpu().double()
    rows = torch.repeat_interleave(torch.arange(n), c.row_nnz.long())
    # the reference's scores in the order of its mask: a row's slots of the 2x1 blocks in block order
    at = c.colIdx.long() if config[0] == 1 else op.colIdx.cpu().long()[op.mask.cpu() // 2]
    dots = (d[rows] * d[at]).sum(1)
    changed = own.clone()
    changed[::3] += 7
    inplace = own.clone()
    for k, col in enumerate((own.unsqueeze(-1), own.clone(), changed, own.unsqueeze(-1), changed.long().unsqueeze(-1), inplace, inplace)):
        if k == 6:
            inplace += 3  # the same tensor, other contents
        print("case", config, width, k, flush=True)
        got, = torch.autograd.grad(G.AGNNFunction.apply(X, W, aw, op, col, False), [aw], dY)
        w = col.reshape(-1).cpu().double()
        # the sums run in fp32: width products per dot, nnz terms; 1e-5 of the terms' sizes is some ten times their random error
        size = ((d[rows].abs() * d[at].abs()).sum(1) * w).sum()
        assert abs(float(got) - float((dots * w).sum())) <= 1e-5 * float(size)
