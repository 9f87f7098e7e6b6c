"""An operator whose attributes are replaced between two calls: the layers use what it holds now."""
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
