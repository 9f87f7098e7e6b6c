"""The activation's backward at pre-activations that are not numbers: the gradient is zero where z <= 0 and passes elsewhere, NaN
included, as PyTorch's threshold_backward has it -- in every kernel that applies it, at the shapes that PyTorch serves and past them."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _with_nan(Z):
    Z = Z.clone()
    Z[::7, 3] = float("nan")
    Z[1::7, 5] = 0.0
    Z[2::7, 1] = -0.0
    Z[3::7, 2] = float("inf")
    Z[4::7, 4] = float("-inf")
    return Z


@pytest.mark.parametrize("n", [1000, 1025, 16400])
@pytest.mark.parametrize("K1,K2", [(16, 16), (48, 32), (96, 96), (128, 128)])
def test_dense_masks(n, K1, K2):
    import paramspmm_ae_amd  # noqa: F401
    import ParamSpCONV as S

    gen = torch.Generator(device="cuda").manual_seed(n + K1)
    Z, G, W = (torch.randn(*s, device="cuda", generator=gen) for s in ((n, K1), (n, K2), (K1, K2)))
    Z = _with_nan(Z)
    rp = torch.arange(n + 1, dtype=torch.int32, device="cuda")
    ci = torch.arange(n, dtype=torch.int32, device="cuda")
    want = torch.ops.aten.threshold_backward((G.cpu().double() @ W.cpu().double().t()), Z.cpu().double(), 0)
    assert int((want[torch.isnan(Z.cpu())] == 0).sum()) == 0  # PyTorch lets them pass
    size = G.cpu().abs().double() @ W.cpu().abs().double().t()
    for got in (S.dense_xwt_masked(G, W, Z), S.relu_input_backward(0, G, Z, W, rp, ci, torch.ones(n, device="cuda"), None, 1, 4)[0]):
        assert bool(((got.cpu().double() - want).abs() <= 2e-6 * size).all())
        assert bool((got.cpu()[want == 0] == 0).all())


@pytest.fixture(scope="module")
def graph():
    from paramspmm_ae_amd import synth
    from paramspmm_ae_amd.graph_input import graph_input

    r, c, n = synth.sbm(2000, 20, 8, 2, seed=3)
    g = graph_input("g", "")
    g.verbose = False
    return g.load_from_csr(*synth.to_gcn_csr(r, c, n)[:3])


@pytest.mark.parametrize("config", [(1, False, 1), (1, True, 1), (2, False, 1), (2, True, 1), None])
@pytest.mark.parametrize("N", [16, 32, 64])
def test_sparse_masks_and_layer_gradients(graph, config, N):
    from paramspmm_ae_amd import gnn_conv
    from paramspmm_ae_amd.PCSR import pcsr_spmm

    import ParamSpCONV as S

    op = (pcsr_spmm(graph=graph, vec_size=config[0], if_split=config[1], CF=config[2]) if config
          else pcsr_spmm(graph=graph, vec_size=1, if_split=False, CF=0, window=True))
    n = graph.mtx_nodes
    c = graph.csr_data
    A = torch.sparse_csr_tensor(c.rowPtr.long(), c.colIdx.long(), c.val.double(), size=(n, n))
    gen = torch.Generator(device="cuda").manual_seed(N)
    D = torch.randn(n, N, device="cuda", generator=gen)
    Z = _with_nan(torch.randn(n, N, device="cuda", generator=gen))
    tr = op.target_row if op.if_split else None
    got = S.aggregate_act(op.fmt_code, D, op.spmm_rowPtr, op.colIdx, op.val, tr, op.CF, 4, False, Z).cpu().double()
    AD = A @ D.cpu().double()
    want = torch.ops.aten.threshold_backward(AD, Z.cpu().double(), 0)
    assert bool(((got - want).abs() <= 1e-5).all()) and bool((got[want == 0] == 0).all())
    # the layer A (relu(Z) W): only the gradient of Z, its forward result holds NaN rows
    W = torch.randn(N, N, device="cuda", generator=gen)
    z = Z.clone().requires_grad_()
    dZ, = torch.autograd.grad(gnn_conv.GCNReLUInputFunction.apply(z, W, op), [z], D)
    want = torch.ops.aten.threshold_backward(AD @ W.cpu().double().t(), Z.cpu().double(), 0)
    size = AD.abs() @ W.cpu().abs().double().t()
    assert bool(((dZ.cpu().double() - want).abs() <= 1e-5 * size + 1e-5).all())
