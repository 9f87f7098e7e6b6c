"""Operands of the dense products that start anywhere: contiguous views into a flat buffer, on every float of a 16-byte piece,
against aligned operands."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _view(t, shift):
    """the values of t as a contiguous view that starts `shift` floats into a buffer"""
    flat = torch.empty(t.numel() + 4, device="cuda")
    view = flat[shift:shift + t.numel()].view(t.shape)
    return view.copy_(t)


@pytest.mark.parametrize("n", [1000, 1024, 16400])
@pytest.mark.parametrize("K1,K2", [(16, 16), (48, 80), (96, 96), (128, 128), (64, 16)])
def test_dense_products_of_unaligned_operands(n, K1, K2):
    import paramspmm_ae_amd  # noqa: F401
    import ParamSpCONV as S

    gen = torch.Generator(device="cuda").manual_seed(n + K1)
    Z, G, W = (torch.randn(*s, device="cuda", generator=gen) for s in ((n, K1), (n, K2), (K1, K2)))
    rp = torch.arange(n + 1, dtype=torch.int32, device="cuda")
    ci = torch.arange(n, dtype=torch.int32, device="cuda")
    one = torch.ones(n, device="cuda")

    def all_products(z, g, w):
        return (S.dense_xw(z, w, False), S.dense_xw(g, w, True), S.dense_relu_xw(z, w), S.dense_xwt_masked(g, w, z),
                S.weight_gradient(z, g), S.weight_gradient_relu(z, g), *S.relu_input_backward(0, g, z, w, rp, ci, one, None, 1, 4))

    want = all_products(Z, G, W)
    xw, xwt, grad = Z.abs() @ W.abs(), G.abs() @ W.abs().t(), Z.abs().t() @ G.abs()
    sizes = (xw, xwt, xw, xwt, grad, grad, xwt, grad)
    for shift in (1, 2, 3):
        for k in range(3):
            print("case", n, K1, K2, shift, k, flush=True)
            args = [Z, G, W]
            args[k] = _view(args[k], shift)
            for a, b, size in zip(all_products(*args), want, sizes):
                # the products that go to PyTorch may take another order of the sum there: two fp32 sums of up to 16400 terms
                # differ by a few roundings of the largest partial sum, far below 1e-5 of the sum of the terms' sizes
                assert bool(((a - b).abs() <= 1e-5 * size).all())


@pytest.mark.parametrize("k1,k2", [(32, 16), (16, 16), (32, 32)])
def test_first_layer_on_a_windowed_operator_takes_an_unaligned_input(k1, k2):
    from paramspmm_ae_amd import gnn_conv, synth
    from paramspmm_ae_amd.PCSR import pcsr_spmm
    from paramspmm_ae_amd.graph_input import graph_input

    r, c, n = synth.sbm(3000, 20, 8, 2, seed=3)
    graph = graph_input("g", "")
    graph.verbose = False
    graph.load_from_csr(*synth.to_gcn_csr(r, c, n)[:3])
    op = pcsr_spmm(graph=graph, vec_size=1, if_split=False, CF=0, window=True)
    gen = torch.Generator(device="cuda").manual_seed(1)
    X, dY = torch.randn(n, k1, device="cuda", generator=gen), torch.randn(n, k2, device="cuda", generator=gen)
    W = torch.randn(k1, k2, device="cuda", generator=gen).requires_grad_()
    got = []
    for x, g in ((X, dY), (_view(X, 1), dY), (X, _view(dY, 3))):
        out = gnn_conv.GCNFunction.apply(x, W, op)
        got.append((out.detach(), *torch.autograd.grad(out, [W], g)))
    for a in got[1:]:
        for x, y in zip(a, got[0]):
            assert torch.equal(x, y)
