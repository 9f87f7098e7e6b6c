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


@pytest.mark.parametrize("n", [1024, 4097, 16383, 16384])
def test_128_wide_products_of_few_rows_are_plain_fp32(n):
    """Below 16384 rows: no larger an error than PyTorch's fp32 product allows, and infinities as IEEE arithmetic has them (the
    bf16 split of 16384 rows and more gives NaN there)."""
    import paramspmm_ae_amd  # noqa: F401
    import ParamSpCONV as S

    gen = torch.Generator(device="cuda").manual_seed(n)
    Z, G, W = (torch.randn(*s, device="cuda", generator=gen) for s in ((n, 128), (n, 128), (128, 128)))
    Zd, Gd, Wd = (t.cpu().double() for t in (Z, G, W))
    for got, want, size, terms in ((S.dense_relu_xw(Z, W), Zd.relu() @ Wd, Zd.relu() @ Wd.abs(), 128),
                                   (S.dense_xw(G, W, True), Gd @ Wd.t(), Gd.abs() @ Wd.abs().t(), 128),
                                   (S.dense_xwt_masked(G, W, Z), (Gd @ Wd.t()) * (Zd > 0), Gd.abs() @ Wd.abs().t(), 128),
                                   (S.weight_gradient(Z, G), Zd.t() @ Gd, Zd.abs().t() @ Gd.abs(), n),
                                   (S.weight_gradient_relu(Z, G), Zd.relu().t() @ Gd, Zd.relu().t() @ Gd.abs(), n)):
        # a sum of m terms has at most m roundings of 2^-24 of the terms' sizes; they are random, so some ten sqrt(m) bound it
        assert bool(((got.cpu().double() - want).abs() <= 10 * terms ** 0.5 * 2.0 ** -24 * size).all())
    if n >= 16384:
        return
    G[5, 3] = float("inf")
    for got, want in ((S.dense_xw(G, W, True), G.cpu() @ W.cpu().t()),
                      (S.weight_gradient(Z, G), Z.cpu().t() @ G.cpu()),
                      (S.dense_xwt_masked(G, W, Z), torch.where(Z.cpu() > 0, G.cpu() @ W.cpu().t(), 0.0))):
        got = got.cpu()
        assert bool(want.isinf().any()) and not bool(want.isnan().any())
        assert torch.equal(got.isinf(), want.isinf()) and torch.equal(got[want.isinf()], want[want.isinf()]) and not bool(got.isnan().any())
