"""What a layer or a loss does under autograd modes that its native node does not serve: it says so, and never returns a result
whose derivative is silently missing."""
import pytest
import torch
import torch.autograd.forward_ad as fwd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def graph():
    from paramspmm_ae_amd import synth
    from paramspmm_ae_amd.graph_input import graph_input

    r, c, n = synth.sbm(1200, 20, 6, 2, seed=5)
    g = graph_input("g", "")
    g.verbose = False
    return g.load_from_csr(*synth.to_gcn_csr(r, c, n)[:3], if_mask=True)


def _ops(graph, window=False):
    from paramspmm_ae_amd.PCSR import pcsr_spmm

    op = pcsr_spmm(graph=graph, vec_size=1, if_split=False, CF=0 if window else 1, window=window)
    return {d: op for d in (16, 32)}


def _layers(graph, window):
    """(name, function of one tensor, that tensor): every layer and loss, as a function of its input and of its weights"""
    from paramspmm_ae_amd import gnn_conv as G

    ops, n = _ops(graph, window), graph.mtx_nodes
    gen = torch.Generator(device="cuda").manual_seed(3)
    X, W, aw = (torch.randn(*s, device="cuda", generator=gen) for s in ((n, 16), (16, 16), (1, 1)))
    labels = torch.randint(0, 16, (n,), device="cuda", generator=gen)
    col = graph.csr_data.on_device("colIdx", "cuda").unsqueeze(-1)
    for f in (G.GCNFunction, G.GCNAggregateFirstFunction, G.GCNReLUInputFunction, G.GINFunction, G.GINReLUInputFunction):
        yield f.__name__, lambda x, f=f: f.apply(x, W, ops[16]), X
        yield f.__name__ + " weights", lambda w, f=f: f.apply(X, w, ops[16]), W
    for relu in (False, True):
        yield "AGNN", lambda x: G.AGNNFunction.apply(x, W, aw, ops[16], col, relu), X
        yield "AGNN weights", lambda w: G.AGNNFunction.apply(X, w, aw, ops[16], col, relu), W
        yield "AGNN attention weight", lambda a: G.AGNNFunction.apply(X, W, a, ops[16], col, relu), aw
    yield "nll", lambda x: G.nll_loss_mean(x, labels), torch.log_softmax(X, 1)
    yield "softmax nll", lambda x: G.softmax_nll_loss_mean(x, labels), X


@pytest.mark.parametrize("window", [False, True])
def test_tangents_are_refused(graph, window):
    for name, f, at in _layers(graph, window):
        print("case", name, flush=True)
        f(at)
        with fwd.dual_level():
            for record in (False, True):
                with torch.set_grad_enabled(record), pytest.raises(NotImplementedError):
                    f(fwd.make_dual(at, torch.ones_like(at)))
            f(at)  # no tangent: as outside


def test_tangent_of_a_whole_network_is_refused(graph):
    from paramspmm_ae_amd import GNN

    model = GNN.build_model("GCN", graph, _ops(graph), 16, 32, 16)
    labels = torch.randint(0, 16, graph.y.shape, device="cuda")
    x = model.x
    with fwd.dual_level():
        model.x = fwd.make_dual(x, torch.ones_like(x))
        with pytest.raises(NotImplementedError):
            GNN.loss_of_step(model, labels)
    model.x = x
    GNN.loss_of_step(model, labels).backward()


@pytest.mark.filterwarnings("ignore")
@pytest.mark.parametrize("window", [False, True])
def test_traced_functions_compute_what_they_compute_untraced(graph, window):
    for name, f, at in _layers(graph, window):
        print("case", name, flush=True)
        traced = torch.jit.trace(f, at, check_trace=False)
        other = (at * 0.5 + 0.25).requires_grad_()
        want = f(other)
        got = traced(other)
        assert torch.equal(got, want), name
        d = torch.randn(want.shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
        for a, b in zip(torch.autograd.grad(got, [other], d), torch.autograd.grad(want, [other], d)):
            # (the windowed attention weight's sum is taken with atomics, in no fixed order)
            assert torch.allclose(a, b, rtol=1e-4 if window and "attention" in name else 0, atol=0), name


@pytest.mark.parametrize("window", [False, True])
def test_saved_tensors_go_through_the_hooks(graph, window):
    """what a node keeps for its backward pass is packed and unpacked by saved-tensor hooks (here: parked in host memory)"""
    from paramspmm_ae_amd import GNN

    for name, f, at in _layers(graph, window):
        print("case", name, flush=True)
        x, packed = at.clone().requires_grad_(), []
        want = f(x)
        d = torch.randn(want.shape, device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
        want_grad, = torch.autograd.grad(want, [x], d)
        with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t.shape), t.cpu())[1], lambda t: t.cuda()):
            got = f(x)
        grad, = torch.autograd.grad(got, [x], d)
        assert packed and torch.equal(got, want)
        assert torch.allclose(grad, want_grad, rtol=1e-4 if window and "attention" in name else 0, atol=0), name
    model = GNN.build_model("GCN", graph, _ops(graph, window), 16, 32, 16)
    labels = torch.randint(0, 16, graph.y.shape, device="cuda")
    want = torch.autograd.grad(GNN.loss_of_step(model, labels), list(model.parameters()))
    with torch.autograd.graph.save_on_cpu():
        loss = GNN.loss_of_step(model, labels)
    assert type(loss.grad_fn).__name__ == "NetworkLossBackward"
    assert all(torch.equal(a, b) for a, b in zip(torch.autograd.grad(loss, list(model.parameters())), want))
