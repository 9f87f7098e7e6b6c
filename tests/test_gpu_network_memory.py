"""The training step as one autograd node holds no more memory than the layers' own nodes, and leaves weights that have hooks to
them, so that each gradient is handed out when it is formed."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _model(net, hidden, n=200000):
    from paramspmm_ae_amd import GNN, synth
    from paramspmm_ae_amd.PCSR import pcsr_spmm
    from paramspmm_ae_amd.graph_input import graph_input

    r, c, n = synth.sbm(n, 100, 4, 1, seed=3)
    graph = graph_input("g", "")
    graph.verbose = False
    graph.load_from_csr(*synth.to_gcn_csr(r, c, n)[:3])
    op = pcsr_spmm(graph=graph, vec_size=1, if_split=False)
    torch.manual_seed(1)
    model = GNN.build_model(net, graph, {d: op for d in (16, 32, hidden)}, hidden, 32, 16)
    return model, torch.randint(0, 16, graph.y.shape, device="cuda")


def _peak(model, labels, retain=False):
    from paramspmm_ae_amd import GNN

    peaks = []
    for _ in range(2):
        model.zero_grad(set_to_none=True)
        loss = GNN.loss_of_step(model, labels)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        base = torch.cuda.memory_allocated()
        loss.backward(retain_graph=retain)
        peaks.append(torch.cuda.max_memory_allocated() - base)
        name = type(loss.grad_fn).__name__
        del loss
    return peaks[1], name


@pytest.mark.parametrize("net", ["GCN", "GIN"])
def test_peak_of_the_backward_pass(net):
    hidden = 128
    model, labels = _model(net, hidden)
    one, name = _peak(model, labels)
    assert name == "NetworkLossBackward"
    hook = model.conv3.register_forward_hook(lambda *a: None)  # layer by layer
    many, name = _peak(model, labels)
    assert name != "NetworkLossBackward"
    hook.remove()
    layer = labels.numel() * hidden * 4  # one layer's matrix: what a layer that is not given back would cost
    print("peak above the forward pass: one node %.1f MB, layer by layer %.1f MB, a layer's matrix %.1f MB"
          % (one / 1e6, many / 1e6, layer / 1e6))
    assert one <= many + layer / 4
    # a graph that is kept can be run again
    from paramspmm_ae_amd import GNN

    loss = GNN.loss_of_step(model, labels)
    first = torch.autograd.grad(loss, list(model.parameters()), retain_graph=True)
    again = torch.autograd.grad(loss, list(model.parameters()))
    assert all(torch.equal(a, b) for a, b in zip(first, again))
    with pytest.raises(RuntimeError):
        loss.backward()


def test_weights_with_hooks_get_their_gradients_layer_by_layer():
    from paramspmm_ae_amd import GNN

    model, labels = _model("GCN", 16, 2000)
    seen = []
    hooks = [model.conv2.weights.register_hook(lambda g: seen.append(2)),
             model.conv4.weights.register_post_accumulate_grad_hook(lambda p: seen.append(4))]
    for h in hooks:
        loss = GNN.loss_of_step(model, labels)
        assert type(loss.grad_fn).__name__ != "NetworkLossBackward"
        loss.backward()
        h.remove()
    assert seen == [4, 2, 4]
    assert type(GNN.loss_of_step(model, labels).grad_fn).__name__ == "NetworkLossBackward"
