"""The two gradients of a ReLU-input layer from one kernel, and the training step as one autograd node, against float64
products and against the layers run one by one."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1024, 1025, 1055, 4097, 140000])
@pytest.mark.parametrize("k1,k2", [(16, 16), (16, 48), (32, 32), (48, 16), (64, 32), (64, 64), (80, 80), (128, 16), (16, 128)])
def test_dense_grads_of_one_kernel(n, k1, k2):
    import paramspmm_ae_amd  # noqa: F401
    import ParamSpCONV as S

    gen = torch.Generator(device="cuda").manual_seed(n + k1)
    Z, W = (torch.randn(*s, device="cuda", generator=gen) for s in ((n, k1), (k1, k2)))
    G = torch.randn(n, k2, device="cuda", generator=gen)
    # the identity as the matrix: the layer's gradients are the dense ones
    rp = torch.arange(n + 1, dtype=torch.int32, device="cuda")
    ci = torch.arange(n, dtype=torch.int32, device="cuda")
    dZ, dW = S.relu_input_backward(0, G, Z, W, rp, ci, torch.ones(n, device="cuda"), None, 1, 4)
    Zd, Gd, Wd = (t.cpu().double() for t in (Z, G, W))
    for got, want, size in ((dZ, torch.where(Zd > 0, Gd @ Wd.t(), 0.0), Gd.abs() @ Wd.abs().t()),
                            (dW, Zd.clamp(min=0).t() @ Gd, Zd.abs().t() @ Gd.abs())):
        assert ((got.cpu().double() - want).abs() <= 2e-6 * size).all()
    again = S.relu_input_backward(0, G, Z, W, rp, ci, torch.ones(n, device="cuda"), None, 1, 4)
    assert torch.equal(again[0], dZ) and torch.equal(again[1], dW)


@pytest.mark.parametrize("net", ["GCN", "GIN"])
@pytest.mark.parametrize("hidden", [16, 48])
@pytest.mark.parametrize("config", [(0, 1, 1, 4), (1, 1, 1, 4), (0, 2, 1, 4), (1, 2, 1, 4), None])
def test_training_step_as_one_node(net, hidden, config):
    from paramspmm_ae_amd import GNN, synth
    from paramspmm_ae_amd.PCSR import pcsr_spmm
    from paramspmm_ae_amd.graph_input import graph_input

    r, c, n = synth.sbm(2000, 20, 8, 2, seed=3)
    graph = graph_input("g", "")
    graph.verbose = False
    graph.load_from_csr(*synth.to_gcn_csr(r, c, n)[:3])
    ops = {d: (pcsr_spmm(graph=graph, vec_size=config[1], if_split=bool(config[0]), CF=config[2], blkWarpNum=config[3]) if config
               else pcsr_spmm(graph=graph, vec_size=1, if_split=False, CF=0, window=True)) for d in (16, 32, hidden)}
    torch.manual_seed(1)
    model = GNN.build_model(net, graph, ops, hidden, 32, 16)
    labels = torch.randint(0, 16, graph.y.shape, device="cuda")
    params = list(model.parameters())

    def step(extra=()):
        return torch.autograd.grad(GNN.loss_of_step(model, labels), params + list(extra), retain_graph=False)

    loss = GNN.loss_of_step(model, labels)
    assert type(loss.grad_fn).__name__ == "NetworkLossBackward"
    one = step()
    parts = torch.autograd.grad(loss, params[1:3])  # some of the weights only
    with pytest.raises(RuntimeError):
        loss.backward()  # its buffers are gone
    hook = model.conv3.register_forward_hook(lambda *a: None)  # a layer with a hook runs by itself
    assert type(GNN.loss_of_step(model, labels).grad_fn).__name__ != "NetworkLossBackward"
    many = step()
    hook.remove()
    for a, b in zip(one, many):
        assert (a - b).abs().max() <= 1e-5 * b.abs().max()
    for a, b in zip(parts, many[1:3]):
        assert (a - b).abs().max() <= 1e-5 * b.abs().max()
    model.x = model.x.detach().requires_grad_()
    for a, b in zip(step([model.x]), many):
        assert (a - b).abs().max() <= 1e-5 * b.abs().max()
    model.zero_grad()
    for _ in range(2):
        GNN.loss_of_step(model, labels).backward()  # accumulates
    for p, b in zip(params, many):
        assert (p.grad - 2 * b).abs().max() <= 3e-5 * b.abs().max()
