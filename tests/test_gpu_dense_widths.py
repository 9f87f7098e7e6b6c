"""The layers' dense products (relu(Z) W, (G W^T) where Z > 0, relu(Z)^T G) at widths across the whole range of multiples of 16
and at row counts that end inside a block, against float64 products."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K1,K2", [(16, 16), (32, 16), (16, 48), (48, 48), (80, 16), (48, 80), (64, 96), (80, 80), (96, 64), (96, 96), (112, 80),
                                   (80, 112), (112, 112), (128, 48), (128, 112), (112, 128), (96, 128), (64, 128)])
@pytest.mark.parametrize("n", [1024, 1027, 40003])
def test_dense_products(K1, K2, n):
    from paramspmm_ae_amd import _capi  # puts lib/ on sys.path

    import ParamSpCONV as S

    assert _capi.lib.psp_gemm_xw_supported(K1, K2) and _capi.lib.psp_gemm_atb_supported(K1, K2)
    gen = torch.Generator(device="cuda").manual_seed(K1 * 1000 + K2)
    Z, G, W = (torch.randn(*s, device="cuda", generator=gen) for s in ((n, K1), (n, K2), (K1, K2)))
    Zd, Gd, Wd = Z.double().cpu(), G.double().cpu(), W.double().cpu()
    print("case", K1, K2, n, flush=True)
    for got, want, scale in ((S.dense_relu_xw(Z, W), Zd.relu() @ Wd, Zd.relu() @ Wd.abs()),
                             (S.dense_xw(G, W, True), Gd @ Wd.t(), Gd.abs() @ Wd.abs().t()),
                             (S.dense_xwt_masked(G, W, Z), (Gd @ Wd.t()) * (Zd > 0), Gd.abs() @ Wd.abs().t()),
                             (S.weight_gradient_relu(Z, G), Zd.relu().t() @ Gd, Zd.relu().t() @ Gd.abs()),
                             (S.weight_gradient(Z, G), Zd.t() @ Gd, Zd.abs().t() @ Gd.abs())):
        assert got.shape == want.shape
        assert bool(((got.double().cpu() - want).abs() <= 1e-6 * scale + 1e-6).all())
    assert torch.equal(S.weight_gradient_relu(Z, G), S.weight_gradient_relu(Z, G))  # no atomics: repeats bit for bit
