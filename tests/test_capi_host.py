"""What the C ABI answers without a device: calls that it refuses before anything is read (the arrays never are), and plans."""
import numpy as np
import pytest


@pytest.mark.parametrize("N", [5, 6, 7, 9, 47, 130])
def test_softmax_weighted_product_off_the_multiples_of_four(N):
    from paramspmm_ae_amd import _capi

    L, a = _capi.lib, np.zeros(4096, np.float32).ctypes.data
    for rc in (L.psp_spmm_csr_softmax_f32(a, a, a, a, a, a, 4, N, 4, 1, 4, None),
               L.psp_spmm_csr_split_softmax_f32(a, a, a, a, a, a, a, a, 4, N, 4, 1, 4, None)):
        assert rc == -1 and b"multiple of 4" in L.psp_last_error()


def test_plan_reports_the_width_of_the_kernels_loads():
    """``vec`` is what the rows are aligned to, ``load_width`` the kernel's template argument"""
    from paramspmm_ae_amd import _capi

    for N, vec, width in ((1, 1, 1), (2, 2, 1), (3, 1, 1), (4, 4, 4), (6, 2, 4), (47, 1, 4), (50, 2, 4), (64, 4, 4)):
        p = _capi.spmm_plan(N, 1, 4)
        assert (p["vec"], p["load_width"]) == (vec, width)
        assert p["lanes_per_row"] * p["coarsen"] * p["load_width"] * p["col_tiles"] >= N
