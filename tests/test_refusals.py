"""Calls that the C ABI refuses before anything reaches a device (no GPU needed: the arrays are never read)."""
import numpy as np
import pytest


@pytest.mark.parametrize("N", [5, 6, 7, 9, 47, 130])
def test_softmax_weighted_product_off_the_multiples_of_four(N):
    from paramspmm_ae_amd import _capi

    L, a = _capi.lib, np.zeros(4096, np.float32).ctypes.data
    for rc in (L.psp_spmm_csr_softmax_f32(a, a, a, a, a, a, 4, N, 4, 1, 4, None),
               L.psp_spmm_csr_split_softmax_f32(a, a, a, a, a, a, a, a, 4, N, 4, 1, 4, None)):
        assert rc == -1 and b"multiple of 4" in L.psp_last_error()
