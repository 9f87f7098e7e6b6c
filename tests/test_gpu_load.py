"""graph_input.load_from_csr on the device (one native call: transfers, statistics, 2x1 blocks, row splits) against the host
builders: same arrays bit for bit, same statistics; sizes on both sides of the threaded upload and of the upload ring's length, odd and even
row counts."""
import numpy as np
import pytest
import torch

from conftest import random_csr

pytestmark = pytest.mark.gpu


def _load(arrays, **kw):
    from paramspmm_ae_amd.graph_input import graph_input

    g = graph_input("t", "")
    g.verbose = False
    return g.load_from_csr(*arrays, **kw)


@pytest.mark.parametrize("n,deg,empty,kw", [(1, 1, 0.0, {}), (2, 2, 0.0, {}), (63, 3, 0.3, {}), (3001, 9, 0.1, {}), (3000, 9, 0.01, {"manual_granularity": 5}),
                                            (200001, 14, 0.05, {}), (70000, 60, 0.0, {"is_avg_granularity": True})])
def test_native_load_equals_host_load(n, deg, empty, kw):
    if n <= 2:
        arrays = (np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32), np.ones(n, np.float32))
    else:
        arrays = random_csr(n, deg, n, empty_frac=empty, hub=(n // 2, min(n // 2, 5000)), values="uniform")
    a, b = _load(arrays, build_on="host", **kw), _load(arrays, build_on="device", **kw)
    print("case", n, deg, flush=True)
    for fa, fb in ((a.csr_data, b.csr_data), (a.bcsr_data, b.bcsr_data)):
        for k in ("rowPtr", "colIdx", "val", "rowPtr_split", "target_row", "row_nnz", "row_split_nnz"):
            x, y = getattr(fa, k), getattr(fb, k)
            assert x.dtype == y.dtype and x.shape == y.shape and torch.equal(x, y), k
            if k in ("rowPtr", "colIdx", "val", "rowPtr_split", "target_row"):
                assert torch.equal(fb.on_device(k, "cuda").cpu(), y), k
        assert fa.split_granularity == fb.split_granularity and float(fa.split_ratio) == float(fb.split_ratio)
    for k in ("max_row_nnz", "real_nrow", "nonempty_rate", "max_bw", "avg_bw"):
        assert getattr(a.csr_data, k).dtype == getattr(b.csr_data, k).dtype and float(getattr(a.csr_data, k)) == float(getattr(b.csr_data, k)), k
    np.testing.assert_allclose(b.get_info(), a.get_info(), rtol=1e-6)
    assert a.pack_rate == b.pack_rate


def test_native_load_reports_bad_arrays():
    arrays = random_csr(500, 6, 3)
    rowPtr, colIdx, val = (x.copy() for x in arrays)
    bad = rowPtr.copy()
    bad[10] = bad[12] + 1
    with pytest.raises(ValueError, match="rowPtr"):
        _load((bad, colIdx, val))
    bad = colIdx.copy()
    bad[7] = 10000
    with pytest.raises(ValueError, match="column index"):
        _load((rowPtr, bad, val))
    # rows that are not strictly ascending: the host builder takes them, the device builder alone does not
    p = int(np.argmax(np.diff(rowPtr) > 1))
    swapped = colIdx.copy()
    swapped[rowPtr[p]], swapped[rowPtr[p] + 1] = colIdx[rowPtr[p] + 1], colIdx[rowPtr[p]]
    from paramspmm_ae_amd import device_builder

    with pytest.raises(device_builder.NotCanonical):
        _load((rowPtr, swapped, val), build_on="device")
    g, want = _load((rowPtr, swapped, val)), _load((rowPtr, swapped, val), build_on="host")
    assert torch.equal(g.bcsr_data.colIdx, want.bcsr_data.colIdx) and torch.equal(g.bcsr_data.val, want.bcsr_data.val)


@pytest.mark.parametrize("n,row", [(1000003, 40), (4000001, 9)])  # 41 and 38 transfers, the row pointers of them one and two
def test_slots_of_the_upload_ring_are_used_again(n, row):
    """Arrays of more than sixteen 8 MB transfers: every slot of the page-locked ring is written again while earlier transfers are
    under way.  What arrives is what was sent, bit for bit, on the first load and on the next with other values."""
    rng = np.random.default_rng(n)
    rowPtr = (np.arange(n + 1, dtype=np.int64) * row).astype(np.int32)
    nnz = int(rowPtr[-1])
    # strictly ascending columns: a start per row, steps of 1 to 7
    start = rng.integers(0, n - 7 * row, n, dtype=np.int32)
    colIdx = (start[:, None] + np.cumsum(rng.integers(1, 8, (n, row), dtype=np.int32), axis=1, dtype=np.int32)).reshape(-1) - 1
    assert (rowPtr.nbytes + colIdx.nbytes + 4 * nnz) > 17 * (8 << 20)
    for turn in range(2):
        val = rng.random(nnz, dtype=np.float32)
        print("case", n, row, turn, flush=True)
        g = _load((rowPtr, colIdx, val), build_on="device")
        c, b = g.csr_data, g.bcsr_data
        for name, want in (("rowPtr", rowPtr), ("colIdx", colIdx), ("val", val)):
            assert torch.equal(c.on_device(name, "cuda").cpu(), torch.from_numpy(want)), name
        # the blocks that were built from the device arrays meanwhile hold every value once
        assert int(torch.count_nonzero(b.val)) == int(np.count_nonzero(val))
        assert abs(float(b.val.double().sum()) - float(val.astype(np.float64).sum())) <= 1e-9 * nnz
        assert int(b.rowPtr[-1]) == b.colIdx.numel()
        del g, c, b
