"""Dense <-> tiles conversion on the device (ttad_matrix_set / _get): odd and even tile sizes, leading dimensions and
offsets, so that both the paired and the single accesses and every group of columns are met. Exact."""
import numpy as np
import pytest

import tasktorrent_amd as tt

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[1], [2], [64, 33, 128, 1, 70], [512, 512, 100], [128, 128, 127], [600, 515], [16, 0, 18]])
@pytest.mark.parametrize("pad", [0, 1, 2])
@pytest.mark.parametrize("storage", ["f64", "f32"])
def test_set_get_device(ctx, sizes, pad, storage):
    import torch
    n = sum(sizes)
    rng = np.random.default_rng(n + pad)
    A = rng.standard_normal((n, n))  # A[r, c]
    buf = torch.full((n, n + pad), 7.0, dtype=torch.float64)
    buf[:, :n] = torch.from_numpy(np.ascontiguousarray(A.T))  # column-major
    M = tt.TiledMatrix(ctx, sizes, storage)
    M.set(buf.cuda())
    out = torch.full((n, n + pad), -3.0, dtype=torch.float64, device="cuda")
    got = M.get(out).cpu().numpy()
    want = np.tril(A if storage == "f64" else A.astype(np.float32).astype(np.float64))
    assert np.array_equal(got[:, :n].T, want)
    assert (got[:, n:] == -3.0).all()  # rows beyond n of a column are not touched
    assert np.array_equal(M.get(), want)  # host copy
    M.close()


@pytest.mark.parametrize("sizes", [[3] * 40, [8] * 33, [16, 15] * 9, [31, 32, 33] * 4, [64, 66, 126, 128, 130], [65, 63, 127, 129],
                                   [4] * 300 + [2048], [257, 3, 1]])
@pytest.mark.parametrize("pad", [0, 1])
@pytest.mark.parametrize("storage", ["f64", "f32"])
def test_set_get_threads_per_column(ctx, sizes, pad, storage):
    # tiles around each number of threads that share a column, and one tall tile among many small ones, whose columns a
    # bounded number of workgroups share
    import torch
    n = sum(sizes)
    A = np.random.default_rng(n).standard_normal((n, n))
    buf = torch.full((n, n + pad), 7.0, dtype=torch.float64)
    buf[:, :n] = torch.from_numpy(np.ascontiguousarray(A.T))
    M = tt.TiledMatrix(ctx, sizes, storage)
    M.set(buf.cuda())
    got = M.get(torch.full((n, n + pad), -3.0, dtype=torch.float64, device="cuda")).cpu().numpy()
    assert np.array_equal(got[:, :n].T, np.tril(A if storage == "f64" else A.astype(np.float32).astype(np.float64)))
    assert (got[:, n:] == -3.0).all()
    M.close()
