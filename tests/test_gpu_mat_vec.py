"""A matrix of ggml blocks times one vector (by = 0), bit for bit against the
oracle's vec_dot of every row: row counts around the changes of kernel (2048
rows) and of lanes per row (16384, 32768), columns of one block, of odd numbers
of blocks around the batches of four, the LDS limit (16384) and past it, and rows
with a byte stride above their length."""
import numpy as np
import pytest

import oracle as O
from test_gpu_headline import E  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,pad", [
    (2047, 320, 0), (2048, 64, 0), (2049, 64 * 5, 4), (2050, 64 * 9, 0), (2111, 16384, 0),
    (2048, 16448, 0), (16383, 192, 0), (16385, 64 * 7, 8), (32767, 128, 0), (32769, 64 * 11, 4)])
def test_matrix_times_vector(E, rows, cols, pad):  # noqa: F811
    from eakv_amd.hipmem import DeviceArray
    rng = np.random.default_rng(0xEA4B + rows + cols)
    L = E.lib()
    x = rng.standard_normal(rows * cols, dtype=np.float32)
    y = rng.standard_normal(cols, dtype=np.float32)
    dx, db = DeviceArray.from_host(x), DeviceArray((rows * cols // 64 * 40,), np.uint8)
    assert L.eakv_ggml_quantize_row_device(dx.ptr, db.ptr, x.size, None) == 0
    E.hipmem.synchronize()
    dx.free()
    vx = np.zeros((rows, cols // 64 * 40 + pad), np.uint8)
    vx[:, :cols // 64 * 40] = db.download().reshape(rows, -1)
    dvx, dy, ds = DeviceArray.from_host(vx), DeviceArray.from_host(y), DeviceArray((rows, 2))
    ds.zero()
    assert L.eakv_ggml_vec_dot_device(cols, ds.ptr, 8, dvx.ptr, vx.shape[1], dy.ptr, 0, rows,
                                      None) == 0
    E.hipmem.synchronize()
    got = ds.download()
    # by slices: the oracle takes a row of y for each row of x
    for r in range(0, rows, 4096):
        part = np.ascontiguousarray(vx[r:r + 4096, :cols // 64 * 40])
        want = O.ggml_vec_dot(part, np.ascontiguousarray(np.broadcast_to(y, (len(part), cols))))
        assert np.array_equal(got[r:r + 4096, 0].view(np.uint32), want.view(np.uint32))
    assert not got[:, 1].any()
