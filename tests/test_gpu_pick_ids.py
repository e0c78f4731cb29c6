"""GPU: qs_batch_pick_ids (the ids stored into host memory by the kernels) against
qs_batch_pick and a copy, through each kernel that writes ids, and its error report."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,V,cfg", [
    (1, 1000, (0.0, 1.0, 0, 0.0, 1.0, 0)), (32, 5000, (0.7, 0.95, 40, 0.05, 1.1, 64)),
    (300, 2000, (0.7, 0.95, 40, 0.05, 1.1, 64)), (8, 30000, (1.0, 1.0, 0, 0.0, 1.0, 0)),
    (3, 2001, (0.7, 0.95, 40, 0.05, 1.1, 64))])
def test_pick_ids_equals_pick(rows, V, cfg):
    import quasar_amd as qa
    x = np.random.default_rng(V).normal(0, 2, (rows, V)).astype(np.float32)
    dev = qa.DeviceBuffer.from_array(x)
    a, b = qa.Batch(rows, V, 64), qa.Batch(rows, V, 64)
    for q in (a, b):
        q.config(0, rows, *cfg, seeds=np.arange(1, rows + 1))
    for k in range(3):
        n = rows if k < 2 else max(1, rows // 2)
        got = a.pick(dev.ptr, V, n, V)
        b.pick_async(dev.ptr, V, n, V)
        b.synchronize()
        assert (got == b._out.download(np.int32, n)).all(), k
    for r in range(rows):
        assert a.get_state(r)[0] == b.get_state(r)[0]
    a.close()
    b.close()
    dev.free()


def test_pick_ids_reports_a_row_to_pick_again():
    """A whole-window row without a scratch slot (a spin limit of 0): QS_EAGAIN once, the id
    -3 stored, and the next pick of the row succeeds."""
    import quasar_amd as qa
    V = 40000
    x = np.random.default_rng(3).normal(0, 1, (1, V)).astype(np.float32)
    dev = qa.DeviceBuffer.from_array(x)
    b = qa.Batch(1, V, 8)
    b.config(0, 1, 1.0, 1.0, 0, 0.0, 1.0, 0, seeds=[5])
    b.set_spin_limit(0)
    ids = np.zeros(1, np.int32)
    lib = qa.load()
    assert lib.qs_batch_pick_ids(b._b, dev.ptr, V, 1, V, ids.ctypes.data) == qa.QS_EAGAIN
    assert ids[0] == -3
    b.set_spin_limit(1 << 20)
    assert 0 <= int(b.pick(dev.ptr, V, 1, V)[0]) < V
    assert lib.qs_batch_pick_ids(b._b, dev.ptr, V, 2, V, ids.ctypes.data) == qa._native.QS_EINVAL
    b.close()
    dev.free()
