"""GPU: the router's choice at the edges of its kernels (4, 8 or 16 experts a lane, up to 16
or up to 64 chosen), token counts at the edges of a wavefront and a workgroup, against the
CPU restatement (forward_cpu.c:165-172, 296-304): indices and weights bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("e,u", [(1, 1), (15, 15), (16, 16), (17, 17), (63, 16), (64, 64), (65, 16),
                                 (65, 17), (128, 16), (128, 17), (129, 8), (255, 64), (256, 16)])
def test_router_edges(oracle, e, u):
    import quasar_amd as qa
    r = np.random.default_rng(e * 100 + u)
    for t in (1, 3, 5, 16, 17, 1003):
        x = (r.normal(0, 2, (t, e + 3))).astype(np.float32)     # (a stride past the experts)
        x[0] = np.round(x[0])
        if t > 8:
            x[1], x[2, 0], x[3, e // 2] = 0.5, np.nan, np.nan
            x[4, e - 1], x[5], x[6, ::2] = np.inf, -np.inf, -np.inf
            x[7] *= 40.0
            x[8, 0] = 3e38
        buf = qa.DeviceBuffer.from_array(x)
        idx, wt = qa.DeviceBuffer(4 * t * u), qa.DeviceBuffer(4 * t * u)
        for norm in (0, 1):
            qa.check(qa.load().qs_router_topk(buf.ptr, e + 3, t, e, u, norm, idx.ptr, wt.ptr, None),
                     "qs_router_topk")
            qa.check(qa.load().qs_device_synchronize(), "sync")
            want_i, want_w = oracle.router_topk(np.ascontiguousarray(x[:, :e]), u, norm)
            got_w = wt.download(np.float32, t * u).reshape(t, u)
            assert (idx.download(np.int32, t * u).reshape(t, u) == want_i).all(), (t, norm)
            assert ((got_w.view(np.uint32) == want_w.view(np.uint32)) |
                    (np.isnan(got_w) & np.isnan(want_w))).all(), (t, norm)
        for b in (buf, idx, wt):
            b.free()
