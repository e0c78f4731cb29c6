"""GPU: rows at any 4-byte alignment (AUTO: the streaming kernels or, where they take longer,
the split ones), against the CPU restatement on the same logits: ids, kept prefixes, generator
states and histories, all whole numbers and compared exactly.  Vocabularies at the edges of a
part (10,240 positions) and of a 16-byte group, every base offset, and neighbours of a row that
must not be read as logits (NaN and +inf around every row)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [4, 5, 7, 63, 2047, 10237, 10238, 10239, 10240, 10241, 20479, 30717, 30718, 40957, 40961,
         100003]
# (temperature, top_p, top_k, min_p, penalty, last_n)
SETTINGS = [(0.7, 0.95, 40, 0.05, 1.1, 64), (0.0, 1.0, 0, 0.0, 1.3, 8), (1.0, 0.9, 0, 0.0, 1.0, 0),
            (1.0, 1.0, 1, 0.0, 1.0, 0), (0.6, 0.9, 200, 0.02, 1.3, 64), (1.0, 1.0, 0, 0.0, 1.2, 16)]
GREEDY = [(0.0, 1.0, 0, 0.0, 1.0, 0), (0.0, 1.0, 0, 0.0, 1.5, 32)]
NARROW = [s for s in SETTINGS if s[2] <= 64]           # (rows without a top-k among them)
# the vocabulary from which AUTO streams the 12 rows
FROM = {"mixed": 39000, "narrow": 10240, "greedy": 1 << 30}


@pytest.mark.parametrize("settings", [SETTINGS, NARROW, GREEDY], ids=["mixed", "narrow", "greedy"])
@pytest.mark.parametrize("V", SIZES)
def test_unaligned_rows(oracle, V, settings, request):
    import quasar_amd as qa
    streams = V >= FROM[request.node.callspec.id.split("-")[1]]
    r = np.random.default_rng(V)
    B = 12
    for off in range(4):
        stride = V + (off + 1) % 4
        if stride % 4 == 0 and off == 0 and V % 4 == 0:
            stride += 1
        x = r.normal(0, 2, (B, V)).astype(np.float32)
        x[1] = np.round(x[1])
        x[2, 0] = x[2, -1] = 9.0
        x[3, V // 2] = np.nan
        x[4] = -np.inf
        x[5, ::2] = -np.inf
        x[6, V - 1] = 11.0
        buf = np.full(off + B * stride + 4, np.nan, np.float32)
        buf[1::2] = np.inf
        for i in range(B):
            buf[off + i * stride:off + i * stride + V] = x[i]
        dev = qa.DeviceBuffer.from_array(buf)
        b = qa.Batch(B, V, 64)
        hist = r.integers(0, V, (B, 40)).astype(np.int32)
        hist[:, :2] = 0, V - 1
        hist[:, 2] = np.nan_to_num(x, nan=-99.0).argmax(1)
        for i in range(B):
            b.config(i, 1, *settings[i % len(settings)], seeds=[50 + i])
        b.set_history(0, hist)
        base = dev.ptr + 4 * off
        assert b.resolve_mode(base, stride, B, V) == (qa.MODE_STREAM if streams else qa.MODE_SPLIT)
        got = [b.pick(base, stride, B, V, diag=True) for _ in range(2)]
        for i in range(B):
            s = oracle.sampler()
            s.config(*settings[i % len(settings)], seed=50 + i)
            s.set_history(hist[i])
            for k in range(2):
                want, od = s.pick_diag(x[i])
                at = (V, off, i, k, got[k][1][i].path, got[k][1][i].fallback)
                assert int(got[k][0][i]) == want, at
                if settings[i % len(settings)][0] > 0:
                    assert got[k][1][i].keep == od["keep"], at
            rng, h = b.get_state(i)
            assert rng == s.rng and (h == s.history()).all(), (V, off, i)
        b.close()
        dev.free()


# top_k, rows, the vocabulary from which AUTO streams
@pytest.mark.parametrize("top_k,rows,first", [
    (1, 4, 25600), (64, 100, 25600), (65, 4, 35840), (128, 100, 35840), (200, 4, 39000),
    (512, 4, 99840), (5000, 4, 99840), (0, 64, 10240), (0, 65, 25600), (0, 1, 10240)])
def test_route_of_unaligned_rows(top_k, rows, first):
    """Which kernels AUTO takes for rows that are not 16-byte aligned: the split kernels below a
    line in the vocabulary, where streaming falls short of candidates (2,048 rows of 1,001 logits
    took 24 ms a pick for 44 us), and for an all-greedy pick."""
    import quasar_amd as qa
    V = 120001
    b = qa.Batch(rows, V, 8)
    b.config(0, rows, 0.7, 0.95, top_k, 0.05, 1.0, 0)
    buf = qa.DeviceBuffer(4)                            # (nothing is read)
    for v, want in ((4, 0), (first - 1, 0), (first, 1), (V, 1)):
        assert (b.resolve_mode(buf.ptr, v + 1 + v % 2, rows, v) == qa.MODE_STREAM) == bool(want), v
    b.config(0, rows, temperature=0.0)
    assert b.resolve_mode(buf.ptr, V, rows, V) == qa.MODE_SPLIT
    b.close()
    buf.free()


@pytest.mark.parametrize("rows,V,cfg", [
    (512, 1001, (0.7, 0.95, 40, 0.05, 1.1, 64)), (256, 10001, (0.8, 0.95, 200, 0.02, 1.0, 0)),
    (100, 100003, (0.0, 1.0, 0, 0.0, 1.0, 0)), (128, 1001, (0.7, 1.0, 0, 0.05, 1.0, 0))])
def test_unaligned_picks_are_not_slower_than_split(rows, V, cfg):
    """AUTO within 1.2 times the split kernels' time where streaming took 1.3 to 48 times."""
    import quasar_amd as qa
    r = np.random.default_rng(V)
    x = r.normal(0, 1.5, (rows, V)).astype(np.float32)
    x[np.arange(rows), r.integers(0, V, rows)] += 12
    dev = qa.DeviceBuffer.from_array(x)
    us = {}
    for mode in (qa.MODE_SPLIT, qa.MODE_AUTO) * 3:
        b = qa.Batch(rows, V, 64)
        b.set_mode(mode)
        b.config(0, rows, *cfg, seeds=np.arange(1, rows + 1))
        us[mode] = min(us.get(mode, 1e9), b.time_picks(dev.ptr, V, rows, V, 30) / 30 * 1e3)
        b.close()
    print(rows, V, us, flush=True)
    assert us[qa.MODE_AUTO] <= 1.2 * us[qa.MODE_SPLIT]
    dev.free()
