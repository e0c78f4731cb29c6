"""GPU: rows at any 4-byte alignment through the streaming kernels (AUTO), against the CPU
restatement on the same logits: ids, kept prefixes, generator states and histories, all
whole numbers and compared exactly.  Vocabularies at the edges of a part (10,240 positions)
and of a 16-byte group, every base offset, and neighbours of a row that must not be read as
logits (NaN and +inf around every row)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [4, 5, 7, 63, 2047, 10237, 10238, 10239, 10240, 10241, 20479, 100003]
# (temperature, top_p, top_k, min_p, penalty, last_n)
SETTINGS = [(0.7, 0.95, 40, 0.05, 1.1, 64), (0.0, 1.0, 0, 0.0, 1.3, 8), (1.0, 0.9, 0, 0.0, 1.0, 0),
            (1.0, 1.0, 1, 0.0, 1.0, 0), (0.6, 0.9, 200, 0.02, 1.3, 64), (1.0, 1.0, 0, 0.0, 1.2, 16)]
GREEDY = [(0.0, 1.0, 0, 0.0, 1.0, 0), (0.0, 1.0, 0, 0.0, 1.5, 32)]


@pytest.mark.parametrize("settings", [SETTINGS, GREEDY], ids=["mixed", "greedy"])
@pytest.mark.parametrize("V", SIZES)
def test_unaligned_rows(oracle, V, settings):
    import quasar_amd as qa
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
        assert b.resolve_mode(base, stride, B, V) == qa.MODE_STREAM
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
