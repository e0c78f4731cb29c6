"""GPU: rows whose streaming candidates lie above a part bound too high for their top-k (one
large logit in each wavefront's share of the first part), so that part is read again
(widen, qs_part.hip), against the CPU restatement: ids, kept prefixes, generator states and
histories, compared exactly; and most of them decided without the exact path."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# two parts, unaligned, 15 parts (one wavefront's lists), 18 and 26 parts (past 16)
@pytest.mark.parametrize("V", [20480, 30001, 151936, 180000, 262144])
@pytest.mark.parametrize("top_k", [40, 64, 200])
def test_rows_with_one_high_part_bound(oracle, V, top_k):
    import quasar_amd as qa
    r = np.random.default_rng(V + top_k)
    B = 8
    x = r.normal(0, 1, (B, V)).astype(np.float32)
    for w in range(8):                                 # float4 64 w: wavefront w of the part
        x[:, 256 * w] = 7.0 + 0.125 * w + r.random(B) * 0.01
    x[6] = np.round(x[6] * 4) / 4                      # ties across the bounds
    x[7, 10:V:3] = -np.inf
    dev = qa.DeviceBuffer.from_array(x)
    cfgs = [(1.0, 1.0, top_k, 0.0, 1.0, 0), (1.5, 0.999, top_k, 0.0, 1.1, 32),
            (1.0, 0.9999, top_k, 1e-4, 1.0, 0), (2.0, 0.95, top_k, 0.01, 1.2, 16)]
    b = qa.Batch(B, V, 32)
    b.set_mode(qa.MODE_AUTO if V % 4 else qa.MODE_STREAM)
    hist = r.integers(0, V, (B, 20)).astype(np.int32)
    for i in range(B):
        b.config(i, 1, *cfgs[i % 4], seeds=[90 + i])
    b.set_history(0, hist)
    got = [b.pick(dev.ptr, V, B, V, diag=True) for _ in range(3)]
    paths = []
    for i in range(B):
        s = oracle.sampler()
        s.config(*cfgs[i % 4], seed=90 + i)
        s.set_history(hist[i])
        for k in range(3):
            want, od = s.pick_diag(x[i])
            d = got[k][1][i]
            assert int(got[k][0][i]) == want, (i, k, d.path, d.fallback)
            assert d.keep == od["keep"] and d.keep_topp == od["keep_topp"], (i, k, d.path)
            paths.append(d.path)
        rng, h = b.get_state(i)
        assert rng == s.rng and (h == s.history()).all(), i
    print(V, top_k, "certified", paths.count(qa.PATH_CERT), "of", len(paths), flush=True)
    if top_k <= 64:
        assert paths.count(qa.PATH_CERT) >= len(paths) // 2
    b.close()
    dev.free()
