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


# 6 parts, 6 unaligned parts, 18 parts (past 16)
@pytest.mark.parametrize("V", [61440, 61433, 184320])
def test_part_bound_of_plus_zero_with_minus_zero_logits(oracle, V):
    """The highest part bound exactly +0.0 and -0.0 logits in that part: a -0.0 lies in the
    part's candidate list with the bound's own key, and is one candidate, not two."""
    import quasar_amd as qa
    r = np.random.default_rng(V)
    B, top_k, part = 8, 40, 10240
    parts = -(-(V + (3 if V % 4 else 0)) // part)
    m = (2 * -(-top_k // parts) + 8 + 15) // 16        # distinct lane maxima a wavefront offers
    x = r.normal(-9, 0.3, (B, V)).astype(np.float32)
    for i in range(B):
        sh = i * V % 4                                 # floats before the row in its 16 bytes
        for w in range(8):                             # float4 64 w + lane: wavefront w
            at = 256 * w - sh + 4
            for k in range(m - 1):
                x[i, at + 4 * k] = 0.5 + 0.01 * (8 * k + w)
            x[i, at + 40] = 0.0
            x[i, [at + 60, at + 81]] = -0.0
            for q in (1, 2):                           # the next bounds, about -2
                x[i, part * q + at:part * q + at + 12:4] = -2.0 + 0.1 * r.random(3)
    dev = qa.DeviceBuffer.from_array(x)
    cfgs = [(1.0, 1.0, top_k, 0.0, 1.0, 0), (1.0, 0.97, top_k, 0.0, 1.0, 0)]
    b = qa.Batch(B, V, 1)
    for i in range(B):
        b.config(i, 1, *cfgs[i % 2], seeds=[30 + i])
    got = [b.pick(dev.ptr, V, B, V, diag=True) for _ in range(6)]
    for i in range(B):
        s = oracle.sampler()
        s.config(*cfgs[i % 2], seed=30 + i)
        for k in range(6):
            want, od = s.pick_diag(x[i])
            d = got[k][1][i]
            assert int(got[k][0][i]) == want, (i, k, d.path, d.fallback)
            assert (d.keep, d.keep_topp, d.rank) == (od["keep"], od["keep_topp"], od["rank"]), (i, k)
            assert d.path == qa.PATH_CERT, (i, k, d.path, d.fallback)
        assert b.get_state(i)[0] == s.rng
    b.close()
    dev.free()
