"""GPU: rows without a top-k whose kept prefix may be the whole window (qs_open.h), against
the CPU restatement (sample.c:111-179) on the same logits: ids, the kept prefixes, the
drawn position, the softmax normaliser, generator states and histories.  All whole numbers
(inv: a float fixed by the definition), so compared exactly.  And the batch's count of rows
decided by selection: every whole-window row of ordinary values (flat, heavy-tailed) is one,
so the sort serves none of them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# vocabularies at the part's edges (4,096 logits) and over the real range
SIZES = [4, 60, 4092, 4096, 4100, 40960, 151936, 262144]
ORDINARY = (0, 1, 4)                   # rows_of's rows of values that seldom repeat
# (temperature, top_p, top_k, min_p, penalty, last_n)
SETTINGS = [
    (1.0, 1.0, 0, 0.0, 1.0, 0), (0.7, 0.9, 0, 0.0, 1.0, 0), (1.0, 0.8, 0, 0.1, 1.2, 64),
    (1.0, 1.0, 0, 0.1, 1.0, 0), (1.3, 0.9999999, 0, 0.0, 1.0, 0), (1.0, 0.95, 1 << 30, 0.0, 1.3, 16),
    (0.05, 1.0, 0, 1e-6, 1.0, 0), (1.0, 1.0, 0, 2.0, 1.0, 0),
]


def rows_of(V, seed):
    """Flat, wide, narrow, peaked and heavy-tailed rows, rows on a bf16 grid, one value only,
    and rows with infinities and NaN."""
    r = np.random.default_rng(seed)
    x = r.normal(0, 2, (10, V)).astype(np.float32)
    x[1] = r.normal(0, 1, V)
    x[2] = r.normal(0, 0.01, V)
    x[3, r.integers(V)] += 12
    x[4] = r.standard_t(3, V) * 2
    bf = (r.normal(0, 2, V).astype(np.float32).view(np.uint32) + 0x8000) & 0xFFFF0000
    x[5] = bf.astype(np.uint32).view(np.float32)
    x[6] = 0.25
    x[7, ::3] = -np.inf
    x[8, V // 2] = np.nan
    x[9] = np.round(x[9])
    return x


@pytest.mark.parametrize("V", SIZES)
def test_open_rows(oracle, V):
    import quasar_amd as qa
    x = rows_of(V, V)
    B = len(SETTINGS) * len(x)
    n = min(B, 64)
    full = np.concatenate([x] * len(SETTINGS))
    for first in range(0, B, n):
        m = min(n, B - first)
        b = qa.Batch(n, V, 64)
        buf = qa.DeviceBuffer.from_array(full[first:first + m])
        b.set_mode(2)
        hist = np.random.default_rng(V + first).integers(0, V, (m, 24)).astype(np.int32)
        for r in range(m):
            b.config(r, 1, *SETTINGS[(first + r) // len(x)], seeds=[1000 + first + r])
        b.set_history(0, hist)
        got = [b.pick(buf.ptr, V, m, V, diag=True) for _ in range(2)]
        selected = b.selected_rows()
        paths, whole, ordinary = {}, 0, 0
        for r in range(m):
            s = oracle.sampler()
            cfg = SETTINGS[(first + r) // len(x)]
            s.config(*cfg, seed=1000 + first + r)
            s.set_history(hist[r])
            for k in range(2):
                want, od = s.pick_diag(full[first + r])
                ids, d = got[k][0], got[k][1][r]
                at = (V, cfg, r % len(x), k, d.path, d.fallback)
                assert int(ids[r]) == want, at
                assert d.keep == od["keep"], at
                if d.path == qa.PATH_FULL:
                    whole += 1
                    ordinary += (first + r) % len(x) in ORDINARY
                    assert np.float32(d.inv) == np.float32(od["inv"]) or np.isnan(od["inv"]), at
                    assert (d.keep_topp, d.n_window, d.rank) == \
                        (od["keep_topp"], od["n_window"], od["rank"]), at
                paths[d.path] = paths.get(d.path, 0) + 1
            rng, h = b.get_state(r)
            assert rng == s.rng and (h == s.history()).all(), at
        print(V, first, "paths", paths, "selected", selected, "ordinary", ordinary, flush=True)
        assert ordinary <= selected <= whole
        b.close()
        buf.free()


@pytest.mark.parametrize("V", [4092, 40963, 151936])
def test_open_rows_summed_in_id_order(oracle, V):
    """The same rows with the denominator always taken in id order (as where the parts' sum
    leaves inv open): the row's last part does every part's share, and the sum is the
    restatement's bit for bit."""
    import quasar_amd as qa
    x = rows_of(V, V + 1)[[0, 1, 4, 5]]
    B = len(x)
    dev = qa.DeviceBuffer.from_array(x)
    for cfg in SETTINGS[:4]:
        b = qa.Batch(B, V, 64)
        b.set_sum_in_order(1)
        b.config(0, B, *cfg, seeds=np.arange(7, 7 + B))
        got = [b.pick(dev.ptr, V, B, V, diag=True) for _ in range(2)]
        ordinary = sum(got[k][1][r].path == qa.PATH_FULL for k in range(2) for r in range(3))
        assert b.selected_rows() >= ordinary, cfg
        for r in range(B):
            s = oracle.sampler()
            s.config(*cfg, seed=7 + r)
            for k in range(2):
                want, od = s.pick_diag(x[r])
                d = got[k][1][r]
                assert int(got[k][0][r]) == want, (cfg, r, k, d.path)
                assert d.keep == od["keep"], (cfg, r, k)
                if d.path == qa.PATH_FULL:
                    assert d.sum == od["sum"] and d.rank == od["rank"], (cfg, r, k)
            assert b.get_state(r)[0] == s.rng
        b.close()
    dev.free()


@pytest.mark.parametrize("B", [32, 60])
def test_certified_rows_without_a_top_k_pay_empty_launches_only(B):
    """Peaked rows without a top-k, decided with a proof: with the whole-window launches behind
    the decision (which leave at once) a pick takes at most 1.25 times what it takes without (a
    spin limit of 0, which such rows do not need; 1.17 and 1.14 measured).  A first pass beside
    every decision made it 1.4 times at 32 rows and 1.9 at 60."""
    import quasar_amd as qa
    V = 151936
    r = np.random.default_rng(B)
    x = r.normal(0, 1.5, (B, V)).astype(np.float32)
    x[np.arange(B), r.integers(0, V, B)] += 12
    dev = qa.DeviceBuffer.from_array(x)
    b = qa.Batch(B, V, 8)
    b.config(0, B, 0.7, 1.0, 0, 0.05, 1.0, 0, seeds=np.arange(1, B + 1))
    assert all(d.path == qa.PATH_CERT for d in b.pick(dev.ptr, V, B, V, diag=True)[1])
    us = {}
    for limit in (0, 1 << 20) * 4:
        b.set_spin_limit(limit)
        t = b.time_picks(dev.ptr, V, B, V, 100)
        us[limit] = min(us.get(limit, 1e9), 10.0 * t)
    b.synchronize()
    print(B, us, flush=True)
    assert us[1 << 20] <= 1.25 * us[0]
    b.close()
    dev.free()


def test_scratch_is_cleared_after_a_failed_launch():
    """The whole-window launch failing after the first pass has filled its histograms, then a
    pick that does not use them, then whole-window rows of other logits: decided by selection,
    as no pick on the failed one's histograms would be."""
    import quasar_amd as qa
    V, B = 40960, 8
    r = np.random.default_rng(8)
    wide = qa.DeviceBuffer.from_array((r.normal(0, 1, (B, V)) * 6).astype(np.float32))
    flat = qa.DeviceBuffer.from_array(r.normal(0, 1, (B, V)).astype(np.float32))
    b = qa.Batch(B, V, 8)
    open_rows = dict(temperature=1.0, top_p=0.9, top_k=0, seeds=np.arange(1, B + 1))
    b.config(0, B, **open_rows)
    want = b.pick(flat.ptr, V, B, V)
    assert b.selected_rows() == B
    b.config(0, B, temperature=3.0, top_p=0.9, top_k=0, seeds=np.arange(1, B + 1))
    qa.check(qa.load().qs_debug_fail_open_launches(1), "qs_debug_fail_open_launches")
    with pytest.raises(qa.QsError) as e:
        b.pick(wide.ptr, V, B, V)
    assert e.value.rc == qa._native.QS_EDEVICE
    b.config(0, B, temperature=1.0, top_k=5, seeds=np.arange(1, B + 1))
    b.pick(flat.ptr, V, B, V)
    b.config(0, B, **open_rows)
    assert (b.pick(flat.ptr, V, B, V) == want).all()
    assert b.selected_rows() == 2 * B
    b.close()
    wide.free()
    flat.free()
