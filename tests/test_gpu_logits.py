"""GPU: the output layer alone, where every CU takes a run of columns (qs_logits.hip: past one
128-column tile a CU, from 256 embedding elements on) and in its tiles, against a float64
product within the bound of any fp32 summation order of exact bf16 products, E 2^-24 sum |h w|,
and bit for bit against the fused kernels' logits, which add in the same order."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,E,V", [
    (1, 64, 32772), (31, 64, 33000), (32, 128, 40960), (33, 192, 32800), (64, 512, 65536),
    (65, 64, 151936), (100, 320, 81920), (128, 128, 90004), (129, 64, 32772), (200, 192, 50000),
    (255, 256, 98304), (256, 64, 262144), (256, 512, 81924), (16, 2048, 60000),
    # the runs at the edges of their row shapes
    (1, 512, 32772), (31, 512, 33000), (32, 576, 40960), (33, 512, 32800), (64, 512, 90004),
    (65, 256, 151936), (100, 320, 40960), (128, 256, 90004), (129, 256, 32772), (200, 256, 50000),
    (256, 256, 262144)])
def test_logits_of_column_runs(rows, E, V):
    import quasar_amd as qa
    g = torch.Generator(device="cuda")
    g.manual_seed(rows * V)
    h = torch.randn((rows, E), generator=g, device="cuda").bfloat16()
    w = (torch.randn((V, E), generator=g, device="cuda") * 2.0 / E ** 0.5).bfloat16()
    packed = torch.empty(qa.head_packed_bytes(E, V), dtype=torch.uint8, device="cuda")
    guard = 64
    out = torch.full((rows * V + guard,), 7.0, device="cuda")
    fused = torch.empty((rows, V), device="cuda")
    torch.cuda.synchronize()
    b = qa.Batch(rows, V, 8)
    b.config(0, rows, 0.7, 0.95, 40, 0.05, 1.0, 0, seeds=np.arange(1, rows + 1))
    b.head_pack(w.data_ptr(), E, V, packed.data_ptr())
    for _ in range(2):
        b.head_logits(h.data_ptr(), packed.data_ptr(), E, rows, V, out.data_ptr())
    b.synchronize()
    assert (out[rows * V:] == 7.0).all()                    # nothing past the last row
    got = out[:rows * V].view(rows, V)
    b.pick_head(h.data_ptr(), packed.data_ptr(), E, rows, V, fused.data_ptr())
    assert torch.equal(got, fused)
    hd, wd = h.double(), w.double()
    want, mag = hd @ wd.t(), hd.abs() @ wd.abs().t()
    assert ((got.double() - want).abs() <= E * 2.0 ** -24 * mag + 1e-30).all()
    b.close()


@pytest.mark.parametrize("rows,E,V", [
    (3, 8128, 262144), (3, 8192, 262144), (70, 8192, 262144), (5, 12288, 256000)])
def test_logits_of_matrices_around_4_gib(rows, E, V):
    """Packed weights a tile row under 2^32 bytes, of 2^32 and of 6.3e9: every column against
    the fused kernels' logits bit for bit, and columns on both sides of the 2^32nd byte (and
    the first and the last) against a float64 product within the bound above."""
    import quasar_amd as qa
    g = torch.Generator(device="cuda")
    g.manual_seed(rows + E)
    h = torch.randn((rows, E), generator=g, device="cuda").bfloat16()
    w = torch.randn((V, E), generator=g, device="cuda", dtype=torch.bfloat16)
    packed = torch.empty(qa.head_packed_bytes(E, V), dtype=torch.uint8, device="cuda")
    got, fused = (torch.full((rows, V), 7.0, device="cuda") for _ in range(2))
    torch.cuda.synchronize()
    b = qa.Batch(rows, V, 8)
    b.config(0, rows, 0.7, 0.95, 40, 0.05, 1.0, 0, seeds=np.arange(1, rows + 1))
    b.head_pack(w.data_ptr(), E, V, packed.data_ptr())
    b.head_logits(h.data_ptr(), packed.data_ptr(), E, rows, V, got.data_ptr())
    b.synchronize()
    b.pick_head(h.data_ptr(), packed.data_ptr(), E, rows, V, fused.data_ptr())
    assert torch.equal(got, fused)
    at = min(2 ** 32 // (2 * E), V)
    cols = torch.tensor(sorted({c for m in (0, at, V) for c in range(max(0, m - 200), min(V, m + 200))}),
                        device="cuda")
    hd, wd = h.double(), w[cols].double()
    want, mag = hd @ wd.t(), hd.abs() @ wd.abs().t()
    assert ((got[:, cols].double() - want).abs() <= E * 2.0 ** -24 * mag).all()
    b.close()
