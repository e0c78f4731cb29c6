"""The work a user of this library has it do, as cases that can be timed and checked.

Every case goes through a public entry point: the `sample.h` call (host logits in, id
out), the batched picks on logits already in device memory, the pick for callers that may
not allocate, the expert choice of a mixture-of-experts router, and the two output layers
followed by a pick.  `listed()` gives one case for each kind of use, `draw(rng)` further
ones over the same ranges.

A pick's outputs are whole numbers fixed bit for bit by the sampler's definition (ids,
generator states, histories), so they are compared exactly.
"""
import ctypes as C
import math

import numpy as np
import torch

import quasar_amd as qa
from quasar_amd import _native

VOCAB = 151936

# temperature, top_p, top_k, min_p, repeat_penalty, repeat_last_n
SERVER = dict(temperature=0.7, top_p=0.95, top_k=40, min_p=0.05, penalty=1.1, last_n=64)
GREEDY = dict(temperature=0.0, top_p=1.0, top_k=0, min_p=0.0, penalty=1.0, last_n=0)
OPEN = dict(temperature=1.0, top_p=1.0, top_k=0, min_p=0.0, penalty=1.0, last_n=0)


def listed():
    return [
        # `quasar serve`: one pick for each generated token, logits in host memory, the
        # request defaults.  The id is used at once.
        dict(name="host_pick", kind="host", rows=1, vocab=VOCAB, dist="normal", sigma=2.0,
             **SERVER),
        # A decode loop for one sequence under a runtime that may not allocate: logits, state
        # and ids stay on the device, on the program's own stream.
        dict(name="device_pick_1", kind="noalloc", rows=1, vocab=VOCAB, dist="normal",
             sigma=2.0, **dict(SERVER, top_p=0.9)),
        # A small server: 32 sequences with settings of their own (greedy ones among them),
        # the ids wanted on the host after each step.
        dict(name="server_32", kind="batch_sync", rows=32, vocab=VOCAB, dist="peaked",
             sigma=1.5, mixed=True, **SERVER),
        # The headline batch: a full sampler over 256 peaked rows, ids left on the device.
        dict(name="peaked_256", kind="batch", rows=256, vocab=VOCAB, dist="peaked", sigma=1.5,
             **dict(SERVER, temperature=0.8, last_n=256)),
        # Heavy-tailed rows with top-p alone.
        dict(name="studentt_1024", kind="batch", rows=1024, vocab=VOCAB, dist="student",
             sigma=2.0, **dict(OPEN, top_p=0.9)),
        # The largest batch: long histories, a wide top-k.
        dict(name="large_4096", kind="batch", rows=4096, vocab=VOCAB, dist="normal", sigma=2.0,
             **dict(SERVER, temperature=0.6, top_k=200, min_p=0.02, penalty=1.3, last_n=512)),
        # A vocabulary that is no multiple of four: rows start at any alignment.
        dict(name="odd_vocab_48", kind="batch_sync", rows=48, vocab=100003, dist="peaked",
             sigma=1.5, **SERVER),
        # Plain sampling at a temperature with every cut off, the default of many clients:
        # the draw is over the whole vocabulary.
        dict(name="open_8", kind="batch_sync", rows=8, vocab=VOCAB, dist="normal", sigma=2.0,
             **OPEN),
        # Nucleus sampling of flat rows: about 36,000 ids survive top-p 0.9.
        dict(name="nucleus_8", kind="batch_sync", rows=8, vocab=VOCAB, dist="normal",
             sigma=2.0, **dict(OPEN, top_p=0.9)),
        # One layer's expert choice for a prefill of 4,096 tokens.
        dict(name="router_4096", kind="router", tokens=4096, experts=128, used=8, norm=True),
        # The bf16 output layer of a large decode batch, then its pick.
        dict(name="head_256", kind="head", rows=256, embd=2048, vocab=VOCAB, **SERVER),
        # The output layer at the reference's arithmetic on a Q6_K matrix, then the pick.
        dict(name="head_exact_1", kind="head_exact", wtype="q6_k", rows=1, embd=2048,
             vocab=VOCAB, **SERVER),
    ]


# ---- drawn cases ---------------------------------------------------------------------------


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _vocab(rng, hi=262144):
    """A vocabulary that the aligned paths take: a multiple of four, half of them of 64."""
    v = _log(rng, 32000, hi)
    return v // 64 * 64 if rng.random() < 0.5 else v // 4 * 4


def _settings(rng):
    return dict(temperature=rng.choice([0.6, 0.7, 0.8, 1.0]), top_p=rng.choice([0.9, 0.95, 1.0]),
                top_k=rng.choice([1, 20, 40, 50, 100, 200]), min_p=rng.choice([0.0, 0.02, 0.05]),
                penalty=rng.choice([1.0, 1.1, 1.3]), last_n=_log(rng, 16, 512))


def draw(rng):
    kind = rng.choice(["host", "noalloc", "batch_sync", "batch", "batch", "odd", "open", "open",
                       "router", "head", "head_exact"])
    dist = rng.choice(["normal", "peaked"])
    sigma = 1.5 if dist == "peaked" else 2.0
    own = GREEDY if rng.random() < 0.2 else _settings(rng)
    if kind == "host":
        return dict(kind="host", rows=1, vocab=_log(rng, 32000, 262144), dist=dist, sigma=sigma,
                    **own)
    if kind == "noalloc":
        return dict(kind="noalloc", rows=_log(rng, 1, 64), vocab=_vocab(rng), dist=dist,
                    sigma=sigma, **own)
    if kind == "batch_sync":
        return dict(kind="batch_sync", rows=_log(rng, 2, 64), vocab=_vocab(rng), dist=dist,
                    sigma=sigma, mixed=rng.random() < 0.5, **own)
    if kind == "batch":
        if rng.random() < 0.25:
            dist, sigma, own = "student", 2.0, dict(OPEN, top_p=rng.choice([0.8, 0.9, 0.95]))
        vocab = _vocab(rng)
        return dict(kind="batch", rows=min(_log(rng, 64, 4096), 4096 * VOCAB // vocab),
                    vocab=vocab, dist=dist, sigma=sigma, **own)
    if kind == "odd":
        vocab = _log(rng, 32000, 262144) | rng.choice([1, 2, 3])
        return dict(kind="batch_sync", rows=_log(rng, 1, 256), vocab=vocab, dist=dist,
                    sigma=sigma, **own)
    if kind == "open":
        return dict(kind="batch_sync", rows=_log(rng, 1, 16), vocab=_vocab(rng, VOCAB),
                    dist="normal", sigma=rng.choice([1.0, 2.0]),
                    **dict(OPEN, temperature=rng.choice([0.7, 1.0]),
                           top_p=rng.choice([0.8, 0.9, 0.95, 1.0, 1.0]),
                           min_p=rng.choice([0.0, 0.0, 0.1])))
    if kind == "router":
        experts, used = rng.choice([(128, 8), (64, 4), (256, 64), (60, 4), (100, 7)])
        return dict(kind="router", tokens=_log(rng, 1, 16384), experts=experts, used=used,
                    norm=rng.random() < 0.5)
    if kind == "head":
        embd = 64 * rng.randint(8, 64)
        return dict(kind="head", rows=_log(rng, 1, 256), embd=embd,
                    vocab=min(_vocab(rng, VOCAB), 2048 * VOCAB // embd // 4 * 4), **SERVER)
    embd = 256 * rng.randint(2, 16)
    return dict(kind="head_exact", wtype=rng.choice(["q6_k", "q6_k", "q8_0", "f16", "f32"]),
                rows=min(_log(rng, 1, 8), 16384 // embd), embd=embd,
                vocab=min(_vocab(rng, VOCAB), 2048 * VOCAB // embd // 4 * 4), **SERVER)


# ---- inputs --------------------------------------------------------------------------------


def _gen(seed, device="cuda"):
    g = torch.Generator(device=device)
    g.manual_seed(int(seed))
    return g


def _logits(case, g):
    """Rows as the samplers meet them: flat, with one token far ahead, or heavy-tailed."""
    shape = (case["rows"], case["vocab"])
    x = torch.randn(shape, generator=g, device="cuda")
    if case["dist"] == "student":
        s = torch.zeros(shape, device="cuda")
        for _ in range(3):
            s += torch.randn(shape, generator=g, device="cuda").square_()
        x /= s.div_(3.0).sqrt_()
    x *= case["sigma"]
    if case["dist"] == "peaked":
        at = torch.randint(case["vocab"], (case["rows"], 1), generator=g, device="cuda")
        x.scatter_add_(1, at, torch.full_like(at, 12.0, dtype=torch.float32))
    return x


def _seeds(rows, seed):
    return np.random.default_rng(int(seed)).integers(1, 1 << 63, rows, dtype=np.uint64)


def _history(case, seed):
    r = np.random.default_rng(int(seed) + 1)
    return r.integers(0, case["vocab"], (case["rows"], case["last_n"]), dtype=np.int32)


def _row_settings(case):
    """(rows of a settings group, settings) for the batch."""
    own = {k: case[k] for k in ("temperature", "top_p", "top_k", "min_p", "penalty", "last_n")}
    if not case.get("mixed"):
        return [((0, case["rows"]), own)]
    kinds = [own, dict(GREEDY), dict(own, temperature=1.0, top_p=0.9, top_k=50, min_p=0.0),
             dict(own, temperature=0.6, top_k=20, penalty=1.0)]
    return [((r, 1), kinds[r % len(kinds)]) for r in range(case["rows"])]


def _batch(case, seed):
    """A configured batch with its rows' generators seeded and histories in place."""
    b = qa.Batch(case["rows"], case["vocab"], max(1, case["last_n"]))
    seeds = _seeds(case["rows"], seed)
    for (row, n), s in _row_settings(case):
        b.config(row, n, s["temperature"], s["top_p"], s["top_k"], s["min_p"], s["penalty"],
                 s["last_n"], seeds=seeds[row:row + n])
    if case["last_n"]:
        b.set_history(0, _history(case, seed))
    return b


class _Pick:
    """A batch as a program over the C interface holds it: its handle, the logits and the
    ids in device memory."""

    def __init__(self, batch, logits, vocab):
        self.batch, self.handle, self.logits, self.vocab = batch, batch._b, logits, vocab
        self.rows, self.stride = logits.shape[0], logits.stride(0)
        self.ids = torch.zeros(self.rows, dtype=torch.int32, device="cuda")
        self.lib = _native.load()

    def pick(self):
        rc = self.lib.qs_batch_pick(self.handle, self.logits.data_ptr(), self.stride, self.rows,
                                    self.vocab, self.ids.data_ptr(), None)
        _native.check(rc, "qs_batch_pick")
        return self.ids


class _NoAlloc:
    """The state of qs_pick_noalloc's rows in the program's own tensors."""

    def __init__(self, case, logits, seed):
        lib = self.lib = _native.load()
        rows, last = case["rows"], max(1, case["last_n"])
        cfg = C.create_string_buffer(32)
        lib.qs_row_config_set(C.addressof(cfg), case["temperature"], case["top_p"],
                              case["top_k"], case["min_p"], case["penalty"], case["last_n"])
        one = torch.frombuffer(bytearray(cfg.raw), dtype=torch.uint8)
        self.logits, self.rows, self.vocab, self.last = logits, rows, case["vocab"], last
        self.config = one.repeat(rows, 1).cuda()
        self.rng = torch.from_numpy(_seeds(rows, seed).view(np.int64)).cuda()
        ring = _history(case, seed) if case["last_n"] else np.zeros((rows, last), np.int32)
        self.ring = torch.from_numpy(ring).cuda()
        self.length = torch.full((rows,), case["last_n"], dtype=torch.int32, device="cuda")
        self.head = torch.zeros(rows, dtype=torch.int32, device="cuda")
        self.ids = torch.zeros(rows, dtype=torch.int32, device="cuda")

    def pick(self):
        rc = self.lib.qs_pick_noalloc(
            self.logits.data_ptr(), self.logits.stride(0), self.rows, self.vocab,
            self.config.data_ptr(), self.rng.data_ptr(), self.ring.data_ptr(), self.last,
            self.length.data_ptr(), self.head.data_ptr(), self.ids.data_ptr(),
            torch.cuda.current_stream().cuda_stream)
        _native.check(rc, "qs_pick_noalloc")
        return {"ids": self.ids, "rng": self.rng, "ring": self.ring, "length": self.length,
                "head": self.head}


class _Router:
    def __init__(self, case, g):
        self.case, self.lib = case, _native.load()
        n, e = case["tokens"], case["experts"]
        self.logits = torch.randn((n, e), generator=g, device="cuda") * 2.0
        self.idx = torch.zeros((n, case["used"]), dtype=torch.int32, device="cuda")
        self.wt = torch.zeros((n, case["used"]), device="cuda")

    def choose(self):
        c = self.case
        rc = self.lib.qs_router_topk(self.logits.data_ptr(), c["experts"], c["tokens"],
                                     c["experts"], c["used"], int(c["norm"]),
                                     self.idx.data_ptr(), self.wt.data_ptr(),
                                     torch.cuda.current_stream().cuda_stream)
        _native.check(rc, "qs_router_topk")
        return {"idx": self.idx, "wt": self.wt}


def _hidden(case, g):
    return torch.randn((case["rows"], case["embd"]), generator=g, device="cuda")


def _weight_bf16(case, g):
    w = torch.randn((case["vocab"], case["embd"]), generator=g, device="cuda",
                    dtype=torch.bfloat16)
    return w.mul_(2.0 / math.sqrt(case["embd"]))


WTYPES = {"f32": _native.WTYPE_F32, "f16": _native.WTYPE_F16, "q8_0": _native.WTYPE_Q8_0,
          "q6_k": _native.WTYPE_Q6_K}


def _weight_gguf(case, g):
    """The output matrix as a GGUF file stores it: uint8 [vocab][row bytes], its weights
    about 2 / sqrt(embd) wide."""
    v, e, t = case["vocab"], case["embd"], case["wtype"]
    width = 2.0 / math.sqrt(e)
    if t in ("f32", "f16"):
        w = torch.randn((v, e), generator=g, device="cuda") * width
        return (w if t == "f32" else w.half()).view(torch.uint8)
    block, size = (32, 34) if t == "q8_0" else (256, 210)
    n = v * (e // block)
    raw = torch.randint(0, 256, (n, size), generator=g, device="cuda", dtype=torch.uint8)
    d = 0.5 + torch.rand((n, 1), generator=g, device="cuda")
    if t == "q8_0":
        raw[:, :2] = (d * (width / 74.0)).half().view(torch.uint8)
    else:
        sc = torch.randint(-32, 32, (n, 16), generator=g, device="cuda", dtype=torch.int8)
        raw[:, 192:208] = sc.view(torch.uint8)
        raw[:, 208:] = (d * (width / 340.0)).half().view(torch.uint8)
    return raw.view(v, -1)


def _dequant64(case, raw):
    """_weight_gguf's bytes as float64 [vocab][embd]."""
    v, e, t = case["vocab"], case["embd"], case["wtype"]
    if t in ("f32", "f16"):
        return raw.view(torch.float32 if t == "f32" else torch.float16).double()
    if t == "q8_0":
        b = raw.view(-1, 34)
        d = b[:, :2].contiguous().view(torch.float16).double()
        return (d * b[:, 2:].contiguous().view(torch.int8).double()).view(v, e)
    b = raw.view(-1, 210)
    ql, qh = b[:, :128].view(-1, 2, 2, 32), b[:, 128:192].view(-1, 2, 32)
    sc = b[:, 192:208].contiguous().view(torch.int8).double().view(-1, 2, 4, 2, 1)
    d = b[:, 208:].contiguous().view(torch.float16).double().view(-1, 1, 1, 1, 1)
    q = torch.empty((b.shape[0], 2, 4, 32), dtype=torch.float64, device=b.device)
    for k in range(4):                       # 32 weights each: nibble k // 2 of half k % 2
        low = (ql[:, :, k % 2] >> (4 * (k // 2))) & 0xF
        q[:, :, k] = (low | (((qh >> (2 * k)) & 3) << 4)).double() - 32.0
    return (d * sc * q.view(-1, 2, 4, 2, 16)).view(v, e)


class _Head:
    """An output layer with its matrix laid out once, and the batch that picks from it."""

    def __init__(self, case, seed, g):
        self.case, self.lib = case, _native.load()
        self.batch = _batch(case, seed)
        rows, embd, vocab = case["rows"], case["embd"], case["vocab"]
        h = _hidden(case, g)
        if case["kind"] == "head":
            self.hidden, w = h.bfloat16(), _weight_bf16(case, g)
            n = qa.head_packed_bytes(embd, vocab)
        else:
            self.hidden, w = h, _weight_gguf(case, g)
            self.wtype = WTYPES[case["wtype"]]
            n = qa.head_exact_packed_bytes(self.wtype, embd, vocab)
        self.packed = torch.empty(n, dtype=torch.uint8, device="cuda")
        self.logits = torch.empty((rows, vocab), device="cuda")
        torch.cuda.synchronize()
        if case["kind"] == "head":
            self.batch.head_pack(w.data_ptr(), embd, vocab, self.packed.data_ptr())
        else:
            self.batch.head_exact_pack(self.wtype, w.data_ptr(), embd, vocab,
                                       self.packed.data_ptr())
        self.batch.synchronize()
        self.picker = _Pick(self.batch, self.logits, vocab)

    def step(self):
        c = self.case
        if c["kind"] == "head":
            self.batch.head_logits(self.hidden.data_ptr(), self.packed.data_ptr(), c["embd"],
                                   c["rows"], c["vocab"], self.logits.data_ptr())
        else:
            self.batch.head_exact_logits(self.wtype, self.packed.data_ptr(),
                                         self.hidden.data_ptr(), c["embd"], c["rows"],
                                         c["vocab"], self.logits.data_ptr())
        return {"logits": self.logits, "ids": self.picker.pick()}


class _Host:
    """sample.h: a sampler and one row of logits in host memory."""

    def __init__(self, case, logits, seed):
        self.logits = logits
        self.sampler = qa.Sampler()
        self.sampler.config(case["temperature"], case["top_p"], case["top_k"], case["min_p"],
                            case["penalty"], case["last_n"], seed=int(_seeds(1, seed)[0]))

    def pick(self):
        return self.sampler.pick(self.logits)


class _Sync:
    """A batch whose ids the program wants on the host after each step."""

    def __init__(self, batch, logits, vocab):
        self.batch, self.logits, self.vocab = batch, logits, vocab

    def pick(self):
        return self.batch.pick(self.logits.data_ptr(), self.logits.stride(0),
                               self.logits.shape[0], self.vocab)


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind == "router":
        s = _Router(case, g).choose
    elif kind in ("head", "head_exact"):
        s = _Head(case, seed, g).step
    else:
        x = _logits(case, g)
        if kind == "host":
            s = _Host(case, x[0].cpu().numpy(), seed).pick
        elif kind == "noalloc":
            s = _NoAlloc(case, x, seed).pick
        elif kind == "batch":
            s = _Pick(_batch(case, seed), x, case["vocab"]).pick
        else:
            s = _Sync(_batch(case, seed), x, case["vocab"]).pick
    torch.cuda.synchronize()
    return s


def run(state):
    return state()


# ---- what a pass cannot do without, and its results ----------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "router":
        n, e = case["tokens"], case["experts"]
        return {"bytes": n * (4 * e + 8 * case["used"]), "flops": n * e * 4}
    rows, vocab = case["rows"], case["vocab"]
    state = rows * (4 * case["last_n"] + 4 + 16)
    if kind not in ("head", "head_exact"):
        return {"bytes": 4 * rows * vocab + state, "flops": 4 * rows * vocab}
    embd = case["embd"]
    weight = {"head": 2.0, "f32": 4.0, "f16": 2.0, "q8_0": 34 / 32, "q6_k": 210 / 256}[
        "head" if kind == "head" else case["wtype"]]
    hidden = rows * embd * (2 if kind == "head" else 4)
    return {"bytes": weight * vocab * embd + hidden + 4 * rows * vocab + state,
            "flops": 2.0 * rows * vocab * embd}


def tolerance(case):
    if case["kind"] == "head":
        # fp32 sums of exact bf16 products, in any order; an id may move where two logits or
        # a cut lie within that rounding
        return {"rel": 1.5e-6, "max": 2e-5, "differ": 0.005}
    return "exact"


def exact(case, seed):
    g, kind = _gen(seed), case["kind"]
    if kind == "router":
        x = torch.randn((case["tokens"], case["experts"]), generator=g, device="cuda") * 2.0
        wt = torch.softmax(x.double(), 1).sort(dim=1, descending=True).values
        wt = wt[:, :case["used"]]
        return {"idx": None, "wt": wt / wt.sum(1, keepdim=True) if case["norm"] else wt}
    if kind == "head":
        h = _hidden(case, g).bfloat16().double()
        return {"logits": h @ _weight_bf16(case, g).double().t(), "ids": None}
    if kind == "head_exact":
        h = _hidden(case, g).double()
        return {"logits": h @ _dequant64(case, _weight_gguf(case, g)).t(), "ids": None}
    return None
