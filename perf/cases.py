"""Timed cases of the integer machine: what a program that uses this package has it do, through its public entry
points (Machine, Plate, stages).

Whole calls (kind "machine"): a layout directory, a Machine made from it, then for every new prompt reset, prefill,
generate.  The last word is generated by a call of its own at a recorded position, so that its logits (stream 0's)
come back beside the words, and the last stream's row with them.  Sizes: one stream and many (up to 64), prompts of a
few words to nearly the whole context of 1024, one word (a prompt is scored) to the hundreds.

Single blocks: one row's plate product (GEMV), up to 64 rows' (int8 MFMA), one new position's attention (one block a
head, and spread over the GPU), the same for many streams, and base2.py's row stages over a batch of rows.

Everything is whole numbers, so every output is compared exactly.
"""
from __future__ import annotations

import collections
import importlib.util
import os
import sys
import tempfile

import numpy as np
import torch

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
VOCAB = {"gpt2": 50257, "pythia": 50304}
MAX_CTX = 1024
LAYERS = 12 * (768 * 2304 + 768 * 768 + 2 * 768 * 3072)        # digits of the twelve layers' plates


def _package():
    if "streaming_machine_amd" in sys.modules:
        return sys.modules["streaming_machine_amd"]
    root = os.path.join(REPO, "streaming-machine_amd")
    spec = importlib.util.spec_from_file_location("streaming_machine_amd", os.path.join(root, "__init__.py"),
                                                  submodule_search_locations=[root])
    mod = importlib.util.module_from_spec(spec)
    sys.modules["streaming_machine_amd"] = mod
    spec.loader.exec_module(mod)
    return mod


# ---------------------------------------------------------------------------------------------------------------
def listed():
    return [
        # a short answer for one user: 8 words in, 16 out (the batch-1 workload of bench.py)
        dict(name="gpt2 1 stream", kind="machine", model="gpt2", streams=1, prompt=8, words=16),
        # a long text scored: the prompt pass and one word's logits
        dict(name="gpt2 long prompt", kind="machine", model="gpt2", streams=1, prompt=1000, words=1),
        # one user's long document continued: decode at contexts where a step's attention runs spread over the GPU
        dict(name="gpt2 long context", kind="machine", model="gpt2", streams=1, prompt=345, words=67),
        # the other model, one user, a medium prompt
        dict(name="pythia 1 stream", kind="machine", model="pythia", streams=1, prompt=37, words=24),
        # serving: the largest batch (bench.py's 64-stream workload)
        dict(name="gpt2 64 streams", kind="machine", model="gpt2", streams=64, prompt=32, words=128),
        # serving, an odd batch whose time is in its prompts
        dict(name="gpt2 19 prompts", kind="machine", model="gpt2", streams=19, prompt=213, words=17),
        # serving the other model (bench.py's 32-stream workload)
        dict(name="pythia 32 streams", kind="machine", model="pythia", streams=32, prompt=64, words=256),
        # one light row through one bank: the smallest call of the operator API
        dict(name="plate one row", kind="plate", nin=768, nout=3072, rows=0),
        # the word table for a whole batch: every stream's piles
        dict(name="plate word table", kind="plate", nin=768, nout=50257, rows=64),
        # one new position's attention at an ordinary context, spread over the GPU
        dict(name="attend", kind="attend", rows=0, context=500, split=True),
        # the same for a batch of streams
        dict(name="attend rows", kind="attend", rows=48, context=331, split=False),
        # the row stages over a batch: gauge and to16 of the stream rows, the edge of the hidden rows, the race over
        # each row's logits
        dict(name="stages", kind="stages", rows=21, logits=50257),
    ]


def _log(rng, lo, hi):
    """a whole number in [lo, hi], spread over the logarithm"""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["machine", "machine", "machine", "plate", "attend", "stages"])
    if kind == "machine":
        model = rng.choice(["gpt2", "gpt2", "pythia"])
        streams = rng.choice([1, 1, _log(rng, 2, 64)])
        # at most 4096 positions of prompt and 2048 words over the streams, within the context
        prompt = _log(rng, 2, max(2, min(1000, 4096 // streams)))
        words = _log(rng, 1, max(1, min(128, MAX_CTX - prompt, 2048 // streams)))
        return dict(kind=kind, model=model, streams=streams, prompt=prompt, words=words)
    if kind == "plate":
        nin = rng.choice([768, 768, 3072])
        nout = _log(rng, 96, 50257) if nin == 768 else _log(rng, 96, 3072)
        return dict(kind=kind, nin=nin, nout=nout, rows=rng.choice([0, _log(rng, 1, 64), rng.randint(1, 64)]))
    if kind == "attend":
        rows = rng.choice([0, 0, _log(rng, 1, 64)])
        return dict(kind=kind, rows=rows, context=_log(rng, 2, MAX_CTX if rows <= 32 else MAX_CTX // 2),
                    split=rows == 0 and rng.random() < 0.5)
    return dict(kind="stages", rows=_log(rng, 1, 64), logits=_log(rng, 1000, 50304))


# ---------------------------------------------------------------------------------------------------------------
# what a program keeps: the layout directory, a few machines, the tables, a few plates
_machines = collections.OrderedDict()
_plates = collections.OrderedDict()
_tables = {}


def _keep(cache, key, make, most):
    if key not in cache:
        while len(cache) >= most:
            cache.popitem(last=False)
        cache[key] = make()
    cache.move_to_end(key)
    return cache[key]


def _layout(model):
    """the converted model's directory (random weights of the named shape), made once on this host"""
    sm = _package()
    path = os.path.join(tempfile.gettempdir(), f"sm_cases_{model}_{os.getuid()}")
    if not os.path.exists(os.path.join(path, "manifest.json")):
        part = tempfile.mkdtemp(prefix=f"sm_cases_{model}_", dir=tempfile.gettempdir())
        if model == "gpt2":
            sm.layout(sm.convert(sm.random_gpt2(seed=0)), part)
        else:
            sm.pythia.pythia_layout(sm.pythia.convert_pythia(*sm.pythia.random_pythia(seed=5)), part)
        try:
            os.rename(part, path)
        except OSError:                # another process was first
            path = part
    return path


def _machine(model, streams, ctx):
    sm = _package()
    return _keep(_machines, (model, streams, ctx),
                 lambda: sm.Machine(_layout(model), max_ctx=ctx, max_streams=streams), 3)


def _plate(nin, nout, tile):
    def make():
        rng = np.random.default_rng(nin * 100003 + nout)
        w = np.clip(np.round(rng.standard_normal((nin, nout), dtype=np.float32) * 9000.0), -32767, 32767).astype(np.int16)
        e = rng.integers(-16, -8, nout).astype(np.int32)
        b = rng.integers(-(1 << 16), 1 << 16, nout).astype(np.int64)
        return _package().Plate(w, e, b, tile_cols=tile), w
    return _keep(_plates, (nin, nout, tile), make, 4)


def _tabs():
    if not _tables:
        sm = _package()
        _tables["host"] = sm.tables()
        _tables["device"] = sm.Tables(_tables["host"])
    return _tables


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _gauss(gen, shape, scale):
    """gauged values: normal, at the machine's 2^-16"""
    return torch.round(torch.randn(shape, generator=gen, device="cuda", dtype=torch.float64) * scale).to(torch.int64)


def _keys(raw):
    """cached keys of raw rows (.., 64): their 16-bit lights (+32768 held as 32767), masks of the +32768, levels"""
    top = torch.frexp(raw.abs().amax(-1).double())[1].to(torch.int64)
    sh = (top - 15).clamp(min=0)
    half = torch.where(sh > 0, torch.ones_like(sh) << (sh - 1).clamp(min=0), torch.zeros_like(sh))
    x = (raw + half[..., None]) >> sh[..., None]
    bit = torch.ones(64, dtype=torch.int64, device=raw.device) << torch.arange(64, device=raw.device)
    return x, torch.where(x == 32768, bit, torch.zeros_like(bit)).sum(-1), (sh - 16).to(torch.int32)


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


# ---------------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    if kind == "machine":
        rng = np.random.default_rng(seed)
        prompts = [rng.integers(0, VOCAB[case["model"]], case["prompt"]).astype(np.int32) for _ in range(case["streams"])]
        m = _machine(case["model"], case["streams"], case["prompt"] + case["words"])
        return dict(case=case, m=m, prompts=prompts)
    gen = _gen(seed)
    if kind == "plate":
        nin, nout, rows = case["nin"], case["nout"], case["rows"]
        tile = 0 if rows else (1 if nin == 3072 else 4 if nout > 3072 else 2)     # the tiles the machine uses
        plate, _ = _plate(nin, nout, tile)
        # a row's largest light needs its whole 16 bits, as to16 leaves it
        x = _gauss(gen, (max(1, rows), nin), 9000.0).clamp(-32768, 32768)
        return dict(case=case, plate=plate, x=x, pile=torch.empty((max(1, rows), nout), dtype=torch.int64, device="cuda"))
    t = _tabs()["device"]
    if kind == "attend":
        r, p = max(1, case["rows"]), case["context"] - 1
        ctx = case["context"]
        k, km, ek = _keys(_gauss(gen, (r, 12, ctx, 64), 65536.0))
        v = _gauss(gen, (r, 12, ctx, 64), 65536.0).to(torch.int32)
        k16 = k.clamp(max=32767).to(torch.int16)
        for c in (k16, km, ek, v):
            c[:, :, p:] = 0                      # the new position's slot is empty
        return dict(case=case, t=t, qkv=_gauss(gen, (r, 2304), 65536.0), k16=k16, km=km, ek=ek, v=v,
                    out=torch.empty((r, 768), dtype=torch.int64, device="cuda"))
    r, n = case["rows"], case["logits"]
    e = lambda *s: torch.empty(s, dtype=torch.int64, device="cuda")      # noqa: E731
    return dict(case=case, t=t, R=_gauss(gen, (r, 768), 70000.0), h=_gauss(gen, (r, 3072), 90000.0),
                logits=_gauss(gen, (r, n), 200000.0), x16=e(r, 768), ex=e(r), LS=e(r), edged=e(r, 3072), hx16=e(r, 3072),
                hex=e(r), word=e(r))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "machine":
        m, n = state["m"], case["words"]
        m.reset()
        for b, ids in enumerate(state["prompts"]):
            m.prefill(ids, b)
        words = m.generate(n - 1) if n > 1 else None
        m.record_at(case["prompt"] + n - 2)                # the last word's step, for its logits
        last = m.generate(1)
        words = last if words is None else np.concatenate([words, last], axis=1)
        return dict(words=words, logits=m.read("logits"), row=m.read("resid", stream=case["streams"] - 1))
    st = _stream()
    if kind == "plate":
        if case["rows"]:
            state["plate"].product_rows(state["x"].data_ptr(), case["rows"], state["pile"].data_ptr(), stream=st)
        else:
            state["plate"].product(state["x"].data_ptr(), state["pile"].data_ptr(), stream=st)
        return state["pile"]
    s = _package().stages
    if kind == "attend":
        args = [state[k].data_ptr() for k in ("k16", "km", "ek", "v")] + [case["context"] - 1, case["context"],
                                                                          state["out"].data_ptr()]
        if case["rows"]:
            s.attend_rows(state["t"], state["qkv"].data_ptr(), case["rows"], *args, stream=st)
        else:
            (s.attend_split if case["split"] else s.attend)(state["t"], state["qkv"].data_ptr(), *args, stream=st)
        return [state[k] for k in ("out", "k16", "km", "ek", "v")]
    t, r = state["t"], case["rows"]
    ptr = lambda k: state[k].data_ptr()                    # noqa: E731
    s.gauge_log(t, ptr("R"), r, ptr("x16"), ptr("ex"), ptr("LS"), stream=st)
    s.edge(t, ptr("h"), ptr("edged"), r * 3072, stream=st)
    s.to16(ptr("edged"), r, 3072, ptr("hx16"), ptr("hex"), stream=st)
    for i in range(r):
        s.race(ptr("logits") + 8 * i * case["logits"], case["logits"], ptr("word") + 8 * i, stream=st)
    return [state[k] for k in ("x16", "ex", "LS", "edged", "hx16", "hex", "word")]


# ---------------------------------------------------------------------------------------------------------------
def work(case):
    """Bytes: int16 digits with their int32 exponent and int64 bias a column, k and v 4 bytes each; operations: two a
    multiply-add."""
    kind = case["kind"]
    if kind == "machine":
        v, b, p, n = VOCAB[case["model"]], case["streams"], case["prompt"], case["words"]
        layers = 2 * LAYERS + 12 * 12 * (2304 + 768 + 3072 + 768)
        head = 2 * 768 * v + 12 * v
        kv = 12 * 768 * 8                                  # one cached position of one stream
        steps = range(p, p + n)                            # the context of each word's step
        rows = b * (p - 1)
        bytes_ = (layers if p > 1 else 0) + 2 * rows * kv + n * (layers + head) + b * kv * (sum(steps) + n)
        att = 12 * 768 * 4                                 # a position attended by a row: q . k and a v
        flops = 2 * LAYERS * (rows + b * n) + 2 * 768 * v * b * n + att * b * (p * (p - 1) // 2 + sum(steps))
        return dict(bytes=bytes_, flops=flops)
    if kind == "plate":
        r = max(1, case["rows"])
        return dict(bytes=2 * case["nin"] * case["nout"] + 8 * r * (case["nin"] + case["nout"]),
                    flops=2 * r * case["nin"] * case["nout"])
    if kind == "attend":
        r, c = max(1, case["rows"]), case["context"]
        return dict(bytes=r * (12 * c * (64 * 6 + 12) + 8 * (2304 + 768)), flops=r * c * 768 * 4)
    r, n = case["rows"], case["logits"]
    return dict(bytes=8 * r * (768 * 2 + 3072 * 4 + n), flops=r * (768 * 8 + 3072 * 8 + n))


def tolerance(case):
    return "exact"


# ---------------------------------------------------------------------------------------------------------------
# base2.py's functions on int64 arrays
def _rsh(x, s):
    x, s = np.broadcast_arrays(np.asarray(x, np.int64), np.asarray(s, np.int64))
    right = (x + (np.int64(1) << np.maximum(s - 1, 0))) >> np.maximum(s, 0)
    return np.where(s > 0, right, x << np.maximum(-s, 0))


def _bits(v):
    return np.frexp(np.abs(v).astype(np.float64))[1].astype(np.int64)      # |v| below 2^53


def _to16(x):
    top = _bits(np.bitwise_or.reduce(np.abs(x), axis=-1))
    sh = np.maximum(top - 15, 0)
    return _rsh(x, sh[..., None]), sh - 16


def _log2fix(v, tab):
    t = _bits(v) - 1
    m = np.where(t >= 16, v >> np.maximum(t - 16, 0), v << np.maximum(16 - t, 0)) & 0xFFFF
    return t * 65536 + tab["log2"][m]


def _power(x, f, tab):
    return _rsh(x * tab["exp2"][f & 0xFFFF], 16 - (f >> 16))


def exact(case, seed):
    kind = case["kind"]
    if kind == "machine":
        return None                        # a model's conversion and its words in 64 bits: far over 20 seconds
    s = prepare(case, seed)
    tab = {k: np.asarray(v) for k, v in _table_formulas().items()}
    if kind == "plate":
        tile = 0 if case["rows"] else (1 if case["nin"] == 3072 else 4 if case["nout"] > 3072 else 2)
        w = torch.from_numpy(_plate(case["nin"], case["nout"], tile)[1]).double()
        return (s["x"].cpu().double() @ w).to(torch.int64)      # below 2^53: every partial sum is exact
    if kind == "attend":
        r, p = max(1, case["rows"]), case["context"] - 1
        qkv = s["qkv"].cpu().numpy().reshape(r, 3, 12, 64)
        q, eq = _to16(qkv[:, 0])
        kn, ekn = _to16(qkv[:, 1])
        km = s["km"].cpu().numpy()[..., None]
        k = s["k16"].cpu().numpy().astype(np.int64) + ((km >> np.arange(64)) & 1)
        ek, v = s["ek"].cpu().numpy().astype(np.int64), s["v"].cpu().numpy().astype(np.int64)
        k[:, :, p], ek[:, :, p], v[:, :, p] = kn, ekn, qkv[:, 2]
        sc = _rsh((q[:, :, None] * k).sum(-1), -(eq[:, :, None] + ek + 7))
        d = sc.max(-1, keepdims=True) - sc
        a = np.where(d < len(tab["arrival"]), tab["arrival"][np.minimum(d, len(tab["arrival"]) - 1)], 0)
        out = _power((a[..., None] * v).sum(2), -_log2fix(a.sum(-1), tab)[..., None], tab)
        return [torch.from_numpy(out.reshape(r, 768)), None, None, None, None]
    R, h, lg = (s[k].cpu().numpy() for k in ("R", "h", "logits"))
    x16, ex = _to16(R)
    s1, s2 = x16.sum(-1), (x16 * x16).sum(-1)
    V = 768 * s2 - s1 * s1 + (tab["eps40"] >> (40 + 2 * ex))
    LS = (_log2fix(V, tab) >> 1) - tab["log2_768"] + 65536 * ex
    i = _rsh(h, 4) + 32768
    edged = _rsh(h * np.where(i < 0, 0, np.where(i > 65535, 65536, tab["phi"][np.clip(i, 0, 65535)])), 16)
    hx16, hex_ = _to16(edged)
    return [torch.from_numpy(np.ascontiguousarray(v)) for v in (x16, ex, LS, edged, hx16, hex_, lg.argmax(-1))]


def _table_formulas():
    """the tables from their formulas (base2_convert.py:48-61)"""
    from math import erf, log2, exp
    i = np.arange(65536)
    arr = np.rint(np.exp(-np.arange(20000) / 1024.0) * (1 << 24)).astype(np.int64)
    return dict(phi=np.array([round(0.5 * (1 + erf((k - 32768) / 4096.0 / 2 ** 0.5)) * 65536) for k in range(65536)]),
                arrival=arr[:int(np.argmin(arr > 0))], log2=np.rint(np.log2(1 + i / 65536.0) * 65536).astype(np.int64),
                exp2=np.rint(2.0 ** (i / 65536.0) * 65536).astype(np.int64), log2_768=round(log2(768) * 65536),
                eps40=np.int64(round(1e-5 * 768 * 768 * 2 ** 40)))
