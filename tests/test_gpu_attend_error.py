"""The attention entry points' error word (host memory that the kernels store to): each call reports its own value past
32 bits, whatever calls came before it or run beside it, at the first position, inside a chunk and in a later one."""
from __future__ import annotations

import threading

import pytest
import torch

pytestmark = pytest.mark.gpu

CTX = 256


def call(sm, t, fn, pos, bad, stream=0):
    rows = 3 if fn == "attend_rows" else 1
    z = lambda dt, *s: torch.zeros(s, dtype=dt, device="cuda")      # noqa: E731
    qkv = z(torch.int64, rows, 2304)
    qkv[rows - 1, 1536 + 700] = 2 ** 31 if bad else 2 ** 31 - 1
    c = (z(torch.int16, rows, 12, CTX, 64), z(torch.int64, rows, 12, CTX), z(torch.int32, rows, 12, CTX),
         z(torch.int32, rows, 12, CTX, 64))
    o = z(torch.int64, rows, 768)
    torch.cuda.synchronize()
    args = [qkv.data_ptr()] + ([rows] if rows > 1 else []) + [x.data_ptr() for x in c] + [pos, CTX, o.data_ptr()]
    try:
        getattr(sm.stages, fn)(t, *args, stream=stream)
    except sm.SmError as e:
        return e.code
    return 0


@pytest.mark.parametrize("fn", ["attend", "attend_split", "attend_rows"])
def test_each_call_its_own(sm, fn):
    t = sm.Tables(sm.tables())
    for pos in (0, 63, 64, 200):
        assert [call(sm, t, fn, pos, bad) for bad in (False, True, False, True, True, False)] == [0, -6, 0, -6, -6, 0]
    t.close()


def test_threads(sm):
    """two threads, each on its own stream, with the same tables; one of them always past 32 bits"""
    t = sm.Tables(sm.tables())
    got = {0: [], 1: []}

    def work(k):
        s = torch.cuda.Stream()
        for _ in range(300):
            got[k].append(call(sm, t, "attend", 5 + k, bool(k), s.cuda_stream))
    ths = [threading.Thread(target=work, args=(k,)) for k in (0, 1)]
    [x.start() for x in ths]
    [x.join() for x in ths]
    assert got == {0: [0] * 300, 1: [-6] * 300}
    t.close()


@pytest.mark.parametrize("fn", ["attend", "attend_split", "attend_rows"])
def test_threads_rows(sm, fn):
    """three threads, each on its own stream with its own caches at a position past several chunks, with the same
    tables: every call gives the row that the same call gives alone (attend_split's scratch belongs to the tables)"""
    t = sm.Tables(sm.tables())
    rows = 3 if fn == "attend_rows" else 1
    jobs = []
    for k in range(3):
        g = torch.Generator(device="cuda")
        g.manual_seed(70 + k)
        n = lambda *s: (torch.randn(s, generator=g, device="cuda", dtype=torch.float64) * 65536).round()      # noqa: E731
        pos = (130, 199, 255)[k]
        c = [n(rows, 12, CTX, 64).clamp(-32768, 32767).to(torch.int16), torch.zeros((rows, 12, CTX), dtype=torch.int64, device="cuda"),
             torch.full((rows, 12, CTX), -13, dtype=torch.int32, device="cuda"), n(rows, 12, CTX, 64).to(torch.int32)]
        qkv, o = n(rows, 2304).to(torch.int64), torch.zeros((rows, 768), dtype=torch.int64, device="cuda")
        args = [qkv.data_ptr()] + ([rows] if rows > 1 else []) + [x.data_ptr() for x in c] + [pos, CTX, o.data_ptr()]
        getattr(sm.stages, fn)(t, *args)
        torch.cuda.synchronize()
        jobs.append((args, o, o.clone(), (c, qkv), torch.cuda.Stream()))
    bad = []

    def work(k):
        args, o, want, _, s = jobs[k]
        for i in range(200):
            getattr(sm.stages, fn)(t, *args, stream=s.cuda_stream)
            with torch.cuda.stream(s):
                if not torch.equal(o, want):
                    bad.append((k, i))
                o.zero_()
    ths = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    [x.start() for x in ths]
    [x.join() for x in ths]
    assert not bad, bad[:4]
    assert any(int(w.abs().max()) > 0 for _, _, w, _, _ in jobs)
    t.close()


def test_calls_that_wait(sm):
    """300 calls, more than there are error words, wait behind long work on one stream, each in a thread of its own: the
    first hundred past 32 bits report that, the others nothing"""
    t = sm.Tables(sm.tables())
    z = lambda dt, *s: torch.zeros(s, dtype=dt, device="cuda")      # noqa: E731
    qs = [z(torch.int64, 2304) for _ in range(2)]
    qs[1][1536 + 700] = 2 ** 31
    c = (z(torch.int16, 12, CTX, 64), z(torch.int64, 12, CTX), z(torch.int32, 12, CTX), z(torch.int32, 12, CTX, 64))
    o = z(torch.int64, 768)
    torch.cuda.synchronize()
    spin = torch.cuda.Stream()
    with torch.cuda.stream(spin):
        torch.cuda._sleep(1_000_000_000)                   # (0.4 s; the calls' launches take a few milliseconds)
    got = [0] * 300

    def work(k):
        try:
            sm.stages.attend(t, qs[k < 100].data_ptr(), *[x.data_ptr() for x in c], 3, CTX, o.data_ptr(), stream=spin.cuda_stream)
        except sm.SmError as e:
            got[k] = e.code
    ths = [threading.Thread(target=work, args=(k,)) for k in range(300)]
    [x.start() for x in ths]
    [x.join() for x in ths]
    assert got == [-6] * 100 + [0] * 200
    t.close()
