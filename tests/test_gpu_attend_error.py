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
