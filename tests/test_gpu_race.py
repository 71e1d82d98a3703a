"""sm_stage_race over one block (up to 1,024 values, and with the index written over the values) and many: the largest
value, ties to the lowest index (base2.py:34-40), at the sizes where the block count and width change, on values that tie
across blocks, that are all the type's lowest, and with the index written over the values."""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def race(sm, v, out=None, stream=0):
    d = torch.from_numpy(v).cuda()
    o = torch.full((1,), 77, dtype=torch.int64, device="cuda")
    ptr = o.data_ptr() if out is None else d.data_ptr() + 8 * out
    sm.stages.race(d.data_ptr(), len(v), ptr, stream=stream)
    torch.cuda.synchronize()
    return int(o[0]) if out is None else int(d[out])


@pytest.mark.parametrize("n", [1, 63, 64, 1000, 1023, 1024, 1025, 1026, 2047, 2048, 2049, 4097])
def test_few(sm, n):
    """fewer values than a block has threads, one, and values on both sides of a trip and of a block's share"""
    rng = np.random.default_rng(n)
    v = rng.integers(-2 ** 62, 2 ** 62, n)
    assert race(sm, v) == int(v.argmax())
    assert race(sm, np.full(n, np.iinfo(np.int64).min)) == 0
    assert race(sm, v, out=n - 1) == int(v.argmax())


def test_route(sm):
    """one launch each: of one block up to 1,024 values and, where the index is written over them, at any count, a value a
    trip up to 12,288; else of many"""
    d = torch.zeros(140000, dtype=torch.int64, device="cuda")
    o = torch.zeros(1, dtype=torch.int64, device="cuda")
    one, eight = "k_stage_race<0, 1024, 1>", "k_stage_race<0, 1024, 8>"
    for n, out, want in ((1, o, one), (1024, o, one), (1025, o, "k_stage_race<1, 256, 8>"), (131072, o, "k_stage_race<1, 256, 8>"),
                         (131073, o, "k_stage_race<1, 512, 8>"), (12288, d, one), (12289, d, eight), (131073, d, eight)):
        sm.machine.kernel_times()
        sm.machine.profile_stages(True)
        sm.stages.race(d.data_ptr(), n, out.data_ptr())
        sm.machine.profile_stages(False)
        got = {k: v for k, v in sm.machine.kernel_times(symbols=True).items() if v[0]}
        assert list(got) == ["stage.race"] and got["stage.race"][0] == 1 and want in got["stage.race"][2], (n, got)


@pytest.mark.parametrize("n", [12288, 12289, 18432, 8192, 8193, 16384, 16385, 18431, 18433, 131072, 131073, 1048577, 2100001])
def test_many_blocks(sm, n):
    rng = np.random.default_rng(n)
    v = rng.integers(-2 ** 62, 2 ** 62, n)
    assert race(sm, v) == int(v.argmax())
    v[[n - 1, n // 2, n // 3, 2000]] = 2 ** 62 + 1             # the same best in several blocks
    assert race(sm, v) == 2000
    v[0] = v[n - 1] = np.iinfo(np.int64).max
    assert race(sm, v) == 0
    assert race(sm, np.full(n, np.iinfo(np.int64).min)) == 0
    low = np.full(n, np.iinfo(np.int64).min)
    low[n - 1] += 1
    assert race(sm, low) == n - 1
    assert race(sm, v, out=n // 2) == 0                        # the index over a value: written after it is read


@pytest.mark.parametrize("n", [1025, 2049, 18433, 50257, 1048577])
def test_word_before(sm, n):
    """the output word before the call: a losing index, the winner, a tied higher index, the value count, -1, the type's ends"""
    rng = np.random.default_rng(n + 1)
    v = rng.integers(-2 ** 40, 2 ** 40, n)
    v[[n // 3, n // 2, n - 1]] = 2 ** 41
    d = torch.from_numpy(v).cuda()
    for before in (0, int(v.argmin()), n // 3, n // 2, n - 1, n, -1, 2 ** 62, -2 ** 63):
        o = torch.full((1,), before, dtype=torch.int64, device="cuda")
        for _ in range(3):
            sm.stages.race(d.data_ptr(), n, o.data_ptr())
            torch.cuda.synchronize()
            assert int(o[0]) == n // 3, before


def test_two_streams(sm):
    """races on two streams at once, each with its own winner"""
    rng = np.random.default_rng(5)
    vs = [rng.integers(-2 ** 40, 2 ** 40, 50257) for _ in range(2)]
    ds = [torch.from_numpy(v).cuda() for v in vs]
    outs = torch.zeros(2, 50, dtype=torch.int64, device="cuda")
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    for i in range(50):
        for k, s in enumerate(streams):
            sm.stages.race(ds[k].data_ptr(), 50257, outs[k, i:].data_ptr(), stream=s.cuda_stream)
    torch.cuda.synchronize()
    for k in range(2):
        assert (outs[k] == int(vs[k].argmax())).all()


def test_shared_word(sm):
    """races of a long and a short row on two streams into one word: neither reads its own row at the other's index,
    and a race after both has its own winner"""
    rng = np.random.default_rng(6)
    vs = [torch.from_numpy(rng.integers(-2 ** 40, 2 ** 40, n)).cuda() for n in (1048577, 18433)]
    vs[0][1048576] = 2 ** 41
    out = torch.zeros(1, dtype=torch.int64, device="cuda")
    streams = [torch.cuda.Stream() for _ in range(2)]
    torch.cuda.synchronize()
    for _ in range(100):
        for v, s in zip(vs, streams):
            sm.stages.race(v.data_ptr(), len(v), out.data_ptr(), stream=s.cuda_stream)
    torch.cuda.synchronize()
    assert 0 <= int(out[0]) < 1048577
    sm.stages.race(vs[1].data_ptr(), len(vs[1]), out.data_ptr())
    torch.cuda.synchronize()
    assert int(out[0]) == int(vs[1].argmax())
