"""sm_reset empties a machine in one launch: every cached key, level and value, the words and the stream row read back
zero at odd sizes, the position and record restart, and the words after it are the first run's."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("streams,ctx,v64", [(1, 1 + 16, False), (1, 37, True), (3, 29, False), (5, 31, True)])
def test_reset(sm, small_dir, streams, ctx, v64):
    prompts = [sm.prompt_ids(40 + s, 9, 1000) for s in range(streams)]
    m = sm.Machine(small_dir, max_ctx=ctx, max_streams=streams, v64=v64)
    first = m.streams(prompts, 5)
    assert np.any(m.read("v", 11, streams - 1, 12)) and np.any(m.read("seq", stream=streams - 1))
    m.record_at(3)
    m.reset()
    for s in range(streams):
        for p in (0, 8, 12):
            for l in (0, 11):
                for name in ("k16", "ek", "v", "v64"):
                    assert not np.any(m.read(name, l, s, p)), (name, l, s, p)
        assert not np.any(m.read("seq", stream=s)) and not np.any(m.read("resid", stream=s))
    assert m.streams(prompts, 5) == first
    m.close()


def test_large(sm, small_npz, tmp_path):
    """64 streams of 500 positions (1.8 GB of caches): the last rows of the last stream read back zero, and emptying them
    takes no longer than filling as much memory does (a fifth more allowed; one grid-stride launch took a third more)"""
    import time

    import torch
    npz = dict(small_npz)
    npz["wpe"] = np.tile(npz["wpe"], (8, 1))
    m = sm.Machine(sm.layout(npz, str(tmp_path / "layout")), max_ctx=500, max_streams=64)
    prompts = [sm.prompt_ids(60 + s, 400, 1000) for s in range(64)]
    first = m.streams(prompts, 100)
    assert np.any(m.read("v", 11, 63, 498))
    m.reset()
    for p in (0, 399, 498, 499):
        for name in ("k16", "ek", "v", "v64"):
            assert not np.any(m.read(name, 11, 63, p)), (name, p)

    def best(f):
        t = []
        for _ in range(12):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            f()
            torch.cuda.synchronize()
            t.append(time.perf_counter() - t0)
        return min(t)
    buf = torch.empty(12 * 64 * 500 * 12 * 400 // 4, dtype=torch.int32, device="cuda")    # 400 bytes a cached row
    assert best(m.reset) < 1.2 * best(buf.zero_) + 20e-6
    assert m.streams(prompts, 100) == first
    m.close()
