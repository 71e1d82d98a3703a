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
