"""Rows through a plate of many columns (Plate.product_rows, nin 768): exact piles at the column counts and row counts
where the kernel changes (16,000 columns up to 32 rows, 36,000 above), columns that end inside a tile and a block, rows
of +-32768 and rows without."""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nout", [15999, 16000, 16017, 35999, 36000, 36049, 50257])
def test_piles(sm, nout):
    rng = np.random.default_rng(nout)
    w = rng.integers(-32768, 32768, (768, nout)).astype(np.int16)
    plate = sm.Plate(w, np.zeros(nout, np.int32), np.zeros(nout, np.int64), tile_cols=0)
    wd = torch.from_numpy(w).cuda().double()
    for rows in (1, 15, 16, 17, 32, 33, 63, 64):
        x = rng.integers(-32768, 32769, (rows, 768))
        x[rows // 2] = 32768
        x[rows - 1, ::3] = -32768
        if rows > 2:
            x[0] = np.minimum(x[0], 32767)
        dx = torch.from_numpy(x).cuda()
        for call in (plate.product_rows, plate.product_rows_noalloc):
            pile = torch.full((rows, nout), -1, dtype=torch.int64, device="cuda")
            call(dx.data_ptr(), rows, pile.data_ptr())
            torch.cuda.synchronize()
            # float64 products: every partial sum below 2^40
            assert torch.equal(pile, (dx.double() @ wd).to(torch.int64)), (rows, call.__name__)
    plate.close()


@pytest.mark.parametrize("nout,rows,bank", [(49152, 1, True), (49153, 1, False), (51456, 1, False), (51457, 1, True), (49153, 2, True),
                                            (15999, 1, False), (16000, 1, True), (36000, 33, True), (35999, 33, False)])
def test_route(sm, nout, rows, bank):
    """which kernel a row count and width take, and its piles"""
    rng = np.random.default_rng(nout + rows)
    w = rng.integers(-32768, 32768, (768, nout)).astype(np.int16)
    plate = sm.Plate(w, np.zeros(nout, np.int32), np.zeros(nout, np.int64), tile_cols=0)
    dx = torch.from_numpy(rng.integers(-32768, 32769, (rows, 768))).cuda()
    pile = torch.full((rows, nout), -1, dtype=torch.int64, device="cuda")
    sm.machine.kernel_times()
    sm.machine.profile_stages(True)
    plate.product_rows(dx.data_ptr(), rows, pile.data_ptr())
    sm.machine.profile_stages(False)
    sym = sm.machine.kernel_times(symbols=True)["plate.head_rows"][2]
    assert ("k_pgemm" in sym) == bank, sym
    assert torch.equal(pile, (dx.double() @ torch.from_numpy(w).cuda().double()).to(torch.int64))
    plate.close()
