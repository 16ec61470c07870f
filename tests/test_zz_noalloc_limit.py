"""The largest batches that eimp_engine_run_batch_noalloc's scratch takes: a
whole-panel target of 64 haplotypes whose condensed reference, split data and one
16-byte work item per block come to 63.5 of 64 MiB."""
from types import SimpleNamespace

import numpy as np
import pytest

from eagleimp_amd.engine import row_stride, unit_words

from conftest import say
from parity import panel_engine
from test_zz_no_alloc import DevMem

pytestmark = pytest.mark.gpu


def test_largest_batch_of_the_scratch(built):
    N, W = 64, 2_549_987
    rng = np.random.default_rng(81)
    site = np.zeros((W, 8), np.uint64)
    site[:, 0] = rng.integers(1, 2**64 - 1, W, dtype=np.uint64)  # no site is the same in all
    panel = SimpleNamespace(N=N, M=W, site=site, hap=None, cM=(1e-4 * np.arange(W)).astype(np.float32))
    eng = panel_engine(panel)
    mem = DevMem()
    say("no-allocation scratch, sites", W)
    try:
        gt = np.zeros(2 * unit_words(W), np.uint64)  # all heterozygous: every site is a split
        ref = eng.run_batch([gt], [0], [W], [N], digest=True, compact=True)
        Mp = 2 * W + 1
        assert int(ref.Mp[0]) == Mp
        rows, c0 = mem.alloc(2 * Mp * row_stride(N, "compact") * 4), mem.alloc(Mp * 4)
        got = eng.run_batch_noalloc([mem.upload(gt)], [0], [W], [N], Mp, [rows], [c0], digest=True,
                                    compact=True)
        for f in ("S", "Mp", "ncalls", "K", "dig_pbwt", "dig_count0"):
            assert np.array_equal(getattr(got, f), getattr(ref, f)), f
    finally:
        mem.close()
        eng.close()
