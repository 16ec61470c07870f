"""The selection's compaction takes 2,048 haplotypes per tile, 512 per wave and
64 per word: panel sizes and K on both sides of those edges, with distances so
coarse that most haplotypes tie at the threshold.  The distances take 32
haplotypes, 8 targets and 4,096 sites at a time: sizes, counts and windows on
both sides of those."""
import numpy as np
import pytest

import oracle
from eagleimp_amd import synth

from conftest import say
from parity import check_target, panel_engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [64, 130, 510, 514, 2046, 2048, 2050, 4094, 4098, 6148])
def test_selection_at_tile_edges(built, N):
    say("selection: N", N)
    panel = synth.make_panel(7, N=N, M=200, F=4, T=6)
    ks = [k for k in (33, 63, 64, 65, 511, 513, 2047, 2049, N - 2, N - 1) if k < N]
    tg = synth.make_targets(panel, 7, 6, kset=[ks[0]], wmin=60, wmax=200, miss=0.01)
    pv = oracle.PanelView(panel.hap, panel.site, panel.cM)
    eng = panel_engine(panel)
    idx = [i % 6 for i in range(len(ks))]
    r = eng.run_batch([tg.gt[i] for i in idx], tg.s0[idx], tg.W[idx],
                      np.asarray(ks, dtype=tg.K.dtype))
    for j, i in enumerate(idx):
        ref = oracle.process_target(pv, tg.gt[i], tg.s0[i], tg.W[i], ks[j])
        check_target(ref, eng.copy_target(j, cref=True), int(r.K[j]), "gpu", f"N {N} K {ks[j]}",
                     monos=eng.copy_monos(j))
    eng.close()


@pytest.mark.parametrize("N,M,T", [(34, 4095, 1), (62, 4097, 7), (66, 8192, 9), (258, 12350, 17)])
def test_distances_at_block_edges(built, N, M, T):
    say("distances: N", N, "M", M, "T", T)
    panel = synth.make_panel(8, N=N, M=M, F=8, T=T)
    tg = synth.make_targets(panel, 8, T, kset=[N // 2, N - 3, 33], wmin=30, wmax=M, miss=0.03)
    pv = oracle.PanelView(panel.hap, panel.site, panel.cM)
    eng = panel_engine(panel)
    r = eng.run_batch(tg.gt, tg.s0, tg.W, tg.K)
    for i in range(T):
        ref = oracle.process_target(pv, tg.gt[i], tg.s0[i], tg.W[i], tg.K[i])
        check_target(ref, eng.copy_target(i, cref=True), int(r.K[i]), "gpu", f"target {i}")
    eng.close()
