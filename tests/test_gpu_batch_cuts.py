"""Batches of very different sizes take different cuts of the same work (block
groups and haplotype parts of the subset cref kernel, row parts of the monos,
chain segments): the same targets give the same outputs alone, in a few and in
a batch that fills the device."""
import numpy as np
import pytest

import oracle
from eagleimp_amd import synth

from conftest import say
from parity import check_target, panel_engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K,M,T", [(300, 70, 400, 1020), (700, 513, 1500, 300)])
def test_alone_few_and_many(built, N, K, M, T):
    panel = synth.make_panel(61, N=N, M=M, F=20, T=T)
    tg = synth.make_targets(panel, 61, T, kset=[K, K - 9, 33], wmin=M // 2 + 1, wmax=M, miss=0.01)
    eng = panel_engine(panel, give_hap=True)
    pv = oracle.PanelView(panel.hap, panel.site, panel.cM)
    say("alone, few, many: N", N, "K", K, "T", T)
    many = eng.run_batch(tg.gt, tg.s0, tg.W, tg.K)
    last = eng.copy_target(T - 1, cref=True)
    check_target(oracle.process_target(pv, tg.gt[T - 1], tg.s0[T - 1], tg.W[T - 1], tg.K[T - 1]), last,
                 int(many.K[T - 1]), "gpu", "many", monos=eng.copy_monos(T - 1))
    for idx in ([0], [T - 1], list(range(0, T, T // 7))):
        r = eng.run_batch([tg.gt[i] for i in idx], tg.s0[idx], tg.W[idx], tg.K[idx])
        for f in ("S", "Mp", "ncalls", "K", "dig_pbwt", "dig_count0"):
            assert np.array_equal(getattr(r, f), getattr(many, f)[idx]), f"{idx}: {f}"
        i = idx[-1]
        check_target(oracle.process_target(pv, tg.gt[i], tg.s0[i], tg.W[i], tg.K[i]),
                     eng.copy_target(len(idx) - 1, cref=True), int(r.K[-1]), "gpu", f"{idx}",
                     monos=eng.copy_monos(len(idx) - 1))
    st = eng.stream(T, M, K, 1 << 30)
    st.submit(tg.gt, tg.s0, tg.W, tg.K)
    got, nd, _ = st.wait()
    assert nd == 0 and np.array_equal(got.dig_pbwt, many.dig_pbwt)
    st.submit(tg.gt[:1], tg.s0[:1], tg.W[:1], tg.K[:1])
    got, nd, _ = st.wait()
    assert nd == 0 and got.dig_pbwt[0] == many.dig_pbwt[0] and got.dig_count0[0] == many.dig_count0[0]
    st.close()
    eng.close()
