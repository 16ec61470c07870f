"""The PBWT's block path (order chain, run lists, rows per block) against the
oracle where it can go wrong: rows per direction at and around multiples of 16,
K at and around the chunk, shape and layout edges, and panels from few runs of
equal keys per block (all k_rows kernels) to as many runs as haplotypes (row by
row)."""
import numpy as np
import pytest

import oracle
from eagleimp_amd import synth

from conftest import say
from parity import check_target, panel_engine

pytestmark = pytest.mark.gpu


def _check(panel, tg, Ks, layout, what):
    kw = dict(compact=layout == "compact", raw=layout == "raw")
    say(what, layout, "K", sorted(set(int(k) for k in Ks)), "W", sorted(set(int(w) for w in tg.W))[:40])
    eng = panel_engine(panel, give_hap=True)
    res = eng.run_batch(tg.gt, tg.s0, tg.W, Ks, digest=True, **kw)
    pv = oracle.PanelView(panel.hap, panel.site, panel.cM)
    for t in range(len(tg.gt)):
        r = oracle.process_target(pv, tg.gt[t], tg.s0[t], tg.W[t], Ks[t])
        assert int(res.Mp[t]) == r["Mp"]
        check_target(r, eng.copy_target(t, cref=True), int(r["K"]), layout, f"{what} target {t}")
        assert int(res.dig_count0[t]) == r["dig_count0"], f"{what} target {t}: count0 digest"
        if layout != "raw":
            assert int(res.dig_pbwt[t]) == r["dig_pbwt"], f"{what} target {t}: digest"
    eng.close()
    return res


@pytest.mark.parametrize("layout", ["gpu", "compact", "raw"])
def test_row_counts_and_k_edges(built, layout):
    panel = synth.make_panel(51, N=2200, M=420, F=12, T=48)
    tg = synth.make_targets(panel, 51, 48, K=1, wmin=1, wmax=420, miss=0.02)
    Ks = np.array([1, 2, 31, 32, 33, 63, 64, 65, 127, 128, 129, 500, 511, 512, 513, 1025, 2047, 2048,
                   2049, 2200] * 3, np.uint32)[:48]
    res = _check(panel, tg, Ks, layout, "edges")
    assert len(set(int(m) % 16 for m in res.Mp)) >= 6  # odd row counts, several remainders


@pytest.mark.parametrize("flip", [0.0, 0.001, 0.006, 0.02, 0.5])
def test_few_to_many_runs(built, flip):
    panel = synth.make_panel(52, N=9000, M=150, F=40, T=3, flip_rate=flip)
    tg = synth.make_targets(panel, 52, 3, K=1, wmin=120, wmax=150, miss=0.01)
    _check(panel, tg, np.array([9000, 8191, 4097], np.uint32), "gpu", f"flip {flip}")


@pytest.mark.parametrize("N,n", [(64, 1), (130, 15), (130, 16), (130, 17), (2049, 33), (6000, 48)])
def test_panel_pbwt_blocks(built, N, n):
    panel = synth.make_panel(53, N=N, M=64, F=20, T=1, flip_rate=0.01)
    say("panel PBWT blocks", N, n)
    eng = panel_engine(panel)
    for absperm in (True, False):
        rows, c0, ap, _ = eng.ref_pbwt(3, n, absperm=absperm)
        want = oracle.build_ref_pbwt(np.ascontiguousarray(panel.site[3:3 + n]), N)
        assert np.array_equal(rows, want[0]) and np.array_equal(c0, want[1])
        if absperm:
            assert np.array_equal(ap, want[2])
    eng.close()


@pytest.mark.parametrize("N,F,flip,K", [(300, 3, 0.0, 300), (300, 3, 0.0, 77), (1500, 40, 0.001, 1300),
                                        (2200, 30, 0.0, 2112)])
def test_cut_chains(built, N, F, flip, K):
    """Few long chains are cut into segments: haplotypes that a segment does
    not tell apart (without flips whole classes are equal), padded and full K,
    the synchronous call, a stream context and the panel's chain."""
    M = 5000
    panel = synth.make_panel(54, N=N, M=M, F=F, T=2, flip_rate=flip)
    tg = synth.make_targets(panel, 54, 2, K=K, wmin=M - 300, wmax=M, miss=0.01)
    res = _check(panel, tg, tg.K, "compact", f"cut N {N} F {F}")
    eng = panel_engine(panel, give_hap=True)
    st = eng.stream(2, M, K, 256 << 20)
    st.submit(tg.gt, tg.s0, tg.W, tg.K)
    got, nd, _ = st.wait()
    assert nd == 0 and np.array_equal(got.dig_pbwt, res.dig_pbwt)
    assert np.array_equal(got.dig_count0, res.dig_count0)
    st.close()
    rows, c0, ap, _ = eng.ref_pbwt(7, M - 40)
    want = oracle.build_ref_pbwt(np.ascontiguousarray(panel.site[7:7 + M - 40]), N)
    assert np.array_equal(rows, want[0]) and np.array_equal(c0, want[1]) and np.array_equal(ap, want[2])
    eng.close()
