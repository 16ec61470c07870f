"""The PBWT's block path by what a block takes: every size of k_rows (entries per
lane) in both directions, blocks row by row, and cut chains in every shape.  What
the cases reach is worked out from the oracle's condensed reference and the
constants in the sources, without a device."""
import os
import re

import numpy as np
import pytest

import oracle
from eagleimp_amd import synth

from conftest import ROOT, say
from parity import check_target, panel_engine
from test_engine_host import host  # noqa: F401 (fixture)

KS = [64, 200, 400, 600, 900, 1200, 1500, 1800, 2100, 2400, 2700, 3000, 3400, 3800, 4200, 4700, 5200, 5700,
      6200, 6700, 7200, 7800, 8400, 9000]
PANELS = [700, 2500]  # founders: few and many runs of equal keys
M = 330


def case(founders):
    panel = synth.make_panel(61, N=9000, M=M, F=founders, T=len(KS), flip_rate=0.004)
    tg = synth.make_targets(panel, 61, len(KS), K=1, wmin=M - 10, wmax=M, miss=0.01)
    pv = oracle.PanelView(panel.hap, panel.site, panel.cM)
    return panel, tg, [oracle.process_target(pv, tg.gt[t], tg.s0[t], tg.W[t], K) for t, K in enumerate(KS)]


def block_runs(cref, K, rev):
    """(runs of equal keys, rows) of each block in processing order."""
    bits = np.unpackbits(cref.view(np.uint8), axis=1, bitorder="little")[:, :K].astype(np.int64)
    kpad, nblk, out = (K + 63) // 64 * 64, (len(bits) + 15) // 16, []
    order = np.arange(kpad)
    for q in range(nblk):
        b = nblk - 1 - q if rev else q
        rows = bits[16 * b:16 * b + 16][::-1 if rev else 1]
        key = np.full(kpad, (1 << len(rows)) - 1)
        key[:K] = (rows << np.arange(len(rows))[:, None]).sum(0)
        k = key[order]
        out.append((1 + int((k[1:] != k[:-1]).sum()), len(rows)))
        order = order[np.argsort(k, kind="stable")]
    return out


def source(name):
    with open(os.path.join(ROOT, "eagleimp_amd", "csrc", name)) as f:
        return f.read()


def test_cases_reach_every_block_size(built):
    pbwt, order = source("eimp_pbwt.hip"), source("eimp_order.h")
    kernels = [int(x) for x in re.search(r"kRowsEntries\[kRowsKernels\] = \{([^}]*)\}", pbwt).group(1).split(",")]
    most = 64 * int(re.search(r"kMaxRuns = 64 \* (\d+) - 1", order).group(1)) - 1
    # entries per lane: row_entries_at
    assert "i <= 8 ? 2 * i + 1 : 17 + 4 * (i - 8)" in pbwt and kernels[-1] * 64 - 1 == most
    sizes = [2 * i + 1 for i in range(9)] + list(range(21, kernels[-1] + 1, 4))
    seen = np.zeros((2, len(sizes) + 1), int)  # the last: row by row
    for founders in PANELS:
        for K, ref in zip(KS, case(founders)[2]):
            for rev in (0, 1):
                for runs, rows in block_runs(ref["cref"], K, bool(rev)):
                    dense = rows < 16 or runs > min(most, (K + 63) // 64 * 32)
                    seen[rev, -1 if dense else int(np.searchsorted(sizes, (runs + 1 + 63) // 64))] += 1
    assert seen.min() > 0, seen.tolist()


@pytest.mark.gpu
@pytest.mark.parametrize("founders", PANELS)
def test_every_block_size(built, founders):
    panel, tg, refs = case(founders)
    say("block sizes, founders", founders)
    eng = panel_engine(panel, give_hap=True)
    res = eng.run_batch(tg.gt, tg.s0, tg.W, np.array(KS, np.uint32), digest=True)
    for t, ref in enumerate(refs):
        check_target(ref, eng.copy_target(t, cref=True), KS[t], "gpu", f"target {t} K {KS[t]}")
        assert int(res.dig_pbwt[t]) == ref["dig_pbwt"] and int(res.dig_count0[t]) == ref["dig_count0"]
    eng.close()


# (K, variants): chains long enough to be cut, for every shape that holds K
CUT = [(300, [-1, 0, 1, 2, 3, 4]), (3000, [-1, 1, 2, 3, 4]), (5000, [-1, 2, 3, 4])]
CUT_M = 4200


def cut_case(K):
    panel = synth.make_panel(62, N=K + 100, M=CUT_M, F=40, T=2, flip_rate=0.001)
    tg = synth.make_targets(panel, 62, 2, K=K, wmin=CUT_M - 700, wmax=CUT_M, miss=0.01)
    pv = oracle.PanelView(panel.hap, panel.site, panel.cM)
    return panel, tg, [oracle.process_target(pv, tg.gt[t], tg.s0[t], tg.W[t], K) for t in range(2)]


@pytest.mark.parametrize("K,variants", CUT)
def test_cases_reach_cut_chains(built, host, K, variants):
    """Both targets' chains are cut into three segments or more, whatever the
    number of workgroups on a compute unit."""
    host("cut", K, *[r["Mp"] for r in cut_case(K)[2]])


@pytest.mark.gpu
@pytest.mark.parametrize("K,variants", CUT)
def test_cut_chains_in_every_shape(built, K, variants):
    panel, tg, refs = cut_case(K)
    eng = panel_engine(panel, give_hap=True)
    for v in variants:
        say("cut chains, K", K, "variant", v, "rows", [r["Mp"] for r in refs])
        eng.set_pbwt_variant(v)
        eng.run_batch(tg.gt, tg.s0, tg.W, tg.K, compact=True)
        for t, ref in enumerate(refs):
            check_target(ref, eng.copy_target(t, cref=True), K, "compact", f"K {K} variant {v} target {t}")
    eng.close()
