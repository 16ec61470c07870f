"""Outputs to host memory go through pinned chunks of 2 MiB, four in flight,
their slices copied by several threads: arrays on both sides of a chunk, of the
four buffers and of the last slice, and many arrays in one chunk."""
import ctypes as C

import numpy as np
import pytest

import oracle
from eagleimp_amd import synth
from eagleimp_amd.engine import lib

from conftest import say
from parity import check_target, panel_engine

pytestmark = pytest.mark.gpu


# (n + 1) * 1024 * 4 bytes of orders after the rows: 2 MiB is n = 511
@pytest.mark.parametrize("n", [1, 380, 400, 511, 512, 1500, 2047, 2600])
def test_panel_orders_at_chunk_edges(built, n):
    say("copy out: sites", n)
    panel = synth.make_panel(31, N=1024, M=2700, F=16, T=1)
    eng = panel_engine(panel)
    er, ec, ea = oracle.build_ref_pbwt(panel.site[3:3 + n], 1024)
    for _ in range(2):  # the second pass finds the buffers and threads there
        rows, c0, ap, _ = eng.ref_pbwt(3, n)
        assert np.array_equal(rows, er) and np.array_equal(c0, ec) and np.array_equal(ap, ea)
    eng.close()


@pytest.mark.parametrize("pinned", [False, True])
def test_rows_to_pageable_and_pinned_memory(built, pinned):
    panel = synth.make_panel(33, N=700, M=9000, F=16, T=2)
    tg = synth.make_targets(panel, 33, 2, kset=[601], wmin=8800, wmax=9000)
    pv = oracle.PanelView(panel.hap, panel.site, panel.cM)
    eng = panel_engine(panel)
    hip = C.CDLL("libamdhip64.so.7")
    r = eng.run_batch(tg.gt, tg.s0, tg.W, tg.K)
    for t in range(2):
        ref = oracle.process_target(pv, tg.gt[t], tg.s0[t], tg.W[t], tg.K[t])
        want = eng.copy_target(t, cref=True)
        check_target(ref, want, int(r.K[t]), "gpu", f"target {t}", monos=eng.copy_monos(t))
        n = want["pbwt"].size
        p = C.c_void_p()
        if pinned:
            assert hip.hipHostMalloc(C.byref(p), C.c_size_t(4 * n), C.c_uint(0)) == 0
            rows = np.frombuffer((C.c_uint32 * n).from_address(p.value), dtype=np.uint32)
        else:
            rows = np.empty(n, dtype=np.uint32)
        rows[:] = 0xFFFFFFFF
        c0 = np.full(want["count0"].size, -1, dtype=np.int32)
        none = C.c_void_p(0)
        rc = lib().eimp_engine_copy_target(eng._h, C.c_size_t(t), none, none, none, none, none,
                                           C.c_void_p(c0.ctypes.data), C.c_void_p(rows.ctypes.data), none)
        assert rc == 0
        assert np.array_equal(rows, want["pbwt"].view(np.uint32).ravel())
        assert np.array_equal(c0, want["count0"].ravel())
        if pinned:
            del rows
            assert hip.hipHostFree(p) == 0
    eng.close()
