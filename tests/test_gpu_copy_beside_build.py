"""A context's outputs are copied to the host while another context builds: the
copy finds room beside the other's kernels instead of waiting for them to end."""
import ctypes as C
import time

import numpy as np
import pytest

from eagleimp_amd import synth
from eagleimp_amd.engine import lib

from conftest import say
from parity import panel_engine

pytestmark = pytest.mark.gpu

N, M, T = 20000, 60000, 128


def longest_copy(founders, variant):
    """(longest copy, build) in ms, of four builds the one with the shortest
    such copy: 128 targets of up to 60,000 sites at K = 10,000 (256 chains, one
    for every compute unit), 380 KB copied again and again meanwhile, by one of two
    contexts in turn (the runtime may put one of their streams on the hardware
    queue of the building one, behind its kernels)."""
    panel = synth.make_panel(71, N, M, founders, T + 1)
    tg = synth.make_targets(panel, 71, T + 1, K=10000, wmin=M - 3000, wmax=M, miss=0.005)
    eng = panel_engine(panel, give_hap=True)
    eng.set_pbwt_variant(variant)
    big = eng.stream(T, M, 10000, 60 << 30, digest=False)
    small = [eng.stream(1, 2000, 300, 256 << 20, digest=False) for _ in range(2)]
    for st in small:
        st.submit([tg.gt[T]], [int(tg.s0[T])], [2000], [300])
        st.wait()
    want = small[0].copy_target(0)
    rows, c0 = np.zeros_like(want["pbwt"]), np.zeros_like(want["count0"])
    none = C.c_void_p(0)
    best = None
    for i in range(4):
        big.submit([tg.gt[t] for t in range(T)], tg.s0[:T], tg.W[:T], tg.K[:T])
        worst = 0.0
        while not big.done():
            rows[:], c0[:] = 0, -1
            t0 = time.perf_counter()
            rc = lib().eimp_stream_copy_target(small[i % 2]._h, C.c_size_t(0), none, none, none, none, none,
                                               C.c_void_p(c0.ctypes.data), C.c_void_p(rows.ctypes.data), none)
            worst = max(worst, 1e3 * (time.perf_counter() - t0))
            assert rc == 0
            assert np.array_equal(rows, want["pbwt"]) and np.array_equal(c0, want["count0"])
        _, deferred, (build, _) = big.wait()
        assert deferred == 0
        if best is None or worst / build < best[0] / best[1]:
            best = (worst, build)
    for st in (*small, big):
        st.close()
    eng.close()
    say(f"founders {founders}, variant {variant}: longest copy {best[0]:.1f} of {best[1]:.1f} ms")
    return best


def test_beside_chains_on_every_cu(built):
    """Chains of 1,024 threads, one on every compute unit, few runs per block."""
    copy, build = longest_copy(60, 4)
    assert copy < 0.2 * build


def test_beside_the_rows_of_all_blocks(built):
    """Chains that leave room, and blocks of more than 1,087 runs (the rows
    kernel for them fills the registers)."""
    copy, build = longest_copy(400, 2)
    assert copy < 0.1 * build
