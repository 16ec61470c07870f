"""Performance cases of the phasing pre-stage: what is timed, with which inputs.

Each case is one call (or one submission and its collection) of the public
entry points in ``eagleimp_amd.engine`` on a resident panel: ``listed()`` names
the fixed ones, ``draw(rng)`` gives more of the same ranges.  Panels and
targets come from the deterministic generator (``eagleimp_amd.synth``) with the
shapes of the benchmark's workloads; where a workload's panel is too long to
make over and over (500,000 sites) its width, founders, K and targets per call
stay and the number of sites shrinks.

Kinds
  batch    Engine.run_batch and eimp_engine_copy_target of every target into
           the program's buffers: the synchronous call of a small program
  device   Engine.run_batch_noalloc: inputs and outputs in device memory, as a
           program keeps them whose next stage runs on the device
  stream   Stream.submit + wait on a context with its own output pool: the
           throughput path.  The rows stay in the pool, where the consumer
           reads them; per target the call returns its sizes and the digests
           over every row word and every count0
  serve    Stream.submit + wait + eimp_stream_copy_target of every target into
           the program's buffers: a request that is phased on the host as soon
           as it is back
  dropin   eimp_engine_run_cref_pbwt: the reference's GPU engine call, host
           buffers in and out
  panel    Engine.ref_pbwt: the whole panel's PBWT for imputation, host
           buffers out
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from eagleimp_amd import synth
from eagleimp_amd.engine import Engine, lib, row_stride, unit_words

KSET = [2000, 4000, 6000, 8000, 10000]
CM_MAX_SPLIT = 0.125
ROWS_PER_SITE = 0.75  # condensed rows per window site on these panels (about)


def case(name, kind, N, M, F, T, K, wmin=None, wmax=None, miss=0.01, beta=0.5, layout="gpu",
         kmin=None, absperm=False):
    c = dict(kind=kind, N=N, M=M, F=F, T=T, K=K, kmin=K if kmin is None else kmin,
             wmin=M if wmin is None else wmin, wmax=M if wmax is None else wmax, miss=miss,
             beta=beta, layout=layout, absperm=absperm)
    return c if name is None else dict(name=name, **c)


def listed():
    return [
        # the smallest call a program makes (the package's own smoke test):
        # launches, copies and the host's part are all there is
        case("tiny-batch", "batch", 256, 3000, 16, 3, 256, kmin=64, wmin=1500, wmax=3000),
        # the 2,000-haplotype panel with K = 1,000, its 20 targets in one call
        case("small-panel-20", "device", 2000, 10000, 50, 20, 1000),
        # many targets with few conditioning haplotypes, odd K and windows
        case("many-small-odd", "device", 1000, 4000, 50, 180, 499, kmin=333, wmin=2111, wmax=3999,
             miss=0.03),
        # one target over a long stretch with the whole panel as conditioning
        # haplotypes: the latency of one long chain of rows
        case("one-long-whole-panel", "device", 10000, 56000, 200, 1, 10000, layout="compact"),
        # one target, a subset of an odd size, an odd window, raw rows
        case("one-subset-raw", "device", 20000, 40000, 200, 1, 3001, wmin=39321, wmax=39321,
             layout="raw"),
        # a few targets with mixed windows and K
        case("few-windows", "device", 20000, 50000, 200, 4, 10000, kmin=2000, wmin=5000, wmax=30000,
             miss=0.02, layout="compact"),
        # whole-panel targets, a full device batch
        case("batch-whole-panel", "stream", 10000, 20000, 200, 192, 10000),
        # windows and K mixed over the benchmark's ranges, a full device batch
        case("batch-windows", "stream", 20000, 100000, 200, 256, 10000, kmin=2000, wmin=10000,
             wmax=100000, miss=0.025, layout="compact"),
        # the 200,000-haplotype panel, K = 10,000
        case("batch-wide-panel", "stream", 200000, 20000, 2000, 96, 10000, beta=0.3),
        # a single request on the serving panel, its rows back on the host
        case("serve-one", "serve", 20000, 50000, 200, 1, 4000, wmin=20000, wmax=20000),
        # the reference's engine call on host buffers
        case("dropin-host", "dropin", 5000, 10000, 100, 12, 2000),
        # the panel's own PBWT with the order after every site, for imputation
        case("panel-pbwt", "panel", 2504, 3000, 100, 1, 2504, absperm=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["batch", "device", "device", "device", "stream", "stream", "serve", "dropin",
                       "panel"])
    layout = rng.choice(["gpu", "compact", "raw"])
    miss = round(rng.uniform(0.0, 0.05), 4)
    if kind == "batch":
        N = 2 * _log(rng, 64, 600)
        M = _log(rng, 700, 4000)
        K = _log(rng, 33, N)
        return case(None, kind, N, M, 16, rng.randint(1, 6), K, wmin=max(64, M // 3), wmax=M,
                    miss=miss)
    if kind == "device":
        # the call's fixed scratch (64 MiB) bounds targets x rows x K
        N = 2 * _log(rng, 400, 10000)
        K = min(N, _log(rng, 100, 10000))
        W = _log(rng, 1500, 40000)
        per = 2.1 * K * 0.9 * W / 16 + 30.0 * W + 5.0 * N
        T = max(1, min(200, int(48e6 / per)))
        T = _log(rng, 1, T) if T > 1 else 1
        return case(None, kind, N, W + rng.randint(0, 4000), rng.choice([50, 200]), T, K,
                    kmin=max(33, K // 3), wmin=max(1000, W // 2), wmax=W, miss=miss, layout=layout)
    if kind == "stream":
        N = 2 * _log(rng, 1000, 60000)
        K = min(N, _log(rng, 500, 10000))
        M = min(_log(rng, 5000, 60000), int(1.2e9 / N))
        T = _log(rng, 16, 160)
        return case(None, kind, N, M, 200 if N <= 20000 else 1000, T, K, kmin=max(200, K // 4),
                    wmin=max(1000, M // 5), wmax=M, miss=miss, layout=rng.choice(["gpu", "compact"]))
    if kind == "serve":
        N = 2 * _log(rng, 1000, 10000)
        K = min(N, _log(rng, 500, 8000))
        W = _log(rng, 3000, 20000)
        return case(None, kind, N, W + rng.randint(0, 9000), 200, rng.randint(1, 3), K, wmin=W,
                    wmax=W, miss=miss, layout=rng.choice(["gpu", "compact"]))
    if kind == "dropin":
        N = 2 * _log(rng, 200, 3000)
        return case(None, kind, N, _log(rng, 1500, 9000), 50, rng.randint(1, 10),
                    min(N, _log(rng, 64, 2000)), miss=miss)
    N = 2 * _log(rng, 100, 4000)
    M = _log(rng, 400, 3000)
    return case(None, kind, N, M, 64, 1, N, absperm=bool(rng.getrandbits(1)))


def _targets(c, seed):
    """Panel and targets of a case, made from the seed alone."""
    panel = synth.make_panel(seed, N=c["N"], M=c["M"], F=c["F"], T=c["T"], beta_a=c["beta"])
    k0, k1 = c["kmin"], c["K"]
    if k0 == k1:
        kset = [k1]
    elif (k0, k1) == (KSET[0], KSET[-1]):
        kset = KSET
    else:  # five K from kmin to K
        kset = [k0 + (k1 - k0) * i // 4 for i in range(5)]
    tg = synth.make_targets(panel, seed, c["T"], kset=kset, wmin=c["wmin"], wmax=c["wmax"],
                            miss=c["miss"])
    return panel, tg


def _flags(layout):
    return dict(compact=layout == "compact", raw=layout == "raw")


def _host_buffers(c, panel):
    """Buffers of a program that copies every target's outputs to the host,
    sized by the case's largest window and K; one row per target."""
    T, W, K = c["T"], c["wmax"], min(c["K"], c["N"])
    mp = _max_rows(W)
    return dict(besthaps=np.zeros((T, K), np.uint32), bhflags=np.zeros((T, unit_words(panel.N)), np.uint64),
                splitsites=np.zeros((T, W), np.uint32), splits=np.zeros((T, unit_words(W)), np.uint64),
                cMdiffs=np.zeros((T, W + 1), np.float32), count0=np.zeros((T, mp), np.int32),
                pbwt=np.zeros((T, 2 * mp * row_stride(K, c["layout"])), np.uint32))


def _max_rows(W):
    """Rows per direction that a buffer for windows of W sites holds: two per
    split site and one, with splits at less than half of the sites."""
    return W + 65


def _ptr(a):
    return C.c_void_p(a.ctypes.data)


def prepare(c, seed):
    panel, tg = _targets(c, seed)
    kind, T = c["kind"], c["T"]
    eng = Engine(0)
    if kind == "dropin":
        K = min(c["K"], c["N"])
        eng.initialize(K, panel.M, panel.N, panel.N, panel.site)
        eng.set_panel_extras(panel.cM, hap=panel.hap)
        # the reference's host pre-phase results of the call's targets
        res = eng.run_batch(tg.gt, tg.s0, tg.W, tg.K, cMmaxSplit=CM_MAX_SPLIT, digest=False)
        outs = [eng.copy_target(t, rows=False) for t in range(T)]
        offs = np.zeros(T + 1, np.uint32)
        offs[1:] = np.cumsum(res.Mp.astype(np.uint32))
        host = dict(rows=np.zeros((T, 8 * _max_rows(panel.M) * unit_words(K)), np.uint32),
                    count0=np.zeros((T, _max_rows(panel.M)), np.int32))
        return dict(c=c, eng=eng, gts=tg.gt, splits=[o["splits"] for o in outs],
                    bhflags=[o["bhflags"] for o in outs], offsets=offs, host=host)
    eng.initialize(2, panel.M, panel.N, panel.N, panel.site)
    eng.set_panel_extras(panel.cM, hap=panel.hap)
    state = dict(c=c, eng=eng, tg=tg)
    if kind in ("batch", "serve"):
        state["host"] = _host_buffers(c, panel)
    if kind == "device":
        state["gt_dev"] = [torch.from_numpy(g.view(np.int64)).cuda() for g in tg.gt]
        mp = state["max_Mp"] = _max_rows(c["wmax"])
        rs = row_stride(min(c["K"], c["N"]), c["layout"])
        state["rows"] = torch.zeros(T, 2 * mp * rs, dtype=torch.int32, device="cuda")
        state["count0"] = torch.zeros(T, mp, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
    elif kind in ("stream", "serve"):
        # the pool holds every target's condensed reference and rows
        pool = 0
        for w, k in zip(tg.W, tg.K):
            k = min(int(k), c["N"])
            Mp = int(1.1 * ROWS_PER_SITE * int(w)) + 64
            pool += (Mp + 16) // 16 * (k + 63) // 64 * 128 + 4 * Mp
            pool += 8 * Mp * row_stride(k, c["layout"]) + 2048
        state["st"] = eng.stream(T, int(tg.W.max()), int(tg.K.max()), pool, **_flags(c["layout"]))
    return state


def _summary(r):
    return dict(S=r.S, Mp=r.Mp, ncalls=r.ncalls, K=r.K, dig_pbwt=r.dig_pbwt, dig_count0=r.dig_count0)


def _copy_targets(fn, handle, T, host):
    """Every target's outputs through the C call, into the caller's buffers."""
    h = host
    for t in range(T):
        if fn(handle, t, *(_ptr(h[k][t]) for k in ("besthaps", "bhflags", "splitsites", "splits",
                                                   "cMdiffs", "count0", "pbwt")), None):
            raise RuntimeError(lib().eimp_last_error().decode())
    return h


def run(s):
    c, eng = s["c"], s["eng"]
    kind, T = c["kind"], c["T"]
    if kind == "panel":
        rows, c0, ap, _ = eng.ref_pbwt(absperm=c["absperm"])
        return dict(rows=rows, count0=c0, **({} if ap is None else dict(absperm=ap)))
    if kind == "dropin":
        A, h = C.c_void_p * T, s["host"]
        at = lambda xs: A(*[x.ctypes.data for x in xs])  # noqa: E731
        if lib().eimp_engine_run_cref_pbwt(eng._h, T, at(s["gts"]), at(s["splits"]), at(s["bhflags"]),
                                           _ptr(s["offsets"]), at(h["rows"]), at(h["count0"])):
            raise RuntimeError(lib().eimp_last_error().decode())
        return h
    tg = s["tg"]
    if kind == "device":
        r = eng.run_batch_noalloc([g.data_ptr() for g in s["gt_dev"]], tg.s0, tg.W, tg.K,
                                  s["max_Mp"], [x.data_ptr() for x in s["rows"]],
                                  [x.data_ptr() for x in s["count0"]], cMmaxSplit=CM_MAX_SPLIT,
                                  **_flags(c["layout"]))
        return dict(_summary(r), rows=s["rows"], count0=s["count0"])
    if kind == "batch":
        r = eng.run_batch(tg.gt, tg.s0, tg.W, tg.K, cMmaxSplit=CM_MAX_SPLIT, **_flags(c["layout"]))
        return dict(_summary(r), **_copy_targets(lib().eimp_engine_copy_target, eng._h, T, s["host"]))
    st = s["st"]
    st.submit(tg.gt, tg.s0, tg.W, tg.K, cMmaxSplit=CM_MAX_SPLIT)
    r, ndeferred, _ = st.wait()
    out = dict(_summary(r), ndeferred=ndeferred)
    if kind == "serve":
        out.update(_copy_targets(lib().eimp_stream_copy_target, st._h, T, s["host"]))
    return out


def work(c):
    """What a pass cannot do without: the panel's windows (haplotype bits) once
    per call, genotypes, the condensed rows' output words and count0; one
    comparison per haplotype, site and target that selects, one placement per
    haplotype, row and direction."""
    N, T = c["N"], c["T"]
    K = min((c["K"] + c["kmin"]) / 2, N)
    if c["kind"] == "panel":
        rows = c["M"]
        b = N * rows / 8 + 8 * math.ceil(N / 32) * rows + 4 * rows + (4 * N * (rows + 1) if c["absperm"] else 0)
        return dict(bytes=b, flops=N * rows)
    W = (c["wmin"] + c["wmax"]) / 2
    rows = ROWS_PER_SITE * W
    b = N * c["wmax"] / 8 + T * (W / 4 + 2 * rows * 8 * math.ceil(K / 32) + 4 * rows)
    f = T * 2 * rows * K
    if K < N and c["kind"] != "dropin":
        f += 2 * T * N * W
    return dict(bytes=b, flops=f)


def _bits(words, n):
    return np.unpackbits(np.ascontiguousarray(words).view(np.uint8), bitorder="little")[:n]


def _exact_target(panel, gt, s0, W, K):
    """Top-K, split sites and cM differences of one target in plain numpy."""
    N = panel.N
    W, s0, K = int(W), int(s0), min(int(K), N)
    g = gt.reshape(-1, 2)
    is0, is2 = _bits(g[:, 0], W).astype(bool), _bits(g[:, 1], W).astype(bool)
    hap = np.stack([_bits(panel.hap[h], s0 + W)[s0:] for h in range(N)]).astype(bool)
    if K < N:
        nerr = np.empty(N, np.int64)
        for h0 in range(0, N, 1024):
            x = hap[h0:h0 + 1024]
            nerr[h0:h0 + 1024] = ((x & is0) | (~x & is2)).sum(1)
        best = np.sort(np.lexsort((np.arange(N), nerr))[:K])
    else:
        best = np.arange(N)
    ones = hap[best].sum(0)
    mono = (ones == 0) | (ones == K)
    cM32 = panel.cM[s0:s0 + W]
    het, miss = ~is0 & ~is2, is0 & is2
    sites, calls, started = [], [], False
    prev = cM32[0]
    for m in range(W):
        started = started or bool(het[m])
        if not started or mono[m] or miss[m]:
            continue
        # the rule itself is stated on float32 positions
        if het[m] or np.float32(cM32[m] - prev) > np.float32(CM_MAX_SPLIT):
            sites.append(m)
            prev = cM32[m]
            if het[m]:
                calls.append(len(sites))
    n = calls[-1] if calls else 0
    sites = np.array(sites[:n], np.int64)
    pos = np.concatenate([[cM32[0]], cM32[sites], [cM32[W - 1]]]).astype(np.float64)
    return dict(S=n, Mp=2 * n + 1, ncalls=len(calls) if n else 0, K=K, besthaps=best,
                splitsites=sites, cMdiffs=np.diff(pos) if n else np.zeros(0))


def exact(c, seed):
    """Selection, split sites and genetic distances in 64 bits for the kinds
    that return them; the other outputs are bit patterns."""
    if c["kind"] not in ("batch", "serve") or c["T"] * c["N"] * c["wmax"] > 5e8:
        return None
    panel, tg = _targets(c, seed)
    ts = [_exact_target(panel, tg.gt[t], tg.s0[t], tg.W[t], tg.K[t]) for t in range(c["T"])]

    def padded(k, n, dtype):
        a = np.zeros((len(ts), n), dtype)
        for row, t in zip(a, ts):
            row[:len(t[k])] = t[k]
        return a

    out = {k: np.array([t[k] for t in ts]) for k in ("S", "Mp", "ncalls", "K")}
    out.update(dig_pbwt=None, dig_count0=None)
    if c["kind"] == "serve":
        out["ndeferred"] = None
    out.update(besthaps=padded("besthaps", min(c["K"], c["N"]), np.int64), bhflags=None,
               splitsites=padded("splitsites", c["wmax"], np.int64), splits=None,
               cMdiffs=padded("cMdiffs", c["wmax"] + 1, np.float64), count0=None, pbwt=None)
    return out
