"""The resident crystal pass (all slices of an instance in one launch) against
the path that launches every stage by itself (OPO_RESIDENT=0): the same
arithmetic in the same order, so the same bits, for every grid size, precision
and samples-per-thread setting it takes, for one instance, a full turn of the
teams and more instances than the teams hold, and beside other streams."""
import threading

import numpy as np
import pytest

from tests.helpers import c1, c2, c5, inputs, rel_l2, to_args

pytestmark = pytest.mark.gpu


def batch_fields(P, cfgs, precision, rts, **tuning):
    made = []
    for k, c in enumerate(cfgs):
        p, T, w, Ap_in, Ap, As, Ai = inputs(c, seed=40 + k, sigma=1e-3)
        made.append((P.params_from(P.derive(to_args(c)), precision), w, T, Ap_in, Ap, As, Ai))
    b = P.Batch([m[0] for m in made])
    for k, m in enumerate(made):
        b.upload(k, *m[1:])
    for N in {c.N for c in cfgs}:
        if tuning:
            b.set_tuning(N, **tuning)
    b.run(rts, check_every=0, tol=0.0)
    out = [b.download(k) for k in range(len(cfgs))], b.power()
    b.close()
    return out


def same(a, b):
    assert np.array_equal(a[1], b[1])
    for x, y in zip(a[0], b[0]):
        for f, g in zip(x, y):
            assert (f is None and g is None) or np.array_equal(f, g)


@pytest.mark.parametrize("three", [False, True])
@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("L", [9, 10, 11, 12, 13, 14, 15, 16])
def test_resident_pass_gives_the_same_bits(gpu, monkeypatch, L, fp32, three):
    P = gpu
    make = c2 if three else c1
    cfgs = []
    for k in range(3):
        c = make(N=1 << L, NZ=5, NRT=4)
        c.Nth *= 1.0 + 0.2 * k
        cfgs.append(c)
    for ce, re, ph in [(8, 8, 0), (4, 4, 1), (4, 8, 0), (8, 4, 0)]:
        if re == 4 and L >= 15 and ce == 8:
            continue
        args = dict(col_spt=ce, row_spt=re, phase_mode=ph)
        monkeypatch.setenv("OPO_RESIDENT", "1")  # read when the batch is created
        got = batch_fields(P, cfgs, P.FP32C if fp32 else P.FP64, 3, **args)
        monkeypatch.setenv("OPO_RESIDENT", "0")
        same(got, batch_fields(P, cfgs, P.FP32C if fp32 else P.FP64, 3, **args))


@pytest.mark.parametrize("count,N", [(8, 1024), (9, 4096), (37, 2048), (130, 1024), (64, 8192)])
def test_resident_batches_of_any_count(gpu, monkeypatch, count, N):
    """More instances than XCDs, than teams, and counts that leave teams idle in the last turn."""
    P = gpu
    cfgs = []
    for k in range(count):
        c = c2(N=N, NZ=3, NRT=4)
        c.Nth = 1.5 + 0.05 * k
        cfgs.append(c)
    monkeypatch.setenv("OPO_RESIDENT", "1")
    got = batch_fields(P, cfgs, P.FP64, 3)
    monkeypatch.setenv("OPO_RESIDENT", "0")
    same(got, batch_fields(P, cfgs, P.FP64, 3))


def test_resident_pulsed_instance_and_crystal_pass(gpu, monkeypatch):
    """EOM and GDD around the pass, pump slots, one slice only, and the bare crystal pass."""
    P = gpu
    outs = []
    for on in ("1", "0"):
        monkeypatch.setenv("OPO_RESIDENT", on)
        one = []
        for cfg in (c5(N=4096, NZ=6, NRT=6), c5(N=2048, NZ=1, NRT=6)):
            p, T, w, Ap_in, Ap, As, Ai = inputs(cfg, seed=3, sigma=1e-3)
            s = P.Solver(P.params_from(P.derive(to_args(cfg)), P.FP64))
            s.upload(w, T, Ap_in, Ap, As, Ai)
            s.enable_save(True)
            s.run(0, 6)
            one += list(s.download()) + list(s.download_saved().values())
            s.crystal_pass()
            one += list(s.download())
            s.close()
        outs.append(one)
    for a, b in zip(*outs):
        assert np.array_equal(a, b)


def test_resident_solvers_side_by_side(gpu):
    """Solvers on several host threads at once: every one gives what it gives alone."""
    P = gpu
    cfgs = [c2(N=1 << (10 + k % 6), NZ=12, NRT=40) for k in range(8)]
    ins = [inputs(c, seed=60 + k, sigma=1e-3) for k, c in enumerate(cfgs)]

    def one(k, out):
        p, T, w, Ap_in, Ap, As, Ai = ins[k]
        s = P.Solver(P.params_from(P.derive(to_args(cfgs[k])), P.FP64))
        s.upload(w, T, Ap_in, Ap, As, Ai)
        s.run(0, 40)
        out[k] = s.download()
        s.close()

    alone, beside = {}, {}
    for k in range(len(cfgs)):
        one(k, alone)
    th = [threading.Thread(target=one, args=(k, beside)) for k in range(len(cfgs))]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for k in range(len(cfgs)):
        assert all(np.array_equal(a, b) for a, b in zip(alone[k], beside[k])), k
        assert rel_l2(alone[k][1], beside[k][1]) == 0


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("config", [c1, c2])
@pytest.mark.parametrize("N,count,ce", [(512, 1100, 8), (1024, 600, 8), (4096, 140, 8), (4096, 70, 4), (32768, 18, 8),
                                        (65536, 9, 8), (262144, 2, 8), (262144, 2, 4)])
def test_wavefront_tiles_give_the_same_bits(gpu, monkeypatch, N, count, ce, config, fp32):
    """Batches whose column stage runs a wavefront per tile (every column length, 8 and 4 samples per thread)
    against the same instances alone, whose launches are below that rule and run one per field."""
    P = gpu
    monkeypatch.setenv("OPO_RESIDENT", "0")  # both launch stage by stage
    monkeypatch.setenv("OPO_SPLIT", "0")  # and the batch as one group
    prec = P.FP32C if fp32 else P.FP64
    cfgs = []
    for k in range(5):
        c = config(N=N, NZ=3, NRT=3)
        c.Nth = 1.5 + 0.5 * k
        cfgs.append(c)
    made = []
    for k, c in enumerate(cfgs):
        p, T, w, Ap_in, Ap, As, Ai = inputs(c, seed=80 + k, sigma=1e-3)
        made.append((P.params_from(P.derive(to_args(c)), prec), w, T, Ap_in, Ap, As, Ai))

    def run(n):
        b = P.Batch([made[k % len(made)][0] for k in range(n)])
        for k in range(n):
            b.upload(k, *made[k % len(made)][1:])
        b.set_tuning(N, col_spt=ce, phase_mode=0)
        b.run(2, check_every=0, tol=0.0)
        out = [b.download(k) for k in ({0, 1, n - 1} if n > 1 else {0})]
        b.close()
        return out

    many, one = run(count), run(1)
    for f, g in zip(many[0], one[0]):
        assert (f is None and g is None) or np.array_equal(f, g)
    assert all(np.isfinite(f).all() for x in many for f in x if f is not None)


@pytest.mark.parametrize("three", [False, True])
@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("L", [15, 16, 17, 18])
def test_chip_pass_gives_the_same_bits(gpu, monkeypatch, L, fp32, three):
    """One instance over all CUs against the stage launches, with both phase sources; NZ of 1 and 2 have no
    column stage and one."""
    P = gpu
    make = c2 if three else c1
    for NZ, ph, ce in [(5, 0, 8), (5, 1, 8), (2, 0, 8), (1, 0, 8), (3, 0, 4)]:
        got = []
        for on in ("1", "0"):
            monkeypatch.setenv("OPO_RESIDENT", on)
            got.append(batch_fields(P, [make(N=1 << L, NZ=NZ, NRT=4)], P.FP32C if fp32 else P.FP64, 3,
                                    col_spt=ce, row_spt=8, phase_mode=ph))
        same(*got)


def test_chip_pulsed_instance_and_crystal_pass(gpu, monkeypatch):
    """EOM and GDD around the whole-chip pass, saved round trips, and the bare crystal pass."""
    P = gpu
    outs = []
    for on in ("1", "0"):
        monkeypatch.setenv("OPO_RESIDENT", on)
        one = []
        for cfg, prec in ((c5(N=1 << 16, NZ=6, NRT=6), P.FP64), (c5(N=1 << 17, NZ=3, NRT=6), P.FP32C)):
            p, T, w, Ap_in, Ap, As, Ai = inputs(cfg, seed=3, sigma=1e-3)
            s = P.Solver(P.params_from(P.derive(to_args(cfg)), prec))
            s.upload(w, T, Ap_in, Ap, As, Ai)
            s.enable_save(True)
            s.run(0, 6)
            one += list(s.download()) + list(s.download_saved().values())
            s.crystal_pass()
            one += list(s.download())
            s.close()
        outs.append(one)
    for a, b in zip(*outs):
        assert np.array_equal(a, b)


def test_chip_solvers_side_by_side(gpu):
    """Large and small solvers on several host threads at once: the whole-chip passes close their teams with the
    blocks they get beside each other, and every solver gives what it gives alone."""
    P = gpu
    cfgs = [c2(N=1 << L, NZ=12, NRT=20) for L in (15, 16, 14, 17, 16, 12)]
    ins = [inputs(c, seed=70 + k, sigma=1e-3) for k, c in enumerate(cfgs)]

    def one(k, out):
        p, T, w, Ap_in, Ap, As, Ai = ins[k]
        s = P.Solver(P.params_from(P.derive(to_args(cfgs[k])), P.FP64))
        s.upload(w, T, Ap_in, Ap, As, Ai)
        s.run(0, 20)
        out[k] = s.download()
        s.close()

    alone, beside = {}, {}
    for k in range(len(cfgs)):
        one(k, alone)
    th = [threading.Thread(target=one, args=(k, beside)) for k in range(len(cfgs))]
    for t in th:
        t.start()
    for t in th:
        t.join()
    for k in range(len(cfgs)):
        assert all(np.array_equal(a, b) for a, b in zip(alone[k], beside[k])), k


def test_noalloc_scratch_holds_as_much_as_without_the_counters(gpu, monkeypatch):
    """The one-launch pass takes its counters from what the scratch has left: the longest power history that the
    scratch holds is the same with and without it, and so are the results just above and below."""
    import ctypes as C

    from tests.test_zz_no_alloc import Dev, hip

    P = gpu
    cfg = c1(N=1024, NZ=3, NRT=4)
    p, T, w, Ap_in, Ap, As, _ = inputs(cfg, seed=9, sigma=1e-3)
    prm = P.params_from(P.derive(to_args(cfg)))
    h = hip()

    def run(rt0):
        df, dp = Dev(h, np.concatenate([Ap, As])), Dev(h, np.ascontiguousarray(Ap_in))
        try:
            rc = P.lib().opo_run_noalloc(C.byref(prm), w.ctypes.data_as(C.c_void_p), T.ctypes.data_as(C.c_void_p),
                                         dp.p, Ap_in.size, df.p, rt0, 1, None, None)
            return df.get(2 * cfg.N) if rc == P.OK else None
        finally:
            df.free()
            dp.free()

    def longest():
        lo, hi = 0, 1 << 21  # 16 MiB of history: more than the scratch
        assert run(hi) is None
        while hi - lo > 1:
            mid = (lo + hi) // 2
            lo, hi = (mid, hi) if run(mid) is not None else (lo, mid)
        return lo

    monkeypatch.setenv("OPO_RESIDENT", "0")
    want, field = longest(), run(0)
    monkeypatch.setenv("OPO_RESIDENT", "1")
    assert longest() == want
    for rt0 in (0, want - (1 << 15), want - 64, want):
        assert np.array_equal(run(rt0), field)
