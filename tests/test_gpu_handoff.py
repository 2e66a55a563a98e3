"""Instances handed to the resident pass's teams where a turn is as short as it gets: passes of one slice, and
finished instances among running ones.  The stage launches (OPO_RESIDENT=0) give the same bits."""
import numpy as np
import pytest

from tests.helpers import c1, c2, inputs, to_args

pytestmark = pytest.mark.gpu


def fields(P, cfgs, rts, bad=(), check=0):
    made = []
    for k, c in enumerate(cfgs):
        p, T, w, Ap_in, Ap, As, Ai = inputs(c, seed=90 + k % 5, sigma=1e-3)
        if k in bad:
            As = As.copy()
            As[k % c.N] = np.nan  # its power is not finite after the first round trip, which ends it
        made.append((P.params_from(P.derive(to_args(c)), P.FP64), w, T, Ap_in, Ap, As, Ai))
    b = P.Batch([m[0] for m in made])
    for k, m in enumerate(made):
        b.upload(k, *m[1:])
    _, states = b.run_ex(rts, check_every=check, tol=1e-14)
    out = [b.download(k) for k in range(len(cfgs))]
    b.close()
    return out, states


def both_routes(P, monkeypatch, cfgs, rts, **kw):
    monkeypatch.setenv("OPO_RESIDENT", "1")  # read when the batch is created
    got, gs = fields(P, cfgs, rts, **kw)
    monkeypatch.setenv("OPO_RESIDENT", "0")
    want, ws = fields(P, cfgs, rts, **kw)
    assert list(gs) == list(ws)
    for k, (x, y) in enumerate(zip(got, want)):
        for f, g in zip(x, y):
            assert (f is None and g is None) or np.array_equal(f, g, equal_nan=True), k
            assert f is None or k in kw.get("bad", ()) or np.isfinite(f).all(), k
    return gs


@pytest.mark.parametrize("make", [c1, c2])
@pytest.mark.parametrize("N,count", [(1024, 300), (4096, 100), (1 << 14, 64)])
def test_one_slice_and_more_instances_than_teams(gpu, monkeypatch, N, count, make):
    cfgs = []
    for k in range(count):
        c = make(N=N, NZ=1, NRT=5)
        c.Nth *= 1.0 + 0.01 * k
        cfgs.append(c)
    both_routes(gpu, monkeypatch, cfgs, 4)


@pytest.mark.parametrize("compact", ["1", "0"])
@pytest.mark.parametrize("N,count", [(1024, 300), (1 << 14, 64), (1 << 14, 8), (4096, 1)])
def test_finished_instances_among_running_ones(gpu, monkeypatch, N, count, compact):
    """Several turns a team at 2^14, the first, neighbouring and last instances among those that end."""
    P = gpu
    monkeypatch.setenv("OPO_COMPACT", compact)
    cfgs = []
    for k in range(count):
        c = c2(N=N, NZ=4, NRT=9)
        c.Nth *= 1.0 + 0.01 * k
        cfgs.append(c)
    bad = {0, 1, count // 2, count - 1} | set(range(count // 3, count // 3 + count // 8))
    for check in (0, 3):
        states = both_routes(P, monkeypatch, cfgs, 8, bad=bad, check=check)
        assert [k for k in range(count) if states[k] == -1] == sorted(b for b in bad if b < count)


@pytest.mark.parametrize("N,fp32", [(4096, False), (1 << 14, False), (1 << 14, True), (1 << 16, False)])
def test_diverged_solver_goes_on_as_by_stage_launches(gpu, monkeypatch, N, fp32):
    """A solver's slices take no notice of its power: after a round trip that is not finite the fields go through
    the rest of the run by either route."""
    P = gpu
    outs = []
    for on in ("1", "0"):
        monkeypatch.setenv("OPO_RESIDENT", on)
        one = []
        for bad in (np.nan, np.inf, 1e30 if fp32 else 1e155):
            cfg = c2(N=N, NZ=4, NRT=9)
            p, T, w, Ap_in, Ap, As, Ai = inputs(cfg, seed=8, sigma=1e-3)
            As = As.copy()
            if np.isfinite(bad):  # without a pump the fields stay finite; at FP64 their power is not
                As *= bad
                Ap_in, Ap, Ai = 0 * Ap_in, 0 * Ap, 0 * Ai
            else:
                As[5] = bad
            s = P.Solver(P.params_from(P.derive(to_args(cfg)), P.FP32C if fp32 else P.FP64))
            s.upload(w, T, Ap_in, Ap, As, Ai)
            s.run(0, 5)
            one += list(s.download()) + [s.power_history(5)]
            s.set_fields(Ap, np.zeros(N), Ai)  # a run from sound fields is sound again
            s.run(0, 2)
            one += list(s.download())
            assert all(np.isfinite(f).all() for f in one[-3:])
            s.close()
        outs.append(one)
    for a, b in zip(*outs):
        assert np.array_equal(a, b, equal_nan=True)
