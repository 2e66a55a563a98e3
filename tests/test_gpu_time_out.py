"""A one-launch crystal pass whose waits give up (forced with a limit of no reads at all: every block then leaves at
its first wait) is an error of the call it happened in."""
import numpy as np
import pytest

from tests.helpers import c1, c2, inputs, to_args

pytestmark = pytest.mark.gpu


def made(P, cfg):
    p, T, w, Ap_in, Ap, As, Ai = inputs(cfg, seed=4, sigma=1e-3)
    return P.params_from(P.derive(to_args(cfg)), P.FP64), (w, T, Ap_in, Ap, As, Ai)


@pytest.mark.parametrize("cfg", [c1(N=4096, NZ=6, NRT=5), c2(N=1 << 14, NZ=1, NRT=5), c2(N=1 << 16, NZ=6, NRT=5)])
def test_run_and_crystal_pass_report_a_time_out(gpu, monkeypatch, cfg):
    P = gpu
    prm, fields = made(P, cfg)
    monkeypatch.setenv("OPO_RESIDENT_POLLS", "0")  # read when the solver is created
    s = P.Solver(prm)
    s.upload(*fields)
    for call in (lambda: s.run(0, 4), s.crystal_pass, lambda: s.run(0, 1)):
        with pytest.raises(P.OpoError, match="timed out"):
            call()
    s.close()
    monkeypatch.delenv("OPO_RESIDENT_POLLS")
    s = P.Solver(prm)
    s.upload(*fields)
    s.run(0, 4)
    assert all(np.isfinite(f).all() for f in s.download() if f is not None)
    s.close()


@pytest.mark.parametrize("batch", [1, 70])
def test_autotune_reports_a_time_out_and_keeps_fields_and_settings(gpu, monkeypatch, batch):
    P = gpu
    prm, fields = made(P, c2(N=4096, NZ=6, NRT=5))
    monkeypatch.setenv("OPO_RESIDENT_POLLS", "0")
    if batch == 1:
        b = P.Solver(prm)
        b.upload(*fields)
        before, tuning = [b.download()], b.get_tuning()
    else:  # two groups of one grid
        b = P.Batch([prm] * batch)
        for k in range(batch):
            b.upload(k, *fields)
        before, tuning = [b.download(k) for k in range(batch)], b.get_tuning()
    with pytest.raises(P.OpoError, match="timed out"):
        b.autotune(iters=3)
    after = [b.download()] if batch == 1 else [b.download(k) for k in range(batch)]
    assert b.get_tuning() == tuning
    for x, y in zip(before, after):
        assert all(np.array_equal(f, g) for f, g in zip(x, y))
    b.close()
