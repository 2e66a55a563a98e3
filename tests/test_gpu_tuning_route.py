"""What the autotuner times: the route that the batch's runs take, with that route's own settings."""
import re

import pytest

from tests.helpers import c1, c2, inputs, to_args

pytestmark = pytest.mark.gpu

LINE = re.compile(r"opo autotune: N (\d+) of (\d+) by (one launch|stages), column tile (\d+) x (\d), rows (\d+) x (\d)")


def tuned(P, monkeypatch, capfd, cfg, count, run_first=False):
    """(by one launch, by stages): the settings timed, each (column tile, samples, row tile, samples)."""
    monkeypatch.setenv("OPO_TUNE_LOG", "1")
    p, T, w, Ap_in, Ap, As, Ai = inputs(cfg, seed=4, sigma=1e-3)
    prm = P.params_from(P.derive(to_args(cfg)), P.FP64)
    b = P.Batch([prm] * count)
    for k in range(count):
        b.upload(k, w, T, Ap_in, Ap, As, Ai)
    if run_first:
        b.run(1, check_every=0, tol=0.0)
    capfd.readouterr()
    b.autotune(iters=2)
    err = capfd.readouterr().err
    b.close()
    out = {"one launch": set(), "stages": set()}
    for m in LINE.finditer(err):
        out[m.group(3)].add(tuple(int(m.group(k)) for k in (4, 5, 6, 7)))
    return out["one launch"], out["stages"]


@pytest.mark.parametrize("run_first", [False, True])
@pytest.mark.parametrize("config", [c1, c2])
def test_batch_beyond_the_one_launch_pass_tunes_all_its_tiles(gpu, monkeypatch, capfd, config, run_first):
    """2^20 samples at 2^10 run by stages, also before the batch has run for the first time."""
    one, stages = tuned(gpu, monkeypatch, capfd, config(N=1024, NZ=6, NRT=5), 1024, run_first)
    assert not one
    # 32 rows of 32 points: 64 threads of 8 samples take 16 rows, more threads all 32
    assert {t[0] for t in stages} >= {4, 8, 16} and {t[2] for t in stages if t[3] == 8} >= {16, 32}


@pytest.mark.parametrize("N,count", [(1 << 14, 64), (1 << 15, 1), (1 << 15, 32), (4096, 3)])
def test_batch_within_the_pass_times_nothing_else(gpu, monkeypatch, capfd, N, count):
    """Settings that would send the batch back to stage launches (two turns of 2^14 with 4 samples per thread are
    four; rows of 512 points do not fit a wavefront at 4) are not tried beside the pass."""
    one, stages = tuned(gpu, monkeypatch, capfd, c2(N=N, NZ=6, NRT=5), count)
    assert one and not stages


@pytest.mark.parametrize("config,N,count,by_pass", [
    (c1, 1 << 14, 128, True), (c1, 1 << 14, 256, False), (c1, 1 << 11, 2048, True),
    (c2, 1 << 14, 256, True), (c2, 1 << 14, 40, False), (c1, 1 << 14, 40, False)])
def test_route_follows_the_equations(gpu, monkeypatch, capfd, config, N, count, by_pass):
    """Eight turns of 2^14 are the faster route at three equations (122 against 137 us a slice), not at two (103
    against 97), where they still are at 2^11 (89 against 93)."""
    one, stages = tuned(gpu, monkeypatch, capfd, config(N=N, NZ=6, NRT=5), count)
    assert bool(one) == by_pass and bool(stages) != by_pass
