"""The column stage with a wavefront per tile against the one with a wavefront per field: a batch above the rule's
line, and the same instance as a solver, whose launches are always per field."""
import numpy as np
import pytest

from tests.helpers import c1, c2, inputs, to_args

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("config", [c1, c2])
@pytest.mark.parametrize("N,count,ce,fp32", [
    (256, 2300, 8, False), (256, 2300, 8, True),  # a tile of 32 columns, of which the grid has 16
    (256, 1200, 4, False), (256, 1200, 4, True),  # one tile an instance
    (1 << 18, 2, 4, False), (1 << 18, 3, 8, True)])  # the longest columns of either precision
def test_batch_above_the_line_gives_a_solvers_bits(gpu, monkeypatch, N, count, ce, fp32, config):
    P = gpu
    monkeypatch.setenv("OPO_RESIDENT", "0")  # stage launches on both sides
    monkeypatch.setenv("OPO_SPLIT", "0")  # and the batch as one group
    made = []
    for k in range(2):
        c = config(N=N, NZ=3, NRT=3)
        c.Nth *= 1.0 + 0.5 * k
        p, T, w, Ap_in, Ap, As, Ai = inputs(c, seed=30 + k, sigma=1e-3)
        made.append((P.params_from(P.derive(to_args(c)), P.FP32C if fp32 else P.FP64), w, T, Ap_in, Ap, As, Ai))
    b = P.Batch([made[k % 2][0] for k in range(count)])
    for k in range(count):
        b.upload(k, *made[k % 2][1:])
    b.set_tuning(N, col_spt=ce, phase_mode=0)
    b.run(2, check_every=0, tol=0.0)
    got = [b.download(k) for k in (0, 1, count - 1)]
    b.close()
    want = []
    for m in made:
        s = P.Solver(m[0])
        s.upload(*m[1:])
        s.set_tuning(col_spt=ce, phase_mode=0)
        s.run(0, 2)
        want.append(s.download())
        s.close()
    for k, x in zip((0, 1, count - 1), got):
        for f, g in zip(x, want[k % 2]):
            assert (f is None and g is None) or (np.isfinite(f).all() and np.array_equal(f, g))
