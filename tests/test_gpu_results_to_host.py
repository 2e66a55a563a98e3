"""Fields and powers to the host: the pinned path of large batches, the direct path of small ones, and single solvers
give the same bytes."""
import numpy as np
import pytest

from tests.helpers import c1, c2, inputs, to_args

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp32", [False, True])
@pytest.mark.parametrize("make", [c1, c2])
def test_results_do_not_depend_on_the_batch_size(gpu, make, fp32):
    P = gpu
    made = []
    for k in range(17):  # two grids, so one staging buffer serves both sizes
        c = make(N=256 if k % 3 else 2048, NZ=4, NRT=12)
        c.Nth *= 1.0 + 0.1 * k
        p, T, w, Ap_in, Ap, As, Ai = inputs(c, seed=20 + k, sigma=1e-3)
        made.append((P.params_from(P.derive(to_args(c)), P.FP32C if fp32 else P.FP64), w, T, Ap_in, Ap, As, Ai))

    def run(which, check):
        b = P.Batch([made[k][0] for k in which])
        for j, k in enumerate(which):
            b.upload(j, *made[k][1:])
        rts = b.run(12, check_every=check, tol=10.0 if check else 0.0)  # (a tolerance that every instance meets)
        out = {k: (rts[j], b.download(j), b.power()[j], b.power_history(j, 12)) for j, k in enumerate(which)}
        b.close()
        return out

    for check in (0, 3):
        many, few = run(range(17), check), {}
        few.update(run(range(9), check))
        few.update(run(range(9, 17), check))
        for k in range(17):
            a, b = many[k], few[k]
            assert a[0] == b[0] and a[2] == b[2]
            assert (a[0] >= 0) == bool(check)
            for x, y in zip(a[1], b[1]):
                assert (x is None and y is None) or np.array_equal(x, y)
            done = a[3][a[3] != 0]
            assert a[2] == done[-1]


@pytest.mark.parametrize("fp32", [False, True])
def test_set_fields_and_download_round_trip(gpu, fp32):
    P = gpu
    c = c2(N=512, NZ=4, NRT=4)
    p, T, w, Ap_in, Ap, As, Ai = inputs(c, seed=5, sigma=1e-3)
    s = P.Solver(P.params_from(P.derive(to_args(c)), P.FP32C if fp32 else P.FP64))
    s.upload(w, T, Ap_in, Ap, As, Ai)
    rng = np.random.default_rng(1)
    x = [rng.standard_normal(512) + 1j * rng.standard_normal(512) for _ in range(3)]
    want = [v.astype(np.complex64).astype(np.complex128) if fp32 else v for v in x]
    s.set_fields(*x)
    for a, b in zip(s.download(), want):
        assert np.array_equal(a, b)
    s.set_fields(x[1], None, x[0])
    for a, b in zip(s.download(), (want[1], np.zeros(512), want[0])):
        assert np.array_equal(a, b)
    s.close()
