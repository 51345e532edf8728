"""The learned operator on both sides of the reverse lists' block size (1024 or 4096 owners, the larger from
1048576 on, with a ragged last block): kept bounds are raised through the lists, so the exact checks hold as often
as in the other learned tests, and a second run, whose lists are filled in another order, gives the same particles
bit for bit."""
import numpy as np
import pytest

from test_gpu_learned import _operator, _train

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2049, 1048576 + 123])
def test_lists_serve_kept_bounds(gpu, n):
    from gamedev_amd import synth
    h = 0.002
    train, _ = _operator("fiducial_3d", synth.fiducial_3d_state(32768, seed=11), gpu, seed=100)
    m, _, safety = _train("fiducial_3d", train, h, 4, gpu)
    st = synth.fiducial_3d_state(n, seed=12)
    runs = []
    for k in range(2):
        print(f"[reverse] n={n} run {k}", flush=True)
        o, d = _operator("fiducial_3d", st, gpu, seed=7)
        o.use_majorant(m, safety, min_owners=1)
        s = [o.evolve(h) for _ in range(3)]
        runs.append((d["size"].cpu().numpy(), d["numr"].cpu().numpy(), o.rng(), s))
    (a, b) = runs
    for x, y in zip(a[:3], b[:3]):
        assert np.array_equal(x, y)
    checks = sum(s["exact_checks"] for s in a[3])
    assert sum(s["events"] for s in a[3]) > 0 and checks > 0
    assert sum(s["violations"] for s in a[3]) <= 0.01*checks + 3
