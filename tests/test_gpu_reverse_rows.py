"""Reverse neighbour lists of given rows: rows whose slots lie close together, as the search's do, and rows of slots
anywhere, so many to a block that its table of 16,384 places fills up and entries take their places one by one; empty
slots, a slot in every row, and both block sizes with ragged ends. Every list holds its owners, each as often as the
slot is in its row."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", ["close", "anywhere", "one"])
@pytest.mark.parametrize("model,n", [("fiducial_3d", 1), ("fiducial_3d", 1023), ("fiducial_3d", 300_001),
                                     ("fiducial_k64", 100_001), ("fiducial_3d", 1_048_576 + 77)])
def test_lists_hold_their_owners(gpu, model, n, rows):
    from gamedev_amd import _lib, model_info
    k = model_info(model)["n_k"]
    rng = np.random.default_rng(n)
    if rows == "close":
        nbr = (np.arange(n)[:, None] + rng.integers(-2*k, 2*k, (n, k))).clip(0, n - 1)
    elif rows == "anywhere":
        nbr = rng.integers(0, n, (n, k))
    else:
        nbr = np.zeros((n, k), np.int64)
        nbr[:, 1:] = rng.integers(0, n, (n, k - 1))
    nbr = np.where(rng.random((n, k)) < 0.05, -1, nbr).astype(np.int32)
    beg, end, rev = np.empty(n, np.uint32), np.empty(n, np.uint32), np.empty((n, k), np.int32)
    print(f"[reverse] {model} n={n} {rows}", flush=True)
    rc = _lib.load(model).gdx_col_check_reverse(n, nbr.ctypes.data, beg.ctypes.data, end.ctypes.data, rev.ctypes.data)
    assert rc == 0
    slots, owners = nbr.ravel(), np.repeat(np.arange(n, dtype=np.int64), k)
    slots, owners = slots[slots >= 0].astype(np.int64), owners[slots >= 0]
    count = np.bincount(slots, minlength=n)
    assert np.array_equal(end.astype(np.int64) - beg, count)
    assert np.array_equal(beg, np.concatenate([[0], np.cumsum(count)[:-1]]))
    got = np.sort(np.repeat(np.arange(n, dtype=np.int64), count)*n + rev.ravel()[:len(slots)])
    assert np.array_equal(got, np.sort(slots*n + owners))
    if rows == "anywhere" and n > 100_000:
        # more slots in a block than places in its table
        block = nbr[:4096 if n >= 1 << 20 else 1024]
        assert len(np.unique(block)) > 16384
