"""The pair terms' device arithmetic against operations rounded once: the quotients, reciprocals and roots without range
scaling against IEEE division and square root (NumPy's), bit for bit over 2^24 operand pairs of exponents within
+-480, mantissas next to all ones and all zeros among them, and the zero, infinite and NaN operands that the forms for
any operand promise; the logarithms, with the table in LDS and in memory, against the host's same form, bit for bit;
and the chain's straight-line pair rate against the rate pass's and the general loop's, bit for bit, for partners that
share a turbulence regime, that do not, with and without sticking packets, and with empty slots."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

QUOT, QUOT_ANY, RECIP, ROOT, LOG1P_LDS, LOG_LDS, LOG1P, LOG = range(8)


def _device(a, b, host=False):
    from gamedev_amd import _lib
    a, b = np.ascontiguousarray(a, np.float64), np.ascontiguousarray(b, np.float64)
    out, ref = np.empty((8, a.size)), np.empty((3, a.size))
    rc = _lib.load("fiducial_3d").gdx_col_check_arithmetic(a.size, a.ctypes.data, b.ctypes.data, out.ctypes.data,
                                                          ref.ctypes.data if host else None)
    assert rc == 0
    return out, ref


def _same(x, y):
    return (x.view(np.uint64) == y.view(np.uint64)) | (np.isnan(x) & np.isnan(y))


def _operands(rng, n, span):
    mantissa = rng.integers(0, 1 << 52, n, dtype=np.uint64)
    kind = rng.integers(0, 8, n)
    mantissa = np.where(kind == 0, mantissa | np.uint64(0xfffffffffff00), mantissa)
    mantissa = np.where(kind == 1, mantissa & np.uint64(0xff), mantissa)
    exponent = (1023 + rng.integers(-span, span + 1, n)).astype(np.uint64)
    return ((exponent << np.uint64(52)) | mantissa).view(np.float64)


@pytest.mark.parametrize("seed,span", [(1, 480), (2, 480), (3, 40), (4, 3)])
def test_quotients_and_roots_round_once(gpu, seed, span):
    rng = np.random.default_rng(seed)
    n = 1 << 22
    a, b = _operands(rng, n, span), _operands(rng, n, span)
    print(f"[arithmetic] seed {seed} span {span}", flush=True)
    sign = rng.random(n) < 0.5
    out, _ = _device(a, np.where(sign, -b, b))
    q = a/np.where(sign, -b, b)
    assert np.all(_same(out[QUOT], q)) and np.all(_same(out[QUOT_ANY], q))
    assert np.all(_same(out[RECIP], 1.0/np.where(sign, -b, b)))
    assert np.all(_same(out[ROOT], np.sqrt(a)))
    # exact quotients and squares, and quotients next to one
    c = np.round(a/np.exp2(np.floor(np.log2(a)))*2**20)
    d = np.round(b/np.exp2(np.floor(np.log2(b)))*2**20)
    out, _ = _device(c*d, d)
    assert np.all(_same(out[QUOT], c)) and np.all(_same(out[QUOT_ANY], c))
    out, _ = _device(c*c, np.nextafter(c*c, 0.0))
    assert np.all(_same(out[ROOT], c)) and np.all(_same(out[QUOT], c*c/np.nextafter(c*c, 0.0)))


def test_special_operands(gpu):
    v = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1.0, -1.0, 3.0, 1e-300, -1e-300, 1e300, -1e300, 2.0**-1022, 2.0**1020])
    a, b = (x.ravel() for x in np.meshgrid(v, v))
    out, _ = _device(a, b)
    with np.errstate(all="ignore"):
        q, r, s = a/b, 1.0/b, np.sqrt(a)
    # a quotient below the normal range is rounded twice: to an ulp of it there
    tiny = np.isfinite(q) & (np.abs(q) < 2.0**-1022) & (q != 0.0)
    assert np.all(_same(out[QUOT_ANY], q) | tiny), [(x, y) for x, y, k in zip(a, b, _same(out[QUOT_ANY], q) | tiny) if not k]
    assert np.all(np.abs(out[QUOT_ANY][tiny] - q[tiny]) <= 2.0**-1074)
    assert np.all(_same(out[RECIP], r)) and np.all(_same(out[ROOT], s))


def test_logarithms_equal_the_host(gpu):
    rng = np.random.default_rng(5)
    n = 1 << 18
    # cell borders of the table, 256 to an octave from 0.703125 on, and a few ulps to either side
    border = ((np.uint64(0x3fe68000) + rng.integers(0, 256, n).astype(np.uint64)*np.uint64(1 << 12)) << np.uint64(32)).view(np.float64)
    border = (border.view(np.int64) + rng.integers(-3, 4, n)).view(np.float64)*np.exp2(rng.integers(-30, 31, n))
    wide = 10.0**rng.uniform(-300, 300, n)
    small = rng.choice([-1.0, 1.0], n)*rng.random(n)*2.0**-rng.integers(0, 60, n)
    special = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, -1.0, -2.0, 5e-324, 2.0**-1022, 1.0])
    for a, b in ((border - 1.0, border), (small, wide), (wide, np.abs(small)), (special, special)):
        out, ref = _device(a, b, host=True)
        finite = np.isfinite(a) & (a > -1.0)
        assert np.all(_same(out[LOG1P_LDS], ref[0])[finite])
        assert np.all(_same(out[LOG1P], ref[2]))
        assert np.all(_same(out[LOG_LDS], ref[1])) and np.all(_same(out[LOG], ref[1]))


@pytest.mark.parametrize("model", ["fiducial_3d", "fiducial_k64", "wedge_2d", "plain_2d"])
def test_solo_rates_equal_the_rate_pass(gpu, model):
    from gamedev_amd import _lib, model_info
    info = model_info(model)
    k, n = info["n_k"], 20000
    rng = np.random.default_rng(6)
    thin = model in ("wedge_2d", "plain_2d")
    y = rng.uniform(0.6, 1.4, n)
    z = np.full(n, 0.5*np.pi) if thin else 0.5*np.pi + rng.normal(0.0, 0.05, n)
    size = 10.0**rng.uniform(-4.0, 4.0, n)
    owner = np.stack([y, z, size, 10.0**rng.uniform(-6.0, 0.0, n), rng.uniform(1.0, 2.0, n)], axis=1)
    slots = np.empty((n, k, 3))
    # partners smaller than the owner, of about its size, far smaller, and anything
    low, high = np.array([(-1.0, -0.01), (-0.3, 0.3), (-4.0, -1.9), (-4.0, 4.0)])[rng.integers(0, 4, n)].T
    slots[:, :, 0] = size[:, None]*10.0**(low[:, None] + (high - low)[:, None]*rng.random((n, k)))
    slots[:, :, 1] = np.where(rng.random((n, k)) < 0.02, -1.0, 10.0**rng.uniform(-3.0, 3.0, (n, k)))
    slots[:, :, 2] = 0.05*y[:, None]*rng.uniform(0.9, 1.1, (n, k))
    rates, speeds, route = np.empty((3, n, k)), np.empty((2, n, k)), np.empty(n, np.int32)
    print(f"[arithmetic] solo rates {model}", flush=True)
    rc = _lib.load(model).gdx_col_check_solo_rates(n, owner.ctypes.data, slots.ctypes.data, rates.ctypes.data,
                                                  speeds.ctypes.data, route.ctypes.data)
    assert rc == 0
    full = slots[:, :, 1] >= 0.0
    assert np.all(np.isfinite(rates[1])) and np.all(rates[1][~full] == 0.0) and np.any(rates[1] > 0.0)
    assert np.all(_same(rates[0], rates[1])) and np.all(_same(rates[2], rates[1]))
    assert np.all(_same(speeds[0], speeds[1])[full])
    kinds = np.bincount(route, minlength=8)
    print(f"[arithmetic] routes {kinds}", flush=True)
    assert np.all(kinds[[0, 4]] > 50)
    if info["coag_kernel"] == 3:
        assert kinds[1] + kinds[5] > 50 and kinds[2] + kinds[6] > 50
