"""The device planner behind cumf_half_sweep_device: the entry point gives the
factors of the resident handle (whose plan is made on the host) on matrices
whose rows sit at the planner's edges, and refuses what it refused."""
import ctypes as C

import numpy as np
import pytest

import cumf
from cumf import als as G
from tests._checks import rel_rows

pytestmark = pytest.mark.gpu


def _device_sweep(rp, ci, cv, theta, m, n, f, lam, split=0, x0=None):
    bufs = [G.DeviceBuffer.from_array(a) for a in (rp, ci, cv, theta)]
    out = G.DeviceBuffer.from_array(np.full((m, f), 7.0, np.float32) if x0 is None else x0)
    opt = G.default_options(split=split or 16384)
    rc = G.lib().cumf_half_sweep_device(None, *[b.ptr for b in bufs], out.ptr, m, n, f, int(ci.shape[0]), lam,
                                        C.byref(opt))
    err = G.last_error()
    X = out.to_array(np.float32, m * f).reshape(m, f)
    for b in bufs + [out]:
        b.free()
    return rc, err, X


def _matrix(deg, n, seed):
    rng = np.random.default_rng(seed)
    rp = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    ci = rng.integers(0, n, rp[-1]).astype(np.int32)
    cv = rng.integers(1, 6, rp[-1]).astype(np.float32)
    return rp, ci, cv


# Row counts on both sides of the one-block planner's limit (16,384) and of a
# placing block (2,048); lengths at the class edges, empty rows, rows cut into
# two, three and many chunks.
@pytest.mark.parametrize("m", [1, 2047, 16384, 16385, 40961])
@pytest.mark.parametrize("f", [8, 10, 144])
def test_device_plan_gives_the_handles_factors(m, f):
    n, lam = 300, 0.05
    rng = np.random.default_rng(m + f)
    edges = np.array([0, 1, 31, 32, 63, 95, 96, 239, 240, 255, 256, 287, 288, 511, 512])
    deg = np.where(rng.random(m) < 0.02, rng.choice(edges, m), rng.integers(0, 6, m))
    deg[rng.integers(0, m, min(m, 6))] = rng.choice([2048, 2049, 4096, 4097, 9001], min(m, 6))
    rp, ci, cv = _matrix(deg, n, m)
    theta = cumf.init_factors(n, f, 3)
    rc, err, X = _device_sweep(rp, ci, cv, theta, m, n, f, lam)
    assert rc == 0, err
    with G.ALS(f, lam) as h:
        h.set_ratings(m, n, rp, ci, cv)
        h.set_factors(theta=theta)
        h.update_x()
        Xh, _ = h.get_factors()
    assert np.all(X[deg == 0] == 0)
    live = deg > 0
    # the same arithmetic, split rows' partial Grams cut elsewhere: FP32
    # rounding of sums of up to 9,001 terms, times the systems' condition
    assert rel_rows(X[live], Xh[live]).max() <= 1e-5
    whole = live & (deg <= 2048)
    np.testing.assert_array_equal(X[whole], Xh[whole])


@pytest.mark.parametrize("m", [5, 20000])
@pytest.mark.parametrize("f", [8, 10])
def test_bad_row_pointers_are_refused_and_write_nothing(m, f):
    n = 50
    rp, ci, cv = _matrix(np.full(m, 3), n, 1)
    theta = cumf.init_factors(n, f, 3)
    x0 = np.full((m, f), 7.0, np.float32)
    for what, text in (("first", "start at 0"), ("last", "start at 0"), ("drop", "decrease at row 2"),
                       ("wild", "decrease at row")):
        b = rp.copy()
        if what == "first":
            b[0] = 1
        elif what == "last":
            b[m] -= 1
        elif what == "drop":
            b[3] = b[2] - 1
        else:
            b[3], b[4] = 2**31 - 1, -2**31
        rc, err, X = _device_sweep(b, ci, cv, theta, m, n, f, 0.05, x0=x0)
        assert rc == 1 and text in err, (what, rc, err)
        np.testing.assert_array_equal(X, x0)
    rc, err, X = _device_sweep(rp, ci, cv, theta, m, n, f, 0.05, x0=x0)
    assert rc == 0 and np.all(np.isfinite(X))


def _handle_sweep(rp, ci, cv, theta, m, n, f, lam, split):
    with G.ALS(f, lam, split=split) as h:
        h.set_ratings(m, n, rp, ci, cv)
        h.set_factors(theta=theta)
        h.update_x()
        return h.get_factors()[0]


# Splits below 2,048 come from the caller alone.  Many split rows on both sides
# of the one-block planner's limit, chunks in the classes of one length (below
# 256) and in wider ones, one to thousands of chunks a row.
@pytest.mark.parametrize("split", [1, 7, 96, 256, 300])
@pytest.mark.parametrize("m", [1, 16384, 16385])
def test_rows_cut_as_the_callers_split_says(m, split):
    """The device planner cuts and orders a row's chunks as the host one does,
    so the factors are the handle's bit for bit."""
    n, lam, f = 500, 0.05, 8
    rng = np.random.default_rng(m + split)
    deg = np.where(rng.random(m) < 0.3, rng.integers(0, 3 * split + 2, m), rng.integers(0, 4, m))
    deg[rng.integers(0, m, min(m, 4))] = rng.choice([split, split + 1, 2 * split + 1, 70 * split + 3, 20011], min(m, 4))
    if m == 1:
        deg[0] = 20011
    rp, ci, cv = _matrix(deg, n, m)
    theta = cumf.init_factors(n, f, 3)
    rc, err, X = _device_sweep(rp, ci, cv, theta, m, n, f, lam, split=split)
    assert rc == 0, err
    np.testing.assert_array_equal(X, _handle_sweep(rp, ci, cv, theta, m, n, f, lam, split))


@pytest.mark.parametrize("f", [100, 140])
def test_partial_grams_beyond_the_bound_that_needs_no_wait(f):
    """Their bound passes 64 MB (28 and 45 KB a chunk), so the host sizes them
    by the plan's own counts; a smaller call then works in the kept buffers."""
    n, lam, split = 400, 0.05, 96
    theta = cumf.init_factors(n, f, 3)
    for m in (2000, 150):
        rng = np.random.default_rng(m)
        rp, ci, cv = _matrix(rng.integers(0, 220, m), n, m)
        rc, err, X = _device_sweep(rp, ci, cv, theta, m, n, f, lam, split=split)
        assert rc == 0, err
        np.testing.assert_array_equal(X, _handle_sweep(rp, ci, cv, theta, m, n, f, lam, split))


def test_large_partial_grams_are_given_back():
    """A small split size makes 1.4 GB of partial Grams (f = 140, 45 KB a
    chunk); the next ordinary call gives them back and is right."""
    n, lam, f = 400, 0.05, 140
    theta = cumf.init_factors(n, f, 3)

    def free_bytes():
        free, total = C.c_size_t(), C.c_size_t()
        assert G.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    rng = np.random.default_rng(0)
    small, big = _matrix(rng.integers(0, 220, 50), n, 50), _matrix(np.full(2100, 100), n, 2100)
    rc, err, X0 = _device_sweep(*small, theta, 50, n, f, lam, split=96)
    assert rc == 0, err
    before = free_bytes()
    rc, err, _ = _device_sweep(*big, theta, 2100, n, f, lam, split=7)
    assert rc == 0, err
    assert before - free_bytes() > 1 << 30
    rc, err, X1 = _device_sweep(*small, theta, 50, n, f, lam, split=96)
    assert rc == 0, err
    assert before - free_bytes() < 64 << 20
    np.testing.assert_array_equal(X1, X0)
