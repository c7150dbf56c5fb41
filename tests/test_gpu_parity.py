"""GPU parity of the HIP path against the FP64 oracle, through the C ABI.

Tolerances (FP32 Gram on MFMA + FP32 Cholesky vs an FP64 oracle):
  * Gram entries: |A_gpu - A_64| <= 2e-5 * max|diag A_64| per row (FP32
    accumulation of up to a few thousand terms).
  * Solve: relative residual of the GPU solution against the system the
    GPU formed, computed in FP64: ||b - A x|| / ||b|| <= 1e-5.
  * Solution vs oracle: ||x_gpu - x_64|| / ||x_64|| <= 1e-3 per row.
  * Held-out RMSE after full training: |RMSE_gpu - RMSE_64| <= 1e-3.
"""
import ctypes as C
import os

import numpy as np
import pytest

import cumf
from cumf import als as G
from oracle import oracle as O
from tests import _data

pytestmark = pytest.mark.gpu


def _als(ds, f, lam, **opt):
    h = G.ALS(f, lam, **opt)
    h.set_dataset(ds)
    return h


def test_mfma_layout():
    out = G.mfma_layout()
    A = 100.0 * np.arange(16)[:, None] + np.arange(4)[None, :]
    B = 1000.0 * np.arange(4)[:, None] + np.arange(16)[None, :]
    D = A @ B
    lane = np.arange(64)
    for r in range(4):
        np.testing.assert_array_equal(out[:, r], D[4 * (lane // 16) + r, lane % 16])


@pytest.mark.parametrize("f", [32, 100])
def test_gram_matches_oracle(f):
    ds = _data.netflix_like_small()
    lam = 0.058
    T0 = cumf.init_factors(ds.n, f, 1)
    with _als(ds, f, lam) as h:
        h.set_factors(theta=T0)
        deg = np.diff(ds.csr_row_ptr)
        rows = np.concatenate([np.argsort(-deg)[:4], np.argsort(deg)[:4], [7, 123, 999]]).astype(np.int32)
        D = h.row_gram(0, rows)
    ldf = (f + 3) // 4 * 4
    for k, u in enumerate(rows):
        A, b = O.row_system(ds.csr_row_ptr, ds.csr_col, ds.csr_val, T0, f, lam, u)
        scale = np.abs(np.diag(A)).max()
        assert np.abs(D[k, :f, :f] - A).max() <= 2e-5 * scale, u
        assert np.abs(D[k, :f, ldf] - b).max() <= 2e-5 * max(np.abs(b).max(), 1.0), u
        # padding columns stay zero
        assert np.all(D[k, :f, f:ldf] == 0)


def _check_sweep(ds_rp, ds_ci, ds_cv, theta, Xg, f, lam, rows):
    Xo, st = O.half_sweep(ds_rp, ds_ci, ds_cv, theta, lam)
    assert st.max() == 0
    rel = np.linalg.norm(Xg - Xo, axis=1) / np.maximum(np.linalg.norm(Xo, axis=1), 1e-30)
    assert rel.max() <= 1e-3, (rel.max(), int(rel.argmax()))
    for u in rows:
        A, b = O.row_system(ds_rp, ds_ci, ds_cv, theta, f, lam, u)
        res = np.linalg.norm(b - A @ Xg[u].astype(np.float64)) / np.linalg.norm(b)
        assert res <= 1e-4, (u, res)
    return rel


@pytest.mark.parametrize("f,split", [(32, 2048), (100, 2048), (100, 64), (10, 200), (128, 300)])
def test_half_sweeps_match_oracle(f, split):
    ds = _data.netflix_like_small()
    lam = 0.058
    T0 = cumf.init_factors(ds.n, f, 2)
    with _als(ds, f, lam, split=split) as h:
        h.set_factors(theta=T0)
        h.update_x()
        X1, _ = h.get_factors()
        h.update_theta()
        _, T1 = h.get_factors()
        assert h.stats()["failed_rows"] == 0
    _check_sweep(ds.csr_row_ptr, ds.csr_col, ds.csr_val, T0, X1, f, lam, [0, 1, 2])
    _check_sweep(ds.csc_col_ptr, ds.csc_row, ds.csc_val, X1, T1, f, lam, [0, 1, 2])


def test_solve_residual_against_gpu_system():
    """Relative residual of each GPU solve, against the Gram the GPU formed,
    in FP64: <= 1e-5."""
    ds = _data.netflix_like_small()
    f, lam = 100, 0.058
    T0 = cumf.init_factors(ds.n, f, 3)
    with _als(ds, f, lam) as h:
        h.set_factors(theta=T0)
        h.update_x()
        X1, _ = h.get_factors()
        rows = np.arange(0, ds.m, 97, dtype=np.int32)
        D = h.row_gram(0, rows).astype(np.float64)
    for k, u in enumerate(rows):
        A, b = D[k, :f, :f], D[k, :f, f]
        res = np.linalg.norm(b - A @ X1[u].astype(np.float64)) / np.linalg.norm(b)
        assert res <= 1e-5, (u, res)


def test_full_als_small_zipf_rmse():
    """m=10,000 n=2,000 (450k training ratings), f=32, lambda=0.05, 10
    iterations: held-out RMSE within 1e-3 of the FP64 oracle."""
    ds = _data.small_zipf()
    f, lam, iters = 32, 0.05, 10
    T0 = cumf.init_factors(ds.n, f, 0)
    _, _, hist = O.als_train(ds, f, lam, iters, T0)
    with _als(ds, f, lam) as h:
        h.set_factors(theta=T0)
        rm = []
        for _ in range(iters):
            h.iterate(1)
            rm.append(h.rmse())
    assert abs(rm[-1] - hist[-1]) <= 1e-3, (rm, hist)
    assert np.all(np.abs(np.array(rm) - hist) <= 1e-3)


def test_deterministic():
    ds = _data.netflix_like_small()
    f, lam = 100, 0.058
    T0 = cumf.init_factors(ds.n, f, 4)
    outs = []
    for _ in range(2):
        with _als(ds, f, lam, split=128) as h:
            h.set_factors(theta=T0)
            h.iterate(2)
            outs.append(h.get_factors())
    np.testing.assert_array_equal(outs[0][0], outs[1][0])
    np.testing.assert_array_equal(outs[0][1], outs[1][1])


def test_empty_rows_give_zero_factors():
    rp = np.array([0, 2, 2, 5, 5], np.int32)  # rows 1 and 3 empty
    ci = np.array([0, 2, 1, 2, 3], np.int32)
    cv = np.array([4, 5, 3, 1, 2], np.float32)
    f, lam = 8, 0.1
    T0 = cumf.init_factors(4, f, 5)
    with G.ALS(f, lam) as h:
        h.set_ratings(4, 4, rp, ci, cv)
        h.set_factors(theta=T0)
        h.update_x()
        X, _ = h.get_factors()
    Xo, _ = O.half_sweep(rp, ci, cv, T0, lam)
    assert np.all(X[[1, 3]] == 0)
    np.testing.assert_allclose(X, Xo, rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("f", [10, 100])
def test_do_als_with_csr_dropin(f):
    """The legacy entry point: CSR in mallocBest memory (consumed)."""
    ds = _data.netflix_like_small()
    lam = 0.058
    T0 = cumf.init_factors(ds.n, f, 6)
    X = G.do_als_with_csr(ds.csr_row_ptr, ds.csr_col, ds.csr_val, T0, ds.m, ds.n, f, lam)
    Xo, _ = O.half_sweep(ds.csr_row_ptr, ds.csr_col, ds.csr_val, T0, lam)
    rel = np.linalg.norm(X - Xo, axis=1) / np.linalg.norm(Xo, axis=1)
    assert rel.max() <= 1e-3


def test_do_als_with_csr_rejects_bad_f():
    ds = _data.tiny()
    T0 = cumf.init_factors(ds.n, 4, 0)
    with pytest.raises(G.CumfError):
        G.do_als_with_csr(ds.csr_row_ptr, ds.csr_col, ds.csr_val, T0, ds.m, ds.n, 0, 0.1)


def test_host_memory_fallback():
    """mallocBest's mapped-host fallback still gives the right answer."""
    ds = _data.tiny()
    f, lam = 16, 0.1
    T0 = cumf.init_factors(ds.n, f, 8)
    G.lib().cumf_debug_force_host_alloc(1)
    try:
        X = G.do_als_with_csr(ds.csr_row_ptr, ds.csr_col, ds.csr_val, T0, ds.m, ds.n, f, lam)
    finally:
        G.lib().cumf_debug_force_host_alloc(0)
    Xo, _ = O.half_sweep(ds.csr_row_ptr, ds.csr_col, ds.csr_val, T0, lam)
    np.testing.assert_allclose(X, Xo, rtol=1e-3, atol=1e-4)


def test_device_transpose_matches_host_csc():
    """Handles built with and without a host CSC (the latter transposed on
    the device) give bit-identical Theta sweeps."""
    ds = _data.netflix_like_small()
    f, lam = 32, 0.058
    T0 = cumf.init_factors(ds.n, f, 9)
    outs = []
    for with_csc in (True, False):
        with G.ALS(f, lam) as h:
            if with_csc:
                h.set_ratings(ds.m, ds.n, ds.csr_row_ptr, ds.csr_col, ds.csr_val,
                              ds.csc_col_ptr, ds.csc_row, ds.csc_val)
            else:
                h.set_ratings(ds.m, ds.n, ds.csr_row_ptr, ds.csr_col, ds.csr_val)
            h.set_factors(theta=T0)
            h.iterate(1)
            outs.append(h.get_factors())
    np.testing.assert_array_equal(outs[0][0], outs[1][0])
    np.testing.assert_array_equal(outs[0][1], outs[1][1])


def test_concurrent_dropin_callers():
    """Several host threads call doALSWithCSR at once (Spark executors share
    a GPU): every result matches the oracle."""
    import threading
    ds = _data.netflix_like_small()
    f, lam = 16, 0.058
    results, errors = {}, []

    def work(i):
        try:
            T0 = cumf.init_factors(ds.n, f, 100 + i)
            results[i] = (T0, G.do_als_with_csr(ds.csr_row_ptr, ds.csr_col, ds.csr_val, T0, ds.m, ds.n, f, lam))
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for i, (T0, X) in results.items():
        Xo, _ = O.half_sweep(ds.csr_row_ptr, ds.csr_col, ds.csr_val, T0, lam)
        rel = np.linalg.norm(X - Xo, axis=1) / np.linalg.norm(Xo, axis=1)
        assert rel.max() <= 1e-3, i


def test_runals_driver_small_preset():
    import json
    import subprocess
    from cumf import _paths
    exe = os.path.join(_paths.PKG_DIR, "runals")
    r = subprocess.run([exe, "gpu", "32", "3", "0.05", "zipf_10k_2k_500k"], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0, r.stderr
    summary = json.loads(r.stdout.strip().splitlines()[-1])
    assert summary["iterations"] == 3 and summary["failed_rows"] == 0
    assert 0.2 < summary["heldout_rmse"] < 1.0


def test_runals_mixed_path_with_autotune(tmp_path):
    import json
    import subprocess
    from cumf import _paths
    exe = os.path.join(_paths.PKG_DIR, "runals")
    table = str(tmp_path / "tiles.txt")
    r = subprocess.run([exe, "gpu", "32", "3", "0.05", "zipf_10k_2k_500k", "--precision", "bf16", "--solver", "cg",
                        "--autotune", table, "--graph", "1"], capture_output=True, text=True, timeout=180)
    assert r.returncode == 0, r.stderr
    summary = json.loads(r.stdout.strip().splitlines()[-1])
    assert summary["precision"] == "bf16" and summary["solver"] == "cg" and summary["failed_rows"] == 0
    assert 0.2 < summary["heldout_rmse"] < 1.0
    r2 = subprocess.run([exe, "gpu", "32", "3", "0.05", "zipf_10k_2k_500k", "--precision", "bf16", "--solver", "cg",
                         "--tiles", table], capture_output=True, text=True, timeout=180)
    assert r2.returncode == 0, r2.stderr
    assert abs(json.loads(r2.stdout.strip().splitlines()[-1])["heldout_rmse"] - summary["heldout_rmse"]) < 1e-6


def test_runals_reads_reference_binary_csr(tmp_path):
    ds = _data.tiny()
    import subprocess
    from cumf import _paths
    pre = str(tmp_path / "r")
    G.save_csr_bin(pre, ds.csr_row_ptr, ds.csr_col, ds.csr_val)
    exe = os.path.join(_paths.PKG_DIR, "runals")
    r = subprocess.run([exe, "gpu", "8", "2", "0.1", f"csr:{ds.m}:{ds.n}:{ds.nnz}:{pre}"], capture_output=True,
                       text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    assert '"failed_rows": 0' in r.stdout


def test_graph_replay_matches_eager():
    """use_graph: one captured graph per half-sweep, replayed several times
    with eager work between replays, equals eager iterations bit for bit."""
    ds = _data.netflix_like_small()
    f, lam = 32, 0.058
    T0 = cumf.init_factors(ds.n, f, 11)
    with _als(ds, f, lam, split=256) as eager, _als(ds, f, lam, split=256, use_graph=1, timing=1) as graph:
        eager.set_factors(theta=T0)
        graph.set_factors(theta=T0)
        for rep in range(3):
            eager.iterate(1)
            graph.iterate(1)
            graph.rmse()  # eager kernels on the same stream between replays
            Xe, Te = eager.get_factors()
            Xg, Tg = graph.get_factors()
            np.testing.assert_array_equal(Xe, Xg, err_msg=f"replay {rep}")
            np.testing.assert_array_equal(Te, Tg, err_msg=f"replay {rep}")
        st = graph.stats()
        assert st["iters"] == 6 and st["iter_ms"] > 0  # two half-sweep replays per iteration


@pytest.mark.parametrize("f", [10, 100])
def test_compat_system_bit_exact(f):
    """compat_hermitian_bug: the system the GPU solver sees equals, bit for
    bit, the oracle's restatement of the reference's FP32 arithmetic
    (sequential FMAs in rating order, the (10I+4, 10J) slip, FP32 ridge)."""
    ds = _data.netflix_like_small()
    lam = 0.058
    T0 = cumf.init_factors(ds.n, f, 12)
    X0 = cumf.init_factors(ds.m, f, 13)
    with _als(ds, f, lam, compat_hermitian_bug=1) as h:
        h.set_factors(X=X0, theta=T0)
        deg = np.diff(ds.csr_row_ptr)
        rows = np.array([0, 5, int(np.argmax(deg)), int(np.argmin(deg))], np.int32)
        M, b = h.compat_system(0, rows)
        for k, u in enumerate(rows):
            Mo, bo = O.compat_system(ds.csr_row_ptr, ds.csr_col, ds.csr_val, T0, f, lam, u)
            np.testing.assert_array_equal(M[k], Mo)
            np.testing.assert_array_equal(b[k], bo)
        cols = np.array([0, 7], np.int32)
        M, b = h.compat_system(1, cols)
        for k, v in enumerate(cols):
            Mo, bo = O.compat_system(ds.csc_col_ptr, ds.csc_row, ds.csc_val, X0, f, lam, v)
            np.testing.assert_array_equal(M[k], Mo)
            np.testing.assert_array_equal(b[k], bo)


@pytest.mark.parametrize("f", [10, 100])
def test_compat_half_sweep_matches_oracle(f):
    """Reference-reproducing factors: LU (no pivoting) of the slipped system,
    against the oracle's FP64 LU of the same system, and within FP32 Gram
    rounding of the FP64 compat half-sweep."""
    ds = _data.netflix_like_small()
    lam = 0.058
    T0 = cumf.init_factors(ds.n, f, 14)
    with _als(ds, f, lam, compat_hermitian_bug=1) as h:
        h.set_factors(theta=T0)
        h.update_x()
        X, _ = h.get_factors()
        assert h.stats()["failed_rows"] == 0
    for u in (0, 1, 2, 99):
        Mo, bo = O.compat_system(ds.csr_row_ptr, ds.csr_col, ds.csr_val, T0, f, lam, u)
        np.testing.assert_allclose(X[u], O.lu_solve(Mo, bo), rtol=1e-5, atol=1e-6)
    Xo, _ = O.half_sweep(ds.csr_row_ptr, ds.csr_col, ds.csr_val, T0, lam, compat=True)
    rel = np.linalg.norm(X - Xo, axis=1) / np.linalg.norm(Xo, axis=1)
    assert rel.max() <= 1e-3
    # and it is NOT the clean update
    Xc, _ = O.half_sweep(ds.csr_row_ptr, ds.csr_col, ds.csr_val, T0, lam)
    assert (np.linalg.norm(X - Xc, axis=1) / np.linalg.norm(Xc, axis=1)).max() > 1e-3


def test_compat_env_switch_on_dropin(monkeypatch):
    ds = _data.netflix_like_small()
    f, lam = 10, 0.058
    T0 = cumf.init_factors(ds.n, f, 15)
    monkeypatch.setenv("CUMF_COMPAT_HERMITIAN_BUG", "1")
    X = G.do_als_with_csr(ds.csr_row_ptr, ds.csr_col, ds.csr_val, T0, ds.m, ds.n, f, lam)
    monkeypatch.delenv("CUMF_COMPAT_HERMITIAN_BUG")
    Xo, _ = O.half_sweep(ds.csr_row_ptr, ds.csr_col, ds.csr_val, T0, lam, compat=True)
    rel = np.linalg.norm(X - Xo, axis=1) / np.linalg.norm(Xo, axis=1)
    assert rel.max() <= 1e-3


def _bf16(x):
    """float32 values rounded to bfloat16 (round to nearest even), as float32."""
    b = np.ascontiguousarray(x, np.float32).view(np.uint32)
    b = (b + (((b >> 16) & 1) + 0x7FFF)) & 0xFFFF0000
    return b.view(np.float32)


def test_mfma_bf16_layout():
    out = G.mfma_bf16_layout()
    k = np.arange(32)
    A = np.arange(16)[:, None] + 2 * (k[None, :] % 4)
    B = (k[:, None] % 5) + 3 * np.arange(16)[None, :]
    D = (A @ B).astype(np.float64)
    lane = np.arange(64)
    for r in range(4):
        np.testing.assert_array_equal(out[:, r], D[4 * (lane // 16) + r, lane % 16])


@pytest.mark.parametrize("f", [32, 100])
def test_bf16_gram_matches_oracle_on_rounded_factors(f):
    """CUMF_PREC_BF16_GRAM: the Gram equals the FP64 Gram of the BF16-rounded
    factors to FP32 accumulation error; b (hi + lo columns) likewise."""
    ds = _data.netflix_like_small()
    lam = 0.058
    T0 = cumf.init_factors(ds.n, f, 21)
    with _als(ds, f, lam, precision=G.CUMF_PREC_BF16_GRAM) as h:
        h.set_factors(theta=T0)
        deg = np.diff(ds.csr_row_ptr)
        rows = np.concatenate([np.argsort(-deg)[:3], np.argsort(deg)[:3], [7]]).astype(np.int32)
        D = h.row_gram(0, rows)
    Tr = _bf16(T0)
    for k, u in enumerate(rows):
        A, b = O.row_system(ds.csr_row_ptr, ds.csr_col, ds.csr_val, Tr, f, lam, u)
        scale = np.abs(np.diag(A)).max()
        assert np.abs(D[k, :f, :f] - A).max() <= 2e-5 * scale, u
        bg = D[k, :f, f].astype(np.float64) + D[k, :f, f + 1]
        assert np.abs(bg - b).max() <= 2e-5 * max(np.abs(b).max(), 1.0), u


def test_bf16_half_sweep_matches_oracle_on_rounded_factors():
    ds = _data.netflix_like_small()
    f, lam = 100, 0.058
    T0 = cumf.init_factors(ds.n, f, 22)
    with _als(ds, f, lam, precision=G.CUMF_PREC_BF16_GRAM, split=256) as h:
        h.set_factors(theta=T0)
        h.update_x()
        X1, _ = h.get_factors()
        assert h.stats()["failed_rows"] == 0
    Xo, _ = O.half_sweep(ds.csr_row_ptr, ds.csr_col, ds.csr_val, _bf16(T0), lam)
    rel = np.linalg.norm(X1 - Xo, axis=1) / np.linalg.norm(Xo, axis=1)
    assert rel.max() <= 1e-3


def test_bf16_gram_training_rmse_vs_fp64_oracle():
    """Full training (10,000 x 2,000, f=32, lambda=0.05, 10 iterations) with
    the BF16 Gram: held-out RMSE within 1e-3 of the (unrounded) FP64 oracle."""
    ds = _data.small_zipf()
    f, lam, iters = 32, 0.05, 10
    T0 = cumf.init_factors(ds.n, f, 0)
    _, _, hist = O.als_train(ds, f, lam, iters, T0)
    with _als(ds, f, lam, precision=G.CUMF_PREC_BF16_GRAM) as h:
        h.set_factors(theta=T0)
        h.iterate(iters)
        rm = h.rmse()
    assert abs(rm - hist[-1]) <= 1e-3, (rm, hist[-1])


@pytest.mark.parametrize("f", [1, 3, 4, 10, 63, 100, 141, 255])
@pytest.mark.parametrize("m,n", [(1, 1), (67, 3), (9001, 130)])
def test_factors_round_trip_every_stride(f, m, n):
    """Factors set on a handle come back bit for bit, whatever the padding of
    the device rows (f a multiple of 4 or not), and again after a smaller and
    a larger matrix through the same handle."""
    rng = np.random.default_rng(f * 100003 + m)
    with G.ALS(f, 0.05) as h:
        for mm in (m, max(1, m // 2), m + 5):
            rp = np.arange(mm + 1, dtype=np.int32)
            h.set_ratings(mm, n, rp, rng.integers(0, n, mm), np.ones(mm, np.float32))
            X = rng.standard_normal((mm, f)).astype(np.float32)
            T = rng.standard_normal((n, f)).astype(np.float32)
            h.set_factors(X=X, theta=T)
            X2, T2 = h.get_factors()
            np.testing.assert_array_equal(X2, X)
            np.testing.assert_array_equal(T2, T)


# One FP32 chunk is 16 ratings, two make a matrix step; four buffers up to
# f = 60 (NB <= 4), two above; NB = 1 .. 9.
@pytest.mark.parametrize("f", [4, 12, 27, 44, 60, 76, 92, 100, 120, 140])
@pytest.mark.parametrize("scale", [1.0, 2.0 ** -50, 2.0 ** 50])
def test_fp32_gram_at_chunk_edges(f, scale):
    """The FP32 Gram from split BF16 products against FP64, rating counts at
    every edge of the staging and of the pairs, columns of mixed magnitude.
    Bound per entry, in units of 2^-24 of the sum of the products' sizes: the
    products left out (2^-24 each) and the summation inside a 32-rating step
    (2 ulp = 2^-22 of its size per instruction that adds to the full value)
    are below 8, and each step's addition costs one more.  Below FP32's normal
    range (the smallest scale's smallest columns) a product's low parts may be
    flushed: 2^-126 for each of its six."""
    counts = [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 79, 80, 81, 96, 97, 127, 128, 129, 257, 1000]
    rng = np.random.default_rng(f)
    n = 400
    m = len(counts)
    rp = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    ci = rng.integers(0, n, rp[-1]).astype(np.int32)
    cv = rng.standard_normal(rp[-1]).astype(np.float32)
    T = rng.standard_normal((n, f)) * np.exp2(rng.integers(-12, 13, (1, f))) * scale
    T = T.astype(np.float32)
    with G.ALS(f, 0.0) as h:
        h.set_ratings(m, n, rp, ci, cv)
        h.set_factors(theta=T)
        got = h.row_gram(0, np.arange(m)).astype(np.float64)
    bcol = (f + 3) // 4 * 4
    for u, cnt in enumerate(counts):
        Y = T[ci[rp[u]:rp[u + 1]]].astype(np.float64)
        r = cv[rp[u]:rp[u + 1]].astype(np.float64)
        unit, low = 2.0 ** -24 * (8 + cnt / 32), 6 * cnt * 2.0 ** -126
        for have, want, size in ((got[u][:f, :f], Y.T @ Y, np.abs(Y).T @ np.abs(Y)),
                                 (got[u][:f, bcol], Y.T @ r, np.abs(Y).T @ np.abs(r))):
            fits = size <= 2.0 ** 127  # (past FP32's range an entry is infinite, as any FP32 sum)
            assert np.all(np.abs(have - want)[fits] <= (unit * size + low)[fits]), (f, cnt)


def test_fp32_rows_with_infinities_and_nans_fail_alone():
    """A factor that is not finite, or whose squares overflow, fails the rows
    that read it (x = 0, counted) and no other."""
    f, lam, n = 20, 0.05, 12
    T = cumf.init_factors(n, f, 9)
    T[0, 3], T[1, 5], T[2, 7], T[3, 0] = np.inf, -np.inf, np.nan, np.finfo(np.float32).max
    ci = np.array([[0, 5, 6], [1, 5, 6], [2, 5, 6], [3, 5, 6], [4, 5, 6]], np.int32)
    rp = np.arange(0, 16, 3, dtype=np.int32)
    with G.ALS(f, lam) as h:
        h.set_ratings(5, n, rp, ci.ravel(), np.full(15, 2.0, np.float32))
        h.set_factors(theta=T)
        h.update_x()
        X, _ = h.get_factors()
        assert h.stats()["failed_rows"] == 4
    assert np.all(X[:4] == 0)
    Xo, _ = O.half_sweep(np.array([0, 3], np.int32), ci[4], np.full(3, 2.0, np.float32), T, lam)
    assert np.linalg.norm(X[4] - Xo[0]) <= 1e-5 * np.linalg.norm(Xo[0])


@pytest.mark.parametrize("f", [12, 32, 50, 76, 92, 100, 128, 140])
def test_short_rows_on_both_sides_of_the_dual_line(f):
    """FP32 rows whose n x n system is smaller than the f x f one are solved in
    it; every length up to 97 and both sides of each block edge, against the
    FP64 system on the same factors: relative residual at most 1e-5."""
    lam, n = 0.05, 700
    rng = np.random.default_rng(f)
    counts = np.arange(0, 114)
    m = len(counts)
    rp = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    ci = np.concatenate([rng.choice(n, c, replace=False) for c in counts]).astype(np.int32)
    cv = rng.standard_normal(rp[-1]).astype(np.float32) * 3
    T = cumf.init_factors(n, f, 5)
    with G.ALS(f, lam) as h:
        h.set_ratings(m, n, rp, ci, cv)
        h.set_factors(theta=T)
        h.update_x()
        X, _ = h.get_factors()
        assert h.stats()["failed_rows"] == 0
    assert np.all(X[0] == 0)
    for u in range(1, m):
        Y = T[ci[rp[u]:rp[u + 1]]].astype(np.float64)
        b = Y.T @ cv[rp[u]:rp[u + 1]].astype(np.float64)
        x = X[u].astype(np.float64)
        res = b - Y.T @ (Y @ x) - float(np.float32(lam) * np.float32(counts[u])) * x
        assert np.linalg.norm(res) <= 1e-5 * np.linalg.norm(b), (f, u, np.linalg.norm(res) / np.linalg.norm(b))


@pytest.mark.parametrize("f", [20, 100, 140])
def test_singular_rows_without_a_ridge_fail_as_before(f):
    """lambda = 0 and fewer ratings than f: the f x f system is singular.  Rows
    of unit-vector factors have an exactly zero pivot: x = 0, counted, though
    their n x n system could be solved."""
    n = f
    T = np.eye(n, f, dtype=np.float32)
    rp = np.array([0, 1, 4, 4 + f], np.int32)
    ci = np.concatenate([[3], [1, 2, 5], np.arange(f)]).astype(np.int32)
    cv = np.full(4 + f, 2.0, np.float32)
    with G.ALS(f, 0.0) as h:
        h.set_ratings(3, n, rp, ci, cv)
        h.set_factors(theta=T)
        h.update_x()
        X, _ = h.get_factors()
        assert h.stats()["failed_rows"] == 2
    assert np.all(X[:2] == 0)
    np.testing.assert_allclose(X[2], 2.0, rtol=1e-6)


@pytest.mark.parametrize("f", [13, 14, 29, 45, 61, 77, 93, 94])
def test_rows_of_more_ratings_than_rank_keep_their_system(f):
    """A few more ratings than f, orthonormal factor columns and next to no
    ridge: Y^T Y is the identity (any FP32 solve of it is good to 1e-5, the
    plain path's bar), Y Y^T has rank f < n and is singular but for 1e-6 of a
    ridge."""
    lam = 1e-7
    rng = np.random.default_rng(f)
    counts = list(range(f + 1, f + 8))  # the dual form ends at a block edge up to 3 past f
    n, m = sum(counts), len(counts)
    rp = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    T = np.concatenate([np.linalg.qr(rng.standard_normal((c, f)))[0] for c in counts]).astype(np.float32)
    cv = rng.integers(1, 6, n).astype(np.float32)
    with G.ALS(f, lam) as h:
        h.set_ratings(m, n, rp, np.arange(n, dtype=np.int32), cv)
        h.set_factors(theta=T)
        h.update_x()
        X, _ = h.get_factors()
        assert h.stats()["failed_rows"] == 0
    for u, cnt in enumerate(counts):
        Y = T[rp[u]:rp[u + 1]].astype(np.float64)
        b = Y.T @ cv[rp[u]:rp[u + 1]].astype(np.float64)
        x = X[u].astype(np.float64)
        res = b - Y.T @ (Y @ x) - float(np.float32(lam) * np.float32(cnt)) * x
        assert np.linalg.norm(res) <= 1e-5 * np.linalg.norm(b), (f, cnt, np.linalg.norm(res) / np.linalg.norm(b))


@pytest.mark.parametrize("f", [1, 2, 3, 4, 7, 8, 10, 12])
def test_rows_of_one_rating_at_small_ranks(f):
    """One rating r with factor y: x = r y / (|y|^2 + lambda).  Solved as that
    1 x 1 system it is off by at most 16 * 2^-24: 4 for the products left out
    of the split of |y|^2, 4 for the rounding of its matrix instructions (two
    of full size, one ulp each), 6 for the pivot's reciprocal square root taken
    twice, 2 for the ridge and the last product."""
    m, n, lam = 4000, 2000, 0.05
    rng = np.random.default_rng(f)
    T = (0.3 + rng.standard_normal((n, f))).astype(np.float32) / np.float32(np.sqrt(f))
    ci = rng.integers(0, n, m).astype(np.int32)
    cv = rng.integers(1, 6, m).astype(np.float32)
    with G.ALS(f, lam) as h:
        h.set_ratings(m, n, np.arange(m + 1, dtype=np.int32), ci, cv)
        h.set_factors(theta=T)
        h.update_x()
        X, _ = h.get_factors()
    Y = T[ci].astype(np.float64)
    want = cv[:, None] * Y / ((Y * Y).sum(1, keepdims=True) + float(np.float32(lam)))
    err = np.linalg.norm(X - want, axis=1) / np.linalg.norm(want, axis=1)
    assert err.max() <= 16 * 2.0 ** -24, err.max()


@pytest.mark.parametrize("f", [10, 13])
def test_factor_transfers_allocate_nothing_and_hold_at_seams(f):
    """Both directions of a handle whose factor rows are padded on the device
    (f not a multiple of 4): no device memory is taken after the ratings are
    set, also for the side that was not uploaded, and rows on both sides of a
    32 MB piece of the transfer arrive whole and in place."""
    m, n = 2 * ((32 << 20) // (4 * f)) + 3, 7  # three pieces, the last of three rows
    rp = np.zeros(m + 1, np.int32)
    rp[1:] = 1
    X0 = np.arange(m * f, dtype=np.float32).reshape(m, f) % 8191
    T0 = cumf.init_factors(n, f, 0)

    def free_bytes():
        free, total = C.c_size_t(), C.c_size_t()
        assert G.lib().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value

    with G.ALS(f, 0.05) as h:
        h.set_ratings(m, n, rp, np.zeros(1, np.int32), np.ones(1, np.float32))
        before = free_bytes()
        h.set_factors(theta=T0)
        Xz, T1 = h.get_factors()
        h.set_factors(X=X0)
        X1, _ = h.get_factors()
        assert free_bytes() == before
    assert np.all(Xz == 0)
    np.testing.assert_array_equal(T1, T0)
    np.testing.assert_array_equal(X1, X0)


@pytest.mark.parametrize("f", [12, 13, 14, 15, 16, 29, 30, 31, 45, 46, 47, 61, 62, 63, 77, 78, 79, 93, 94, 95, 109, 110,
                               111, 125, 126, 127, 128])
@pytest.mark.parametrize("solver", [G.CUMF_SOLVER_CHOLESKY, G.CUMF_SOLVER_CG])
def test_bf16_ranks_up_to_a_block_edge(f, solver):
    """BF16 Gram at ranks whose factor columns end one to three columns before
    a 16-column block does: the rating's columns then lie in the block after
    it.  Rows with and without a split; each one's residual against the FP64
    system on the BF16 factors is at most 1e-5 (Cholesky; CG: twice its
    tolerance of 1e-5), as at every other rank."""
    lam, n = 0.05, 900
    rng = np.random.default_rng(f)
    counts = np.array([1, 2, 15, 16, 31, 32, 33, 64, 95, 96, 97, 128, 200, 256, 257, 600, 899])
    m = counts.shape[0]
    rp = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    ci = np.concatenate([rng.choice(n, c, replace=False) for c in counts]).astype(np.int32)
    cv = rng.integers(1, 6, rp[-1]).astype(np.float32)
    T = cumf.init_factors(n, f, 5)
    with G.ALS(f, lam, precision=G.CUMF_PREC_BF16_GRAM, solver=solver, split=256) as h:
        h.set_ratings(m, n, rp, ci, cv)
        h.set_factors(theta=T)
        h.update_x()
        X, _ = h.get_factors()
        assert h.stats()["failed_rows"] == 0
    Tr = _bf16(T)
    for u, cnt in enumerate(counts):
        Y = Tr[ci[rp[u]:rp[u + 1]]].astype(np.float64)
        b = Y.T @ cv[rp[u]:rp[u + 1]].astype(np.float64)
        x = X[u].astype(np.float64)
        res = np.linalg.norm(b - Y.T @ (Y @ x) - float(np.float32(lam) * np.float32(cnt)) * x) / np.linalg.norm(b)
        assert res <= (1e-5 if solver == G.CUMF_SOLVER_CHOLESKY else 2e-5), (f, cnt, res)
