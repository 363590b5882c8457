"""The ALS update at the edges of its kernels: the factorisation's register
and LDS forms over ranks, updates whose partial sums need a fold and ones
that do not in one batch, and factors read back between sweeps."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [0, 1])
def test_solve_over_ranks(B, gpu, dtype):
    """U = M V^{-1} against numpy; V of a condition number below 1e4, so FP64
    errors stay below 1e4 * 2^-53 * rank and FP32 ones at the rounding of U."""
    for R in (1, 2, 15, 16, 17, 31, 32, 33, 48, 49, 64):
        rng = np.random.default_rng(R)
        grams = [u.T @ u for u in (rng.standard_normal((4 * R + 9, R)) for _ in range(3))]
        for rows in (1, 17, 4099):
            M = rng.standard_normal((rows, R))
            if dtype == 1:
                M = M.astype(np.float32).astype(np.float64)
            G = [B.DeviceArray.from_numpy(g) for g in grams]
            Md = B.DeviceArray.from_numpy(M, dtype)
            U = B.DeviceArray((rows, R), dtype)
            assert B.solve(G, 1, R, Md, U, dtype, rows) == 0
            want = np.linalg.solve(grams[0] * grams[2], M.T).T
            e = np.linalg.norm(U.numpy() - want) / np.linalg.norm(want)
            assert e <= (1e-10 if dtype == 0 else 1e-6), (R, rows, e)


@pytest.mark.parametrize("precision", [0, 1])
def test_batch_of_long_and_short_modes(B, gpu, precision):
    """Modes above and below the 8192 rows whose partial sums are folded
    first, orders 2 to 4, odd rank: every tensor as decomposed alone."""
    shapes = [((9001, 40, 300), 60000), ((50, 60, 70, 30), 20000), ((8193, 100), 30000), ((20, 30, 40), 4000)]
    R, iters = 7, 4
    devs, U0 = [], []
    for k, (dims, nnz) in enumerate(shapes):
        t = B.Coo.generate(dims, nnz, gen_rank=3, value_kind=1, seed=40 + k)
        devs.append(B.DeviceTensor(B.encode(t), value_dtype=precision))
        U0.append(B.init_factors(900 + k, dims, R))
    bt = B.Batch(devs)
    tol = 1e-9 if precision == 0 else 1e-3
    for _ in range(2):  # the second call finds its chunk lists
        U, lam, fits, its, _ = bt.cpals(U0, R, max_iters=iters, precision=precision)
        for k, dev in enumerate(devs):
            Us, ls, fs = B.cpals(dev, U0[k], R, iters, precision=precision)
            assert its[k] == iters and abs(fits[k] - fs[-1]) <= tol
            for a, b in zip(U[k], Us):
                assert np.linalg.norm(a - b) <= tol * np.linalg.norm(b), k
            assert np.linalg.norm(lam[k] - ls) <= tol * np.linalg.norm(ls)
    bt.free()
    for d in devs:
        d.free()


@pytest.mark.parametrize("graph", [False, True])
def test_factors_read_between_sweeps(B, gpu, graph):
    """get() borrows the MTTKRP buffer: the sweeps after it see it cleared."""
    dims, R = (700, 300, 200), 9
    t = B.Coo.generate(dims, 30000, gen_rank=3, value_kind=1, seed=3)
    dev = B.DeviceTensor(B.encode(t))
    U0 = B.init_factors(5, dims, R)
    whole = B.CpAls(dev, U0, R, use_graph=graph)
    want = whole.iterate(6)
    s = B.CpAls(dev, U0, R, use_graph=graph)
    got = []
    for _ in range(3):
        got.extend(s.iterate(2))
        s.get()
    assert np.allclose(got, want, rtol=0, atol=1e-10)
    for a, b in zip(s.get()[0], whole.get()[0]):
        assert np.linalg.norm(a - b) <= 1e-9 * np.linalg.norm(b)
    dev.free()


def test_iterate_after_a_failed_sweep(B, gpu):
    """A sweep that an error ended (here values of the wrong type) leaves F to be
    formed anew: the solver goes on as one that never failed."""
    dims, R = (700, 300, 200), 9
    t = B.Coo.generate(dims, 30000, gen_rank=3, value_kind=0, seed=4)
    dev = B.DeviceTensor(B.encode(t))
    U0 = B.init_factors(6, dims, R)
    whole = B.CpAls(dev, U0, R)
    want = whole.iterate(5)
    s = B.CpAls(dev, U0, R)
    got = list(s.iterate(2))
    dev.set_value_dtype(B.F32)  # whole numbers: exact there and back
    with pytest.raises(B.BlcoError):
        s.iterate(1)
    dev.set_value_dtype(B.F64)
    got.extend(s.iterate(3))
    assert np.allclose(got, want, rtol=0, atol=1e-10)
    for a, b in zip(s.get()[0], whole.get()[0]):
        assert np.linalg.norm(a - b) <= 1e-9 * np.linalg.norm(b)
    dev.free()


def test_step_calls_from_threads(B, gpu):
    """The stand-alone step calls share idle scratch between calls, not between
    calls that run at the same time: threads with sizes and streams of their
    own."""
    import ctypes
    import threading

    create = B.lib().hipStreamCreate  # of the HIP runtime that the library is linked to
    create.restype = ctypes.c_int
    ran, wrong = [], []

    def work(k):
        R, rows = 5 + 9 * k, 3000 * (k + 1) + k
        rng = np.random.default_rng(k)
        U, M = rng.standard_normal((rows, R)), rng.standard_normal((rows, R))
        grams = [u.T @ u for u in (rng.standard_normal((4 * R + 9, R)) for _ in range(2))]
        st = ctypes.c_void_p()
        assert create(ctypes.byref(st)) == 0
        Ud, Md = B.DeviceArray.from_numpy(U), B.DeviceArray.from_numpy(M)
        Gd, X = B.DeviceArray((R, R)), B.DeviceArray((rows, R))
        gd = [B.DeviceArray.from_numpy(g) for g in grams]
        for _ in range(20):
            B.gram(Ud, B.F64, rows, R, Gd, stream=st.value)
            B.solve(gd + [Gd], 2, R, Md, X, B.F64, rows, stream=st.value)
            want = np.linalg.solve(grams[0] * grams[1], M.T).T
            if np.linalg.norm(Gd.numpy() - U.T @ U) > 1e-12 * np.linalg.norm(U.T @ U) * np.sqrt(rows) or \
               np.linalg.norm(X.numpy() - want) > 1e-10 * np.linalg.norm(want):
                wrong.append(k)
        ran.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(5)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert sorted(ran) == list(range(5)) and not wrong
