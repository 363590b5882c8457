"""k_mttkrp_rows (kernel 14) at the edges of its lane layouts and rounds,
against the oracle: ranks around every change of columns per lane and lanes
per nonzero, chunks of one and of several rounds, rows that end inside,
across and at the end of a round."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# FP64 sums of at most a few thousand terms; FP32: 2^-24 per operation over
# the same; BF16 factors are exact in FP32, the oracle takes the rounded ones
TOL = {0: 1e-12, 1: 2e-6, 2: 2e-6}


def mttkrp(B, dev, U, m, dtype, tpw):
    R = U[0].shape[1]
    F = [B.DeviceArray.from_numpy(u, dtype) for u in U]
    out = B.DeviceArray((U[m].shape[0], R), B.F64 if dtype == 0 else B.F32)
    B.mttkrp(dev, m, R, F, out, factor_dtype=dtype, kernel=B.K_SORTED, thread_cf=tpw)
    return out.numpy(), [f.numpy() for f in F]


@pytest.mark.parametrize("dtype", [0, 1, 2])
@pytest.mark.parametrize("dims,nnz", [((4000, 600, 500), 40000), ((3, 700, 40, 90), 9000), ((5000, 3000), 20000),
                                      ((9, 80, 7, 60, 5), 12000), ((30, 40, 20), 57)])
def test_ranks_and_rounds(B, O, gpu, dtype, dims, nnz):
    t = B.Coo.generate(dims, nnz, gen_rank=3, value_kind=1, seed=5)
    at = O.Alto(dims, t.cidx, t.vals, nprtn=4)
    dev = B.DeviceTensor(B.encode(t), value_dtype=B.F64 if dtype == 0 else B.F32)
    for rank in (1, 3, 4, 5, 8, 9, 16, 17, 31, 33, 64, 65, 130):
        rng = np.random.default_rng(rank)
        U = [rng.random((d, rank)) for d in dims]
        for tpw in (1, 16):
            for m in range(len(dims)):
                got, held = mttkrp(B, dev, U, m, dtype, tpw)
                want = at.mttkrp(held, m)
                e = np.linalg.norm(got - want) / np.linalg.norm(want)
                assert e <= TOL[dtype], (dims, dtype, rank, tpw, m, e)
    dev.free()


def test_infinities_stay_in_their_rows(B, O, gpu):
    """Positions past a slot's share gather nothing: an infinite factor row
    reaches only the output rows that meet it."""
    dims, R = (500, 300, 200), 20
    t = B.Coo.generate(dims, 7000, gen_rank=3, seed=9)
    at = O.Alto(dims, t.cidx, t.vals, nprtn=4)
    dev = B.DeviceTensor(B.encode(t), value_dtype=B.F32)
    U = [np.random.default_rng(m).random((d, R)).astype(np.float32).astype(np.float64) for m, d in enumerate(dims)]
    want = at.mttkrp(U, 0)
    hit = np.zeros(dims[0], bool)
    hit[t.cidx[0][t.cidx[1] == 7].astype(int)] = True
    assert 0 < hit.sum() < dims[0]
    U[1][7] = np.inf
    for tpw in (1, 2, 16):
        got, _ = mttkrp(B, dev, U, 0, 1, tpw)
        assert np.all(np.isinf(got[hit])) and np.all(np.isfinite(got[~hit]))
        assert np.linalg.norm(got[~hit] - want[~hit]) <= 2e-6 * np.linalg.norm(want[~hit])
    dev.free()


@pytest.mark.parametrize("rank,dtype", [(32, 0), (33, 1), (32, 1)])
def test_default_chunk_lengths_of_large_tensors(B, O, gpu, rank, dtype):
    """Just past 2^22 nonzeros, from where copies are grouped by XCD tiles:
    output rows of more than 128 bytes in a mode of many rows (untiled, chunks
    of 2 tiles of 64) and in modes of long ones (8, the kernel's long rounds), a
    most frequent row of over 32768 nonzeros (pieces of 2048), and 128-byte
    rows (2 everywhere)."""
    dims, nnz = (100_000, 1500, 900), (1 << 22) + 4321
    t = B.Coo.generate(dims, nnz, zipf=(0.3, 1.1, 0.0), gen_rank=4, seed=22, topup=True)
    assert t.nnz == nnz and np.bincount(t.cidx[1].astype(int)).max() > 32768
    at = O.Alto(dims, t.cidx, t.vals, nprtn=8)
    dev = B.DeviceTensor(B.encode(t), value_dtype=B.F64 if dtype == 0 else B.F32)
    U = [np.random.default_rng(m).random((d, rank)) for m, d in enumerate(dims)]
    for m in range(3):
        got, held = mttkrp(B, dev, U, m, dtype, 0)
        # (FP32 copies are in fiber order here, whose outer factors L2 holds)
        assert (dev.row_copy(m, rank, dtype)["tiles"] > 1) == (m > 0 and dtype == 0)
        want = at.mttkrp(held, m)
        e = np.linalg.norm(got - want) / np.linalg.norm(want)
        assert e <= TOL[dtype], (rank, dtype, m, e)
    dev.free()


def test_default_chunk_length_with_a_hot_row(B, gpu):
    """A very frequent row (7% of 165M nonzeros) lengthens no chunks: the
    default runs within 10% of the best of 2 and 8 tiles (16 tiles: 22% more)."""
    dims, rank = (600_000, 400_000, 500_000), 32
    dev = B.DeviceTensor.generate(dims, 165_000_000, zipf=(1.0, 1.0, 1.0), gen_rank=20, value_kind=1,
                                  seed=1005, topup=True)
    F = [B.DeviceArray((d, rank)) for d in dims]
    out = B.DeviceArray((dims[1], rank))
    ms = {tpw: min(B.mttkrp_time(dev, 1, rank, F, out, kernel=B.K_SORTED, reps=3, thread_cf=tpw)[0] for _ in range(3))
          for tpw in (0, 2, 8)}
    dev.free()
    assert ms[0] <= 1.1 * min(ms[2], ms[8]), ms


def test_order_switch_after_the_copy_changes_nothing(B, gpu, monkeypatch):
    """BLCO_FIBERS chooses the order of a copy, and windows for that copy, when
    it is built; set later it reaches no launch."""
    monkeypatch.delenv("BLCO_FIBERS", raising=False)
    dims = (3000, 2000, 500)
    dev = B.DeviceTensor.generate(dims, 2_000_000, zipf=(0.9, 0.9, 0.0), gen_rank=4, seed=3, topup=True,
                                  value_dtype=B.F32)
    for switch, rank in ((None, 32), ("0", 16)):
        if switch:
            monkeypatch.setenv("BLCO_FIBERS", switch)
        F = [B.DeviceArray((d, rank), B.F32) for d in dims]
        out = B.DeviceArray((dims[0], rank), B.F32)
        B.mttkrp(dev, 0, rank, F, out, factor_dtype=B.F32, kernel=B.K_SORTED, thread_cf=1)
        assert dev.rows_plan(0, rank, B.F32) == (1, False, 0)
    dev.free()


@pytest.mark.parametrize("nnz", [3_000_000, (1 << 22) + 99])
def test_wide_factors_with_a_long_row(B, O, gpu, nnz):
    """A factor of more than 2 GiB (64-bit offsets) beside a mode whose most
    frequent row has over 32768 nonzeros, below and above the size from which
    that row's pieces are longer than the chunks."""
    dims, rank = (17_000_000, 2000, 300), 32
    assert dims[0] * rank * 4 >= 1 << 31
    t = B.Coo.generate(dims, nnz, zipf=(0.9, 1.0, 0.0), gen_rank=2, seed=17, topup=True)
    assert np.bincount(t.cidx[1].astype(int)).max() > 32768
    dev = B.DeviceTensor(B.encode(t), value_dtype=B.F32)
    U = [np.random.default_rng(m).random((d, rank), dtype=np.float32) for m, d in enumerate(dims)]
    for m in (1, 2):
        got, _ = mttkrp(B, dev, U, m, 1, 0)
        want = np.zeros((dims[m], rank))
        for at in range(0, nnz, 1 << 20):
            i = [c[at:at + (1 << 20)].astype(np.int64) for c in t.cidx]
            p = t.vals[at:at + (1 << 20), None] * U[0][i[0]]
            p *= U[3 - m][i[3 - m]]
            for c in range(rank):
                want[:, c] += np.bincount(i[m], weights=p[:, c], minlength=dims[m])
        e = np.linalg.norm(got - want) / np.linalg.norm(want)
        assert e <= TOL[1], (nnz, m, e)
    dev.free()


@pytest.mark.parametrize("dims,nnz,tpw", [((160, 6000, 5000), 2_000_000, 4), ((300, 3000, 2000), 4_300_000, 16)])
@pytest.mark.parametrize("dtype", [1, 2])
def test_float_error_of_rows_cut_into_pieces(B, O, gpu, dims, nnz, tpw, dtype):
    """Every piece of a row ends in a float add to the output.  Rows of 12,500
    and 14,300 nonzeros are cut no finer than by chunks of the length that
    leaves 4096 to 8192 of them (`tpw` tiles): the default's error against the
    oracle is that of those chunks, to the tenth that the order of the adds
    moves it by at most (pieces of 256 nonzeros: 1.4 and 1.8 times)."""
    R = 32
    t = B.Coo.generate(dims, nnz, gen_rank=3, value_kind=0, seed=12)
    at = O.Alto(dims, t.cidx, t.vals, nprtn=8)
    dev = B.DeviceTensor(B.encode(t), value_dtype=B.F32)
    U = [np.random.default_rng(m).random((d, R)) for m, d in enumerate(dims)]
    error = {}
    for cf in (0, tpw):
        got, held = mttkrp(B, dev, U, 0, dtype, cf)
        want = at.mttkrp(held, 0)
        error[cf] = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert error[0] <= 1.1 * error[tpw], (dims, dtype, error)
    dev.free()
