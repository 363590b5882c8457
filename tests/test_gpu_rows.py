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
