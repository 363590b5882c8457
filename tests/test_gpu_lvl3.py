"""lvl3 over the row gathers (k_mttkrp_lvl3_rows) at the edges of its lane
layouts and rounds, against the oracle: ranks around every change of layout,
one to a hundred output rows, chunks shorter than a round, streamed units."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = {0: 1e-12, 1: 2e-6, 2: 2e-6}  # BF16 factors are exact in FP32; the oracle takes the rounded ones


@pytest.mark.parametrize("dtype", [0, 1, 2])
@pytest.mark.parametrize("dims,nnz,stream", [((1, 300, 200), 3000, False), ((100, 90, 80, 7), 20000, False),
                                             ((24, 5000), 50, False), ((33, 600, 500), 30000, True)])
def test_lvl3_rows(B, O, gpu, dtype, dims, nnz, stream):
    t = B.Coo.generate(dims, nnz, gen_rank=3, value_kind=1, seed=6)
    at = O.Alto(dims, t.cidx, t.vals, nprtn=4)
    dev = B.DeviceTensor(B.encode(t), value_dtype=B.F64 if dtype == 0 else B.F32, stream_data=stream,
                         slot_nnz=8192 if stream else 0)
    for rank in (1, 4, 5, 8, 10, 16, 17, 32, 33, 48, 60):
        rng = np.random.default_rng(rank)
        F = [B.DeviceArray.from_numpy(rng.random((d, rank)), dtype) for d in dims]
        for nprtn in (1, 3):
            out = B.DeviceArray((dims[0], rank), B.F64 if dtype == 0 else B.F32)
            B.mttkrp(dev, 0, rank, F, out, factor_dtype=dtype, kernel=B.K_LVL3, nprtn=nprtn)
            want = at.mttkrp([f.numpy() for f in F], 0)
            e = np.linalg.norm(out.numpy() - want) / np.linalg.norm(want)
            assert e <= TOL[dtype], (dims, dtype, rank, nprtn, e)
    dev.free()


@pytest.mark.parametrize("dtype", [1, 2])
@pytest.mark.parametrize("nnz", [40_000, 300_000, 3_300_000])
@pytest.mark.parametrize("rows", [1, 3, 24, 100])
def test_lvl3_float_error(B, O, gpu, dtype, nnz, rows):
    """Sums of positive terms in a float output.  A workgroup's sums are
    doubles; its one add per element rounds at k / G of the final sum in the
    k-th of G adds, 2^-24 / sqrt(3) of that at most in root mean square: 2^-24
    sqrt(G) / 3 over all, of G = max(16, nnz / 16384) workgroups, and half a
    unit for the products' and the last rounding."""
    dims = (rows, 6100, 4500)
    t = B.Coo.generate(dims, nnz, gen_rank=3, value_kind=0, seed=8)
    at = O.Alto(dims, t.cidx, t.vals, nprtn=4)
    dev = B.DeviceTensor(B.encode(t), value_dtype=B.F32)
    rng = np.random.default_rng(rows)
    bound = 2.0 ** -24 * (0.5 + np.sqrt(max(16, -(-nnz // 16384))) / 3)
    for rank in (10, 32):
        F = [B.DeviceArray.from_numpy(rng.random((d, rank)), dtype) for d in dims]
        out = B.DeviceArray((dims[0], rank), B.F32)
        B.mttkrp(dev, 0, rank, F, out, factor_dtype=dtype, kernel=B.K_LVL3)
        want = at.mttkrp([f.numpy() for f in F], 0)
        e = np.linalg.norm(out.numpy() - want) / np.linalg.norm(want)
        assert e <= bound, (rows, nnz, dtype, rank, e, bound)
    dev.free()


@pytest.mark.parametrize("rows,rank,dtype", [(12288, 1, 1), (6144, 2, 1), (6144, 2, 2), (3072, 2, 0), (16, 64, 1), (3, 4096, 1)])
def test_lvl3_largest_output(B, O, gpu, rows, rank, dtype):
    """Outputs of 48 KB, the most that kernel 3 takes: up to 144 KB of LDS as
    doubles with odd row strides."""
    dims = (rows, 300, 200)
    t = B.Coo.generate(dims, 30000, gen_rank=3, value_kind=0, seed=9)
    at = O.Alto(dims, t.cidx, t.vals, nprtn=4)
    dev = B.DeviceTensor(B.encode(t), value_dtype=B.F64 if dtype == 0 else B.F32)
    rng = np.random.default_rng(rank)
    F = [B.DeviceArray.from_numpy(rng.random((d, rank)), dtype) for d in dims]
    out = B.DeviceArray((dims[0], rank), B.F64 if dtype == 0 else B.F32)
    B.mttkrp(dev, 0, rank, F, out, factor_dtype=dtype, kernel=B.K_LVL3)
    want = at.mttkrp([f.numpy() for f in F], 0)
    e = np.linalg.norm(out.numpy() - want) / np.linalg.norm(want)
    assert e <= TOL[dtype], (rows, rank, dtype, e)
    dev.free()
