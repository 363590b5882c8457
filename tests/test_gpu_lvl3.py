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
