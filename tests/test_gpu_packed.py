"""Streamed tensors, whose words cross the host link packed per fine chunk of
1024 nonzeros (k_unpack): one nonzero (no bits at all), chunk edges, fields of
no bits and of many, blocks whose last chunk is short, several units a pass,
and words too wide to pack.  Against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-12  # the FP64 MTTKRP tolerance of the other kernels


@pytest.mark.parametrize("dims,nnz,max_block", [
    ((7, 5, 3), 1, 0),
    ((60, 50, 40), 1023, 0),
    ((60, 50, 40), 1024, 0),
    ((60, 50, 40), 1025, 0),
    ((5000, 1, 3000), 9000, 0),
    ((900, 800, 700, 5), 30011, 3001),
    ((2 ** 21, 2 ** 20, 2 ** 20), 6000, 0),
])
def test_streamed_words(B, O, gpu, dims, nnz, max_block):
    t = B.Coo.generate(dims, nnz, gen_rank=3, value_kind=1, seed=11)
    h = B.encode(t, max_block_size=max_block) if max_block else B.encode(t)
    at = O.Alto(dims, t.cidx, t.vals, nprtn=4)
    dev = B.DeviceTensor(h, stream_data=True, slot_nnz=4096)
    rng = np.random.default_rng(12)
    U = [rng.random((d, 8)) for d in dims]
    F = [B.DeviceArray.from_numpy(u) for u in U]
    for kernel in (B.K_BATCHED, B.K_BATCHED2, B.K_ATOMIC):
        for m in range(len(dims)):
            out = B.DeviceArray((dims[m], 8), B.F64)
            B.mttkrp(dev, m, 8, F, out, kernel=kernel)
            want = at.mttkrp(U, m)
            assert np.linalg.norm(out.numpy() - want) <= TOL * np.linalg.norm(want), (kernel, m)
    dev.free()


@pytest.mark.parametrize("dims,nnz,max_block,slot", [
    ((3000, 2000, 1000), 2_600_000, 0, 0),          # one block in two equal units
    ((3000, 2000, 1000), 2_600_000, 0, 500_000),    # in six, as small as the slots ask
    ((3000, 2000, 1000), 2_600_000, 2_300_000, 0),  # a large block that little follows, then a small one
    ((3000, 2000, 1000), 2_600_000, 1_000_000, 0),  # blocks that stay whole
    ((16000, 16000, 16000, 4000, 4000), 2_200_000, 0, 0),  # 66 bits: blocks of uneven sizes, words not packed
])
def test_streamed_units(B, O, gpu, dims, nnz, max_block, slot):
    t = B.Coo.generate(dims, nnz, zipf=[0.5] * len(dims), gen_rank=3, value_kind=1, seed=13, topup=True)
    h = B.encode(t, max_block_size=max_block) if max_block else B.encode(t)
    at = O.Alto(dims, t.cidx, t.vals, nprtn=8)
    dev = B.DeviceTensor(h, stream_data=True, slot_nnz=slot)
    U = [np.random.default_rng(m).random((d, 8)) for m, d in enumerate(dims)]
    F = [B.DeviceArray.from_numpy(u) for u in U]
    want = at.mttkrp(U, 1)
    for kernel in (B.K_BATCHED, B.K_BATCHED2, B.K_ATOMIC):
        for _ in range(2):  # the second pass meets both slots used
            out = B.DeviceArray((dims[1], 8))
            B.mttkrp(dev, 1, 8, F, out, kernel=kernel)
            e = np.linalg.norm(out.numpy() - want) / np.linalg.norm(want)
            assert e <= TOL, (dims, nnz, max_block, slot, kernel, e)
    dev.free()
