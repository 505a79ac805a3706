"""Mixed batches whose eb_sr products are large run them in a launch of their
own: every product of both launches has the bits of a call of its own, captured
or not, and the batch costs what its two halves cost."""
import numpy as np
import pytest

import segtaco_amd as S
from gpu_util import DeviceCSR, dense_dev, run_spmm, stream_ptr, torch

pytestmark = pytest.mark.gpu


def _matrix(dtype, rows=60000, mean=16.0):
    pos, crd, vals = S.gen_csr(S.GEN_POWERLAW, 3, rows, rows, mean=mean)[:3]
    return DeviceCSR(pos, crd, vals, rows, dtype=dtype), pos


def _small(dtype):
    rng = np.random.default_rng(5)
    lens = rng.integers(0, 30, 3000)
    pos = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    crd = np.concatenate([np.sort(rng.choice(500, int(l), replace=False)) for l in lens])
    return DeviceCSR(pos, crd.astype(np.int32), rng.uniform(-1, 1, len(crd)).astype(np.float32),
                     500, dtype=dtype), pos


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_parts_have_the_bits_of_single_calls(dtype):
    t = torch()
    big, big_pos = _matrix(dtype)
    small, small_pos = _small(dtype)
    none = DeviceCSR(np.zeros(78, np.int32), np.zeros(0, np.int32), np.zeros(0, np.float32), 9,
                     dtype=dtype)
    bd = S.DTYPES[dtype]
    rng = np.random.default_rng(7)
    B = {n: dense_dev(rng.uniform(-1, 1, (big.K, n)), dtype) for n in (16, 32, 128)}
    b = {n: dense_dev(rng.uniform(-1, 1, (small.K, n)), dtype) for n in (1, 24)}
    E = S.make_plan("eb_sr", tile=128, comp_threshold=0)
    # an rb_sr, an eb_pr at one column, an eb_sr of the widest slices, an empty and a
    # no-column product between the large ones
    products = [(big, big_pos, B[16], 16, E), (small, small_pos, b[24], 24, S.make_plan("rb_sr"))]
    products += [(big, big_pos, B[32], 32, E)] * 17
    products += [(small, small_pos, b[1], 1, S.make_plan("eb_pr", tile=64)),
                 (none, np.zeros(78, np.int32), b[24], 24, E),
                 (small, small_pos, b[24], 24, S.make_plan("eb_sr", tile=8, col_lanes=2)),
                 (big, big_pos, B[128], 128, E)]
    assert big.nnz * 18 > 1 << 24
    outs, items = [], []
    for A, pos, Bd, n, p in products:
        outs.append(t.full((A.M, n), float("nan"), dtype=t.float32, device="cuda"))
        items.append(S.batch_item(A.desc, Bd.data_ptr(), n, outs[-1].data_ptr(), n, n, p, pos))
    want = {}
    for A, pos, Bd, n, p in products:
        if A.nnz and (id(A), n, p.schedule) not in want:
            want[id(A), n, p.schedule] = run_spmm(A, Bd, n, p, b_dtype=dtype)
    batch = S.Batch(items, dtype, stream_ptr())
    alone = [S.Batch([i], dtype, stream_ptr()) for i in items]
    assert all(a.units() > 0 for a in alone)
    assert batch.units() == sum(a.units() for a in alone)
    for a in alone:
        a.destroy()
    batch.capture()
    for step in range(4):
        for o in outs:
            o.fill_(float("nan"))
        if step % 2 == 0:
            batch.replay(stream_ptr())
        else:
            batch.run(stream_ptr())
        t.cuda.synchronize()
        for o, (A, pos, Bd, n, p) in zip(outs, products):
            if A.nnz == 0:
                assert not o.any()
            else:
                assert t.equal(o.view(t.int32), want[id(A), n, p.schedule].view(t.int32))
    batch.destroy()


def test_mixed_batch_costs_its_halves():
    t = torch()
    big, big_pos = _matrix("bf16")
    small, small_pos = _small("bf16")
    rng = np.random.default_rng(9)
    B = [dense_dev(rng.uniform(-1, 1, (big.K, 32)), "bf16") for _ in range(4)]
    b = dense_dev(rng.uniform(-1, 1, (small.K, 24)), "bf16")
    E, R = S.make_plan("eb_sr", tile=128), S.make_plan("rb_sr")
    C = [t.empty((big.M, 32), dtype=t.float32, device="cuda") for _ in range(40)]
    c = t.empty((small.M, 24), dtype=t.float32, device="cuda")
    large = [S.batch_item(big.desc, B[i % 4].data_ptr(), 32, C[i].data_ptr(), 32, 32, E, big_pos)
             for i in range(40)]
    other = [S.batch_item(small.desc, b.data_ptr(), 24, c.data_ptr(), 24, 24, R, small_pos)]

    def best_us(items):
        batch = S.Batch(items, "bf16", stream_ptr())
        batch.capture()
        batch.replay(stream_ptr())
        best = 1e9
        for _ in range(8):
            e0, e1 = t.cuda.Event(enable_timing=True), t.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(4):
                batch.replay(stream_ptr())
            e1.record()
            t.cuda.synchronize()
            best = min(best, e0.elapsed_time(e1) * 250)
        batch.destroy()
        return best

    halves, mixed = best_us(large) + best_us(other), best_us(large + other)
    print(f"[parts] halves {halves:.0f} us, mixed {mixed:.0f} us", flush=True)
    assert mixed < 1.12 * halves
