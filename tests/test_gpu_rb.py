"""Row-balanced schedules at the edges of their batches: rows of 0, 1, one
below, at and above the entries of a batch or step, one long (compensated)
row, the same lengths again up to the last stored entry, with and without
stored values, in products of few and of many workgroups. Whole-number inputs,
so every summation order gives the exact result."""
import numpy as np
import pytest

import segtaco_amd as S
from gpu_util import DeviceCSR, dense_dev, run_spmm, stream_ptr, torch

pytestmark = pytest.mark.gpu

EDGES = [0, 1, 7, 8, 9, 15, 16, 17, 2, 31, 33, 63, 64, 65, 0, 129, 3, 1100, 5, 0]


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("values", [True, False])
@pytest.mark.parametrize("M", [len(EDGES), 66000])
@pytest.mark.parametrize("sched,N", [("rb_sr", 1), ("rb_sr", 6), ("rb_sr", 40), ("rb_pr", 1),
                                     ("rb_pr", 3), ("rb_pr", 8), ("rb_pr", 40)])
def test_edges(sched, N, M, values, dtype):
    rng = np.random.default_rng(N)
    K = 2000
    lens = np.full(M, 2)
    lens[:len(EDGES)] = EDGES
    lens[M - len(EDGES):] = EDGES
    pos = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    crd = np.concatenate([np.sort(rng.choice(K, int(l), replace=False)) if l > 2
                          else np.arange(l) * 7 for l in lens]).astype(np.int32)
    vals = rng.integers(-3, 4, len(crd)).astype(np.float32) if values else None
    B = rng.integers(-4, 5, (K, N)).astype(np.float32)
    A = DeviceCSR(pos, crd, vals, K, dtype=dtype)
    Bd = dense_dev(B, dtype)
    plan = S.plan_resolve(A.desc, N, S.DTYPES[dtype], S.make_plan(sched), N, N)
    print(f"[rb] {sched} N={N} M={M} values={values} {dtype}", flush=True)
    C = run_spmm(A, Bd, N, plan, b_dtype=dtype).cpu().numpy()
    e = B[crd] if vals is None else B[crd] * vals[:, None]
    want = np.concatenate([np.zeros((1, N)), np.cumsum(e, axis=0)])
    want = (want[pos[1:]] - want[pos[:-1]]).astype(np.float32)
    assert np.array_equal(C, want)
    t = torch()
    D = t.full((M, N), float("nan"), dtype=t.float32, device="cuda")
    batch = S.Batch([S.batch_item(A.desc, Bd.data_ptr(), N, D.data_ptr(), N, N, plan, pos)],
                    dtype, stream_ptr())
    batch.run(stream_ptr())
    t.cuda.synchronize()
    assert np.array_equal(D.cpu().numpy(), want)
    batch.destroy()
