"""The batched kernel is chosen by the schedules of the products: eb_sr in
slices of up to four columns alone, all schedules, or those and the N = 1 form
of eb_pr. An eb_sr product has to give the same bits in each and in a call of
its own, whatever slice width and lanes its plan names."""
import numpy as np
import pytest

import segtaco_amd as S
from gpu_util import DeviceCSR, dense_dev, run_spmm, stream_ptr, torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("N,kw", [(16, {}), (64, {}), (128, {}), (264, {}), (64, dict(vec=8)),
                                  (64, dict(vec=8, col_lanes=2)), (64, dict(vec=1)),
                                  (66, dict(vec=2, col_lanes=4)), (70, {}), (129, {})],
                         ids=lambda v: str(v) if isinstance(v, int) else str(list(v.items())))
def test_forms(N, kw, dtype):
    if dtype == "f32" and kw.get("vec") == 8:
        pytest.skip("FP32 slices hold up to four columns")
    t = torch()
    rng = np.random.default_rng(N)
    M, K = 3000, 500
    lens = rng.integers(0, 30, M)
    lens[[7, 1500]] = [0, 480]
    pos = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    crd = np.concatenate([np.sort(rng.choice(K, int(l), replace=False)) for l in lens])
    vals = rng.uniform(-1, 1, len(crd)).astype(np.float32)
    A = DeviceCSR(pos, crd.astype(np.int32), vals, K, dtype=dtype)
    B = dense_dev(rng.uniform(-1, 1, (K, N)), dtype)
    x = dense_dev(rng.uniform(-1, 1, (K, 1)), dtype)
    plan = S.plan_resolve(A.desc, N, S.DTYPES[dtype], S.make_plan("eb_sr", tile=64, **kw), N, N)
    rb = S.plan_resolve(A.desc, N, S.DTYPES[dtype], S.make_plan("rb_sr"), N, N)
    sv = S.plan_resolve(A.desc, 1, S.DTYPES[dtype], S.make_plan("eb_pr", tile=64), 1, 1)
    products = [(B, N, plan), (B, N, rb), (x, 1, sv)]
    print(f"[forms] N={N} {kw} {dtype}", flush=True)
    want = [run_spmm(A, b, n, p, b_dtype=dtype).cpu().numpy() for b, n, p in products]
    for count in (1, 2, 3):
        outs, items = [], []
        for b, n, p in products[:count]:
            outs.append(t.full((M, n), float("nan"), dtype=t.float32, device="cuda"))
            items.append(S.batch_item(A.desc, b.data_ptr(), n, outs[-1].data_ptr(), n, n, p, pos))
        batch = S.Batch(items, dtype, stream_ptr())
        batch.run(stream_ptr())
        t.cuda.synchronize()
        for o, w in zip(outs, want):
            assert np.array_equal(o.cpu().numpy().view(np.uint32), w.view(np.uint32))
        batch.destroy()
