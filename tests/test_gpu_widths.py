"""Widths that no wide vector divides: a row's columns are taken in wider
slices, the last one moved back to end at N. Every schedule, at widths one off
the slice and panel sizes, odd leading dimensions, on products large enough to
take the wide slices and on one that keeps narrow ones: within 1e-5 of the
FP64 oracle, nothing written outside [0, N), and the same bits in a batch."""
import numpy as np
import pytest

import oracle as O
import segtaco_amd as S
from gpu_util import DeviceCSR, dense_dev, run_spmm, stream_ptr, torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("N", [9, 31, 33, 65, 67, 127, 131, 257])
@pytest.mark.parametrize("sched,kw", [("rb_sr", {}), ("rb_pr", {}), ("eb_sr", dict(tile=8)),
                                      ("eb_pr", dict(tile=8)), ("eb_cs", {}),
                                      ("rb_sr", dict(col_lanes=2)), ("bd", {})],
                         ids=lambda v: v if isinstance(v, str) else str(list(v)))
def test_odd_widths(sched, kw, N, dtype):
    if sched == "bd" and dtype == "f32":
        pytest.skip("bd takes 16-bit storage")
    t = torch()
    for M in (4200, 40):
        rng = np.random.default_rng(N)
        K, ldb, ldc = 300, N + 2 * (N % 4), N + 1
        lens = rng.integers(0, 24, M)
        lens[M // 2] = 250
        pos = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        crd = np.concatenate([np.sort(rng.choice(K, int(l), replace=False)) for l in lens])
        crd = crd.astype(np.int32)
        vals = rng.uniform(-1, 1, len(crd)).astype(np.float32)
        A = DeviceCSR(pos, crd, vals, K, dtype=dtype)
        B = rng.uniform(-1, 1, (K, N)).astype(np.float32)
        Bp = np.full((K, ldb), np.nan, np.float32)
        Bp[:, :N] = B
        Bd = dense_dev(Bp, dtype)
        print(f"[widths] {sched} {kw} N={N} {dtype} M={M}", flush=True)
        plan = S.plan_resolve(A.desc, N, S.DTYPES[dtype], S.make_plan(sched, **kw), ldb, ldc)
        C = run_spmm(A, Bd, N, plan, ldb=ldb, ldc=ldc, b_dtype=dtype).cpu().numpy()
        v, Br = (vals, B) if dtype == "f32" else (O.round_to(dtype, vals)[1],
                                                  O.round_to(dtype, B)[1])
        err = O.scaled_err(C[:, :N].copy(), O.spmm_f64(pos, crd, v, Br),
                           O.spmm_absbound(pos, crd, v, Br))
        assert err <= 1e-5
        assert np.isnan(C[:, N:]).all(), "wrote outside [0, N)"
        if sched in ("eb_cs", "bd"):
            continue
        D = t.full((M, ldc), float("nan"), dtype=t.float32, device="cuda")
        batch = S.Batch([S.batch_item(A.desc, Bd.data_ptr(), ldb, D.data_ptr(), ldc, N, plan,
                                      pos)], dtype, stream_ptr())
        batch.run(stream_ptr())
        t.cuda.synchronize()
        assert np.array_equal(C.view(np.uint32), D.cpu().numpy().view(np.uint32))
        batch.destroy()
