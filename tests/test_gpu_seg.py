"""The segment form of eb_sr (narrow and small products): the same sums as the
walk for the same tile, so a standalone call is bit-identical to the same plan
in a batch (which walks), within 1e-5 of the FP64 oracle, and leaves the same
partition records; at the edges of its ranges, lane groups and vectors."""
import numpy as np
import pytest

import oracle as O
import segtaco_amd as S
from gpu_util import DeviceCSR, dense_dev, run_spmm, stream_ptr, torch

pytestmark = pytest.mark.gpu


def _mk(rng, lens, K):
    lens = np.minimum(lens, K)
    pos = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    crd = np.concatenate([np.sort(rng.choice(K, int(l), replace=False)) for l in lens]
                         + [np.zeros(0, np.int64)]).astype(np.int32)
    return pos, crd, rng.uniform(-1, 1, len(crd)).astype(np.float32)


def _structure(name, rng):
    if name == "skewed":  # rows inside a piece, over tiles and over ranges
        lens = rng.lognormal(2.0, 1.5, 1500).astype(np.int64)
        lens[700] = 3000
        return _mk(rng, lens, 4000)
    if name == "empty_runs":  # runs of more than 64 empty rows inside a range
        lens = rng.integers(1, 9, 3000)
        lens[:130] = 0
        lens[500:700] = 0
        lens[1000:1900:3] = 0
        lens[-200:] = 0
        return _mk(rng, lens, 900)
    if name == "one_entry_rows":
        return _mk(rng, np.ones(1025, np.int64), 300)
    if name == "one_row":
        return _mk(rng, np.array([2500]), 3000)
    assert name == "one_entry"
    return _mk(rng, np.array([0, 1, 0]), 5)


@pytest.mark.parametrize("N,dtype", [(1, "f32"), (2, "bf16"), (3, "f32"), (4, "f32"), (5, "fp16"),
                                     (8, "bf16"), (16, "f32"), (17, "f32"), (33, "bf16"),
                                     (63, "fp16"), (64, "f32")])
@pytest.mark.parametrize("tile", [8, 33, 128, 384, 1024])
def test_same_bits_as_the_walk(N, dtype, tile):
    t = torch()
    for name in ("skewed", "empty_runs", "one_entry_rows", "one_row", "one_entry"):
        rng = np.random.default_rng(N * 1000 + tile)
        pos, crd, vals = _structure(name, rng)
        M, K = len(pos) - 1, int(crd.max()) + 1
        vals = None if name == "one_entry_rows" else vals
        A = DeviceCSR(pos, crd, vals, K, dtype=dtype)
        B = rng.uniform(-1, 1, (K, N)).astype(np.float32)
        B[0, 0] = np.inf  # stays in the rows that refer to it
        ldb, ldc = N + N % 2, N + 3
        Bp = np.full((K, ldb), np.nan, np.float32)
        Bp[:, :N] = B
        Bd = dense_dev(Bp, dtype)
        bd = S.DTYPES[dtype]
        plan = S.plan_resolve(A.desc, N, bd, S.make_plan("eb_sr", tile=tile, comp_threshold=500),
                              ldb, ldc)
        print(f"[seg] {name} N={N} {dtype} tile={tile}", flush=True)
        C = run_spmm(A, Bd, N, plan, ldb=ldb, ldc=ldc, b_dtype=dtype).cpu().numpy()
        D = t.full((M, ldc), float("nan"), dtype=t.float32, device="cuda")
        batch = S.Batch([S.batch_item(A.desc, Bd.data_ptr(), ldb, D.data_ptr(), ldc, N, plan,
                                      pos)], dtype, stream_ptr())
        batch.run(stream_ptr())
        t.cuda.synchronize()
        assert np.array_equal(C.view(np.uint32), D.cpu().numpy().view(np.uint32)), name
        assert np.isnan(C[:, N:]).all()
        fine = np.isfinite(C[:, :N])
        if name == "skewed":
            hit = np.zeros(M, bool)
            hit[np.repeat(np.arange(M), np.diff(pos))[crd == 0]] = True
            assert np.array_equal(~fine[:, 0], hit)
        v = vals if dtype == "f32" or vals is None else O.round_to(dtype, vals)[1]
        B[0, 0] = 0
        Br = B if dtype == "f32" else O.round_to(dtype, B)[1]
        ref, scale = O.spmm_f64(pos, crd, v, Br), O.spmm_absbound(pos, crd, v, Br)
        err = np.abs(C[:, :N].astype(np.float64) - ref)[fine] / (scale[fine] + 1e-30)
        assert err.max(initial=0) <= 1e-5, name
        batch.destroy()
