"""eb_sr takes a tile's entries in short batches: one in which no row of the
wave ends is summed without looking at rows, and the staged entries are padded
to whole batches. Tiles and rows that end one before, at and one after a batch,
against the exact sums of whole numbers (every order gives the same)."""
import numpy as np
import pytest

import segtaco_amd as S
from gpu_util import DeviceCSR, dense_dev, run_spmm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("N", [72, 128, 260])
@pytest.mark.parametrize("tile", [8, 9, 15, 17, 129, 256])
@pytest.mark.parametrize("row", [3, 4, 5, 8, 0])
def test_batch_edges(row, tile, N, dtype):
    rng = np.random.default_rng(tile * 10 + row)
    K = 1500
    # row 0: all lengths, and one long (compensated in BF16)
    lens = np.full(700, row) if row else np.r_[rng.integers(0, 40, 300), 1200, np.arange(20), 1]
    pos = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    crd = np.concatenate([np.sort(rng.choice(K, int(l), replace=False)) for l in lens])
    crd = crd.astype(np.int32)
    vals = rng.integers(-3, 4, len(crd)).astype(np.float32)
    B = rng.integers(-4, 5, (K, N)).astype(np.float32)
    A = DeviceCSR(pos, crd, vals, K, dtype=dtype)
    plan = S.plan_resolve(A.desc, N, S.DTYPES[dtype], S.make_plan("eb_sr", tile=tile), N, N)
    print(f"[eb] row={row} tile={tile} N={N} {dtype}", flush=True)
    C = run_spmm(A, dense_dev(B, dtype), N, plan, b_dtype=dtype).cpu().numpy()
    want = np.concatenate([np.zeros((1, N)), np.cumsum(B[crd] * vals[:, None], axis=0)])
    assert np.array_equal(C, (want[pos[1:]] - want[pos[:-1]]).astype(np.float32))
