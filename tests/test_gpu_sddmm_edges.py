"""SDDMM rows are taken in the widest slices whatever J, the leading dimensions
and the alignment, the last slice moved back to end at J; and each wave finds
the rows of its own tile. Widths around the slices and panels, operands that
start at any element with NaN around every row, runs of empty rows, and entry
counts of each tile length, against the exact sums of whole numbers."""
import numpy as np
import pytest

import segtaco_amd as S
from gpu_util import DeviceCSR, dense_dev, dev, stream_ptr, torch

pytestmark = pytest.mark.gpu


def _check(lens, K, J, off, dtype, seed):
    t = torch()
    rng = np.random.default_rng(seed)
    pos = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    nnz, M = int(pos[-1]), len(lens)
    crd = rng.integers(0, K, nnz).astype(np.int32)
    vals = rng.integers(1, 4, nnz).astype(np.float32)
    A = DeviceCSR(pos, crd, vals, K, dtype=dtype)
    ld = J + off
    host, dense = [], []
    for rows in (M, K):
        full = np.full((rows, ld), np.nan, np.float32)
        full[:, off:] = rng.integers(-3, 4, (rows, J))
        host.append(full[:, off:])
        dense.append(dense_dev(full, dtype))
    eb = 4 if dtype == "f32" else 2
    out = t.full((nnz + 1,), float("nan"), dtype=t.float32, device="cuda")
    nbytes = S.sddmm_workspace_bytes(A.desc)
    ws = t.empty(max(nbytes, 1), dtype=t.uint8, device="cuda")
    print(f"[sddmm] nnz={nnz} J={J} off={off} {dtype}", flush=True)
    S.sddmm(A.desc, dense[0].data_ptr() + off * eb, ld, dense[1].data_ptr() + off * eb, ld, J,
            S.DTYPES[dtype], out.data_ptr(), ws.data_ptr(), nbytes)
    t.cuda.synchronize()
    rows = np.repeat(np.arange(M), lens)
    want = np.zeros(nnz, np.float32)
    for p in range(0, nnz, 1 << 16):
        q = slice(p, p + (1 << 16))
        want[q] = (host[0][rows[q]] * host[1][crd[q]]).sum(axis=1) * vals[q]
    got = out.cpu().numpy()
    assert np.array_equal(got[:nnz], want)
    assert np.isnan(got[nnz])


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("off", [0, 1, 3])
@pytest.mark.parametrize("J", [1, 2, 3, 4, 5, 7, 8, 9, 15, 17, 31, 33, 63, 65, 77, 127, 129, 255,
                               257, 513])
def test_widths(J, off, dtype):
    lens = np.r_[0, 0, np.arange(40), np.zeros(300, int), 1, 0, 700, 3, np.zeros(90, int)]
    _check(lens, 400, J, off, dtype, J)


@pytest.mark.parametrize("nnz,J", [(1, 6), (129, 6), (512 * 1024, 6), (1536 * 1024, 3),
                                   (3584 * 1024, 3), (3584 * 1024, 33)])
def test_tiles(nnz, J):
    rng = np.random.default_rng(nnz)
    lens = np.bincount(np.sort(rng.integers(0, max(nnz // 9, 2), nnz)) // 2 * 2)
    _check(lens, 3000, J, 0, "f32", J)
