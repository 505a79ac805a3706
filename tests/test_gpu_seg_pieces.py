"""The segment form where a wave's range holds several tiles: rows in 2 to 48
pieces inside a range, over neighbouring ranges and over many, with and without
compensation, at the range's and the entries' edges, have the bits of the same plan in
a batch (which walks) and leave the partition records of segtaco_tile_rows. Every
cell asserts that the segment form runs, and with how many tiles."""
import numpy as np
import pytest

import segtaco_amd as S
from gpu_util import DeviceCSR, dense_dev, dev, stream_ptr, torch

pytestmark = pytest.mark.gpu


def _csr(lens, K, rng):
    pos = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    crd = np.empty(pos[-1], np.int32)
    for r, n in enumerate(lens):  # distinct, ascending
        crd[pos[r]:pos[r] + n] = np.sort(rng.integers(0, K - n + 1, n)) + np.arange(n)
    return pos, crd


def _lens(kind, nnz, tile, rng):
    out, left = [], nnz
    while left > 0:
        if kind == "spanning":  # 3 to 40 tiles, whole tiles and one entry beside them
            n = int(rng.integers(3, 41)) * tile + int(rng.integers(-1, 2))
        elif kind == "mixed":  # short rows, empty rows, and every tenth over tiles
            n = int(rng.integers(0, 6)) if rng.random() < 0.9 else int(rng.integers(1, 5 * tile))
        else:  # a few rows over hundreds of ranges between rows of one entry
            n = 1 if rng.random() < 0.97 else int(rng.integers(5000, 60000))
        out.append(min(n, left))
        left -= out[-1]
    return np.array(out)


# (tile, N, dtype, tiles per range): ranges are up to 384 entries
CELLS = [(8, 1, "f32", 48), (8, 5, "bf16", 32), (8, 8, "f32", 32), (8, 16, "f32", 16),
         (33, 1, "fp16", 11), (33, 4, "f32", 11), (33, 7, "f32", 7), (33, 12, "bf16", 3),
         (128, 1, "f32", 3), (128, 3, "f32", 3), (128, 4, "bf16", 3), (128, 8, "fp16", 2)]


@pytest.mark.parametrize("comp", [0, 100])
@pytest.mark.parametrize("tile,N,dtype,tiles", CELLS)
def test_pieces(tile, N, dtype, tiles, comp):
    t = torch()
    nnz = 900_001 if N <= 8 else 500_003
    for kind in ("spanning", "mixed", "far"):
        rng = np.random.default_rng(tile * 100 + N)
        lens = _lens(kind, nnz, tile, rng)
        K = int(lens.max()) + 50
        pos, crd = _csr(lens, K, rng)
        M = len(lens)
        A = DeviceCSR(pos, crd, rng.uniform(-1, 1, nnz).astype(np.float32), K, dtype=dtype)
        Bd = dense_dev(rng.uniform(-1, 1, (K, N)), dtype)
        bd = S.DTYPES[dtype]
        plan = S.plan_resolve(A.desc, N, bd, S.make_plan("eb_sr", tile=tile, comp_threshold=comp))
        f = S.spmm_form(A.desc, N, bd, plan)
        assert f["seg_vec"] > 0 and f["seg_tiles"] == tiles, (kind, f)
        print(f"[pieces] {kind} tile={tile} N={N} {dtype} comp={comp}", flush=True)
        C = t.full((M, N), float("nan"), dtype=t.float32, device="cuda")
        D = C.clone()
        nb = S.workspace_bytes(A.desc, N, plan)
        ws = t.zeros(nb, dtype=t.uint8, device="cuda")
        S.spmm(A.desc, Bd.data_ptr(), bd, N, N, C.data_ptr(), N, plan, ws.data_ptr(), nb,
               stream_ptr())
        batch = S.Batch([S.batch_item(A.desc, Bd.data_ptr(), N, D.data_ptr(), N, N, plan, pos)],
                        dtype, stream_ptr())
        batch.run(stream_ptr())
        t.cuda.synchronize()
        assert t.equal(C.view(t.int32), D.view(t.int32)), kind
        batch.destroy()
        L = S.workspace_layout(A.desc, N, plan)
        nt = L["ntiles"]
        rows = ws[L["rows_off"]:L["rows_off"] + 4 * (nt + 1)].view(t.int32).cpu().numpy()
        want = t.empty(nt + 1, dtype=t.int32, device="cuda")
        S.tile_rows(A.pos.data_ptr(), M, tile, nt, want.data_ptr(), S.ROWS_SCATTER)
        t.cuda.synchronize()
        assert np.array_equal(rows, want.cpu().numpy()), kind
        # the record of a tile: where the row that ends in it, having begun before, began
        fix = ws[L["fix_off"]:L["fix_off"] + 4 * nt].view(t.int32).cpu().numpy()
        ref = np.full(nt, -1, np.int32)
        a, b = pos[:-1] // tile, (pos[1:] - 1) // tile
        over = (lens > 0) & (a < b)
        ref[b[over]] = a[over]
        assert np.array_equal(fix, ref), kind


@pytest.mark.parametrize("lens", [[1], [2], [0, 1], [7, 0, 1], [8], [9]])
@pytest.mark.parametrize("N", [1, 4, 16])
def test_smallest(lens, N):
    t = torch()
    rng = np.random.default_rng(len(lens) + N)
    pos, crd = _csr(np.array(lens), 20, rng)
    vals = rng.integers(-3, 4, len(crd)).astype(np.float32)
    B = rng.integers(-4, 5, (20, N)).astype(np.float32)
    A = DeviceCSR(pos, crd, vals, 20)
    plan = S.plan_resolve(A.desc, N, S.DT_F32, S.make_plan("eb_sr"))
    assert S.spmm_form(A.desc, N, S.DT_F32, plan)["seg_vec"] > 0
    C = t.full((len(lens), N), float("nan"), dtype=t.float32, device="cuda")
    nb = S.workspace_bytes(A.desc, N, plan)
    ws = t.empty(nb, dtype=t.uint8, device="cuda")
    Bd = dev(B)
    S.spmm(A.desc, Bd.data_ptr(), S.DT_F32, N, N, C.data_ptr(), N, plan, ws.data_ptr(), nb,
           stream_ptr())
    t.cuda.synchronize()
    want = np.zeros((len(lens), N), np.float32)
    np.add.at(want, np.repeat(np.arange(len(lens)), lens), B[crd] * vals[:, None])
    assert np.array_equal(C.cpu().numpy(), want)


# SpMM slices from operands that are aligned to one element only.
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("sched,N", [("eb_sr", 8), ("eb_sr", 64), ("eb_sr", 128), ("rb_sr", 32),
                                     ("rb_pr", 64), ("eb_pr", 64), ("eb_cs", 64)])
def test_element_aligned_operands(sched, N, dtype):
    t = torch()
    rng = np.random.default_rng(N)
    lens = rng.integers(0, 40, 6000)
    lens[[5, 4000]] = [900, 0]
    pos, crd = _csr(lens, 1500, rng)
    M = len(lens)
    vals = rng.integers(-3, 4, len(crd)).astype(np.float32)
    B = rng.integers(-4, 5, (1500, N)).astype(np.float32)
    A = DeviceCSR(pos, crd, vals, 1500, dtype=dtype)
    eb = 4 if dtype == "f32" else 2
    flat = dense_dev(np.concatenate([[0.0], B.reshape(-1)]), dtype)
    C = t.full((M * N + 1,), float("nan"), dtype=t.float32, device="cuda")
    plan = S.make_plan(sched)
    nb = S.workspace_bytes(A.desc, N, plan)
    ws = t.empty(max(nb, 1), dtype=t.uint8, device="cuda")
    S.spmm(A.desc, flat.data_ptr() + eb, S.DTYPES[dtype], N, N, C.data_ptr() + 4, N, plan,
           ws.data_ptr(), nb, stream_ptr())
    t.cuda.synchronize()
    e = B[crd] * vals[:, None]
    want = np.concatenate([np.zeros((1, N)), np.cumsum(e, axis=0)])
    want = (want[pos[1:]] - want[pos[:-1]]).astype(np.float32)
    got = C.cpu().numpy()
    assert np.isnan(got[0]) and np.array_equal(got[1:].reshape(M, N), want)
