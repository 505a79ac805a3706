"""Which kernel form a plan runs with, and sizing for plans whose fields no
call would accept (host logic, no GPU)."""
import math
import os
import subprocess
import sys

import numpy as np
import pytest

import segtaco_amd as S

PROBE = """
import sys
sys.path.insert(0, {root!r})
import segtaco_amd as S
A = S.csr_desc(1000, 1000, 5000, 0x1000, 0x2000, 0x3000, S.DT_F32)
p = S.make_plan("eb_cs", vec={vec}, col_lanes={lanes}, group=64, tile=64, comp_threshold=0)
print(S.{call}(A, 64, p))
"""


# In a process of its own: a sizing query must neither hang nor raise a signal.
@pytest.mark.parametrize("call,vec,lanes", [("cs_workspace_layout", 4, 0),
                                            ("cs_workspace_layout", 1, 0),
                                            ("workspace_bytes", -1, 8),
                                            ("workspace_bytes", -2, 8)])
def test_eb_cs_sizing_of_unusual_plans(call, vec, lanes):
    root = os.path.dirname(os.path.dirname(os.path.abspath(S.__file__)))
    r = subprocess.run([sys.executable, "-c", PROBE.format(root=root, call=call, vec=vec,
                                                           lanes=lanes)],
                       capture_output=True, text=True, timeout=20)
    assert r.returncode == 0, (r.returncode, r.stderr)
    if call == "cs_workspace_layout":
        A = S.csr_desc(1000, 1000, 5000, 0x1000, 0x2000, 0x3000, S.DT_F32)
        full = S.make_plan("eb_cs", vec=vec, col_lanes=8, group=64, tile=64, comp_threshold=0)
        assert r.stdout.strip() == str(S.cs_workspace_layout(A, 64, full))


def _form(N, dtype, sched="eb_sr", M=60000, nnz=1_000_000, ldb=None, B=0, batch=False, **kw):
    A = S.csr_desc(M, M, nnz, 0x1000, 0x2000, 0x3000, S.DTYPES[dtype])
    return S.spmm_form(A, N, S.DTYPES[dtype], S.make_plan(sched, **kw), ldb, ldb, B, 0, batch)


# A form that the plan names is the one that runs; each row once gave another's.
@pytest.mark.parametrize("sched,dtype,N,kw", [
    ("eb_sr", "f32", 64, dict(vec=1)), ("eb_sr", "f32", 64, dict(vec=2)),
    ("eb_sr", "bf16", 64, dict(vec=4)), ("eb_sr", "f32", 4, dict(vec=1)),
    ("eb_sr", "f32", 128, dict(vec=4, col_lanes=8)), ("rb_sr", "f32", 256, dict(vec=1)),
    ("rb_pr", "f32", 128, dict(vec=1)), ("rb_pr", "bf16", 128, dict(vec=2, group=8)),
    ("eb_pr", "f32", 128, dict(vec=1)), ("eb_pr", "bf16", 128, dict(vec=4))],
    ids=lambda v: str(v) if not isinstance(v, dict) else "-".join(f"{k}{x}" for k, x in v.items()))
@pytest.mark.parametrize("batch", [False, True])
def test_named_slices_are_kept(sched, dtype, N, kw, batch):
    f = _form(N, dtype, sched, tile=128 if sched[:2] == "eb" else 0, batch=batch, **kw)
    A = S.csr_desc(60000, 60000, 1_000_000, 0x1000, 0x2000, 0x3000, S.DTYPES[dtype])
    p = S.plan_resolve(A, N, S.DTYPES[dtype], S.make_plan(sched, **kw))
    assert f == dict(vec=kw["vec"], lanes=p.col_lanes, seg_vec=0, seg_tiles=0)


# The presets of one schedule that differ in their columns per lane run apart.
@pytest.mark.parametrize("N", [32, 64])
def test_column_presets_differ(N):
    forms = [_form(N, "f32", "eb_sr", tile=256, vec=c) for c in (1, 2, 4)]
    assert len({(f["vec"], f["lanes"], f["seg_vec"]) for f in forms}) >= 2
    assert [f["vec"] for f in forms[:2]] == [1, 2]


# Open plans, and plans resolved from them, keep the widths chosen for the call.
def test_open_plans_choose():
    assert _form(77, "fp16", tile=128)["vec"] == 4
    assert _form(77, "f32", "rb_pr")["vec"] > 1
    assert _form(128, "f32", ldb=129, tile=128)["vec"] == 4
    assert _form(128, "f32", B=0x1004, tile=128)["vec"] == 4
    assert _form(4, "f32")["seg_vec"] == 4
    A = S.csr_desc(60000, 60000, 1_000_000, 0x1000, 0x2000, 0x3000, S.DT_F32)
    for N in (4, 16, 64, 77, 128):
        p = S.plan_resolve(A, N, S.DT_F32, S.make_plan("eb_sr"))
        assert S.spmm_form(A, N, S.DT_F32, p) == S.spmm_form(A, N, S.DT_F32,
                                                             S.make_plan("eb_sr"))


# Short tiles keep wide slices: a batch's unit holds 1024 entries where slices of
# four columns allow it, and a call's tiles of up to 16 entries are not spread thin.
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("N", [4, 8, 16, 24, 32, 64, 128, 256])
@pytest.mark.parametrize("tile", [8, 16, 32, 64, 128])
def test_short_tiles_keep_wide_slices(N, tile, dtype):
    f = _form(N, dtype, tile=tile, batch=True)
    assert tile * 256 // f["lanes"] >= 1024 or f["vec"] == 4
    assert f["vec"] <= 4  # eight columns would take the kernel with every schedule
    if tile <= 16 and N > 8:
        assert _form(N, dtype, tile=tile, M=1_000_000, nnz=1_500_000)["vec"] >= 2
    if tile == 128:  # the narrow forms
        assert f["vec"] == max(1, min(4, N // 32))


# The segment form takes narrow products of any size, those of 9 to 16 columns up
# to the size from which the walk is faster, and never a plan that names its slices.
@pytest.mark.parametrize("dtype,tile,N,nnz,seg", [
    ("f32", 128, 8, 4_000_000, True), ("bf16", 16, 8, 4_000_000, True),
    ("f32", 128, 16, 1 << 20, True), ("f32", 128, 16, (1 << 20) + 1, False),
    ("f32", 64, 9, 1 << 20, True), ("f32", 32, 9, (1 << 19) + 1, False),
    ("f32", 16, 12, 1 << 19, True), ("f32", 16, 12, 1_000_000, False),
    ("bf16", 128, 16, 1 << 19, True), ("bf16", 128, 12, 1_000_000, False),
    ("fp16", 16, 9, 2_000_000, False), ("f32", 128, 17, 1 << 20, False)])
def test_segment_form_by_size(dtype, tile, N, nnz, seg):
    assert (_form(N, dtype, nnz=nnz, tile=tile)["seg_vec"] > 0) == seg
    assert _form(N, dtype, nnz=nnz, tile=tile, batch=True)["seg_vec"] == 0
    assert _form(N, dtype, nnz=nnz, M=2 * nnz + 1, tile=tile)["seg_vec"] == 0
    if N % 2 == 0:
        assert _form(N, dtype, nnz=nnz, tile=tile, vec=1)["seg_vec"] == 0


# Plans that were measured with kernels of another generation are not taken from a
# saved cache: the signature they were saved under is no matrix's any more.
def test_old_cache_entries_do_not_match():

    def signature(st, N, dtype, salt):
        h = 1469598103934665603
        near = lambda x: int(math.floor(x + 0.5))
        for v in (st.M.bit_length() - 1, near(math.log2(st.mean_len) * 4), near(st.cv * 4),
                  near(st.frac_nnz_long * 10), (st.max_len + 1).bit_length() - 1, N, dtype, salt):
            for b in (v & (2 ** 64 - 1)).to_bytes(8, "little"):
                h = ((h ^ b) * 1099511628211) & (2 ** 64 - 1)
        return h

    st = S.row_stats(np.cumsum([0] + [3, 9, 27, 1] * 500).astype(np.int32), 4000)
    for N in (16, 64, 128):
        assert S.tune_signature(st, N) == signature(st, N, S.DT_F32, 8)
        S.tune_cache_clear()
        S.tune_cache_put(signature(st, N, S.DT_F32, 7), S.make_plan("rb_pr", vec=1, col_lanes=4,
                                                                    group=16, comp_threshold=0))
        assert S.tune(st, N).as_dict() == S.tune_model(st, N).as_dict()
    S.tune_cache_clear()
