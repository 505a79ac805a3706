"""The calls whose speed is tracked: what programs that use segtaco_amd have it do.

A case is a dict of plain values:

    op        spmm      C = A * B, partition and fix-up included, on every call
              prepared  the same for an A that stays resident (prepared once)
              sddmm     out[p] = s_p * <X[row(p)], Y[col(p)]>
              batch     a list of products in one captured launch
              host      an operator-surface entry point on host operands
    matrix    powerlaw (log-normal row lengths, sigma 1.5, cap 8192), uniform
              (`mean` entries in every row) or banded (|i - j| <= bw)
    M, K      rows and columns of A; mean or bw: its row lengths
    N         columns of B (of X and Y for sddmm)
    dtype     storage of A's values, B, X and Y: f32, bf16 or fp16
    schedule  the plan's schedule, or "auto": what the autotuner's model picks
              from the row lengths (rb_sr for even rows, eb_sr for skewed ones)

Row lengths depend on the case alone (their order on the seed), so that every
seed gives the same number of entries. Inputs are made with torch on the GPU.
"""
import math
import random

import numpy as np
import torch

import segtaco_amd as S

SIGMA, CAP = 1.5, 8192
ELEM = {"f32": 4, "bf16": 2, "fp16": 2}
TORCH = {"f32": torch.float32, "bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    return [
        # A small graph's feature aggregation: latency and launches count.
        dict(name="small_1000_n16", op="spmm", matrix="powerlaw", M=1000, K=1000, mean=16.0,
             N=16, dtype="f32", schedule="auto"),
        # The sweep driver's default width (4 columns) on a mid-sized matrix:
        # the element-balanced schedule, and the row-balanced tree reduction
        # on a rectangular, ragged one.
        dict(name="sweep_200k_n4_eb_sr", op="spmm", matrix="powerlaw", M=200000, K=200000,
             mean=12.0, N=4, dtype="f32", schedule="eb_sr"),
        dict(name="sweep_60013_n4_rb_pr", op="spmm", matrix="powerlaw", M=60013, K=50021,
             mean=24.0, N=4, dtype="f32", schedule="rb_pr"),
        # SpMV: the inner step of iterative solvers and PageRank.
        dict(name="spmv_262144", op="spmm", matrix="powerlaw", M=262144, K=262144, mean=16.0,
             N=1, dtype="f32", schedule="eb_pr"),
        # Even row lengths (meshes, fixed-degree sampling), ragged sizes.
        dict(name="uniform_100003_n32", op="spmm", matrix="uniform", M=100003, K=90001,
             mean=20.0, N=32, dtype="f32", schedule="auto"),
        # The headline benchmark: one full call, column sort included.
        dict(name="powerlaw_262144_n128_eb_cs", op="spmm", matrix="powerlaw", M=262144,
             K=262144, mean=16.0, N=128, dtype="f32", schedule="eb_cs"),
        # A resident adjacency multiplied many times (GNN layers at width 64).
        dict(name="resident_131072_n64_eb_cs", op="prepared", matrix="powerlaw", M=131072,
             K=131072, mean=24.0, N=64, dtype="f32", schedule="eb_cs"),
        # Wide 16-bit features.
        dict(name="powerlaw_262144_n256_bf16", op="spmm", matrix="powerlaw", M=262144,
             K=262144, mean=16.0, N=256, dtype="bf16", schedule="auto"),
        # An odd width and ragged sizes in 16-bit: no wide loads possible.
        dict(name="ragged_50021_n77_fp16", op="spmm", matrix="powerlaw", M=50021, K=40009,
             mean=20.0, N=77, dtype="fp16", schedule="auto"),
        # Banded systems (stencils) on the matrix cores.
        dict(name="banded_1048576_n256_bf16", op="spmm", matrix="banded", M=1048576,
             K=1048576, bw=32, N=256, dtype="bf16", schedule="bd"),
        # Attention scores / gradients with respect to A's values.
        dict(name="sddmm_262144_j128", op="sddmm", matrix="powerlaw", M=262144, K=262144,
             mean=16.0, N=128, dtype="f32", schedule=""),
        # Many graphs of different sizes and widths in one launch.
        dict(name="batch_24_products", op="batch", matrix="powerlaw", M=200000, K=200000,
             mean=64.0, N=128, dtype="f32", schedule="auto", count=24, sizes=41),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case. No drawn case costs more than the largest listed one."""
    op = rng.choices(["spmm", "spmv", "banded", "prepared", "sddmm", "batch", "host"],
                     [50, 8, 8, 10, 10, 6, 8])[0]
    M = _log(rng, 500, 300000)
    K = M if rng.random() < 0.5 else _log(rng, 500, 300000)
    mean = round(math.exp(rng.uniform(math.log(4), math.log(40))), 1)
    mean = min(mean, 4.5e6 / M, K / 16)
    N = rng.choice([4, 4, 8, 16, 32, 64, 128, 256, rng.randint(2, 160), rng.randint(2, 160)])
    dtype = rng.choice(["f32", "f32", "f32", "bf16", "fp16"])
    matrix = "uniform" if rng.random() < 0.2 else "powerlaw"
    if op == "spmv":
        return dict(op="spmm", matrix=matrix, M=M, K=K, mean=mean, N=1, dtype=dtype,
                    schedule="eb_pr")
    if op == "banded":
        M = _log(rng, 4000, 1000000)
        return dict(op="spmm", matrix="banded", M=M, K=M, bw=rng.choice([8, 16, 32, 48]),
                    N=rng.choice([32, 64, 128, 256, rng.randint(16, 200)]),
                    dtype=rng.choice(["bf16", "fp16"]), schedule="bd")
    if op == "prepared":
        return dict(op="prepared", matrix="powerlaw", M=M, K=K, mean=mean, N=max(N, 16),
                    dtype="f32", schedule="eb_cs")
    if op == "sddmm":
        return dict(op="sddmm", matrix=matrix, M=M, K=K, mean=mean, N=max(N, 8), dtype=dtype,
                    schedule="")
    if op == "batch":
        return dict(op="batch", matrix="powerlaw", M=_log(rng, 2000, 150000), K=0, mean=40.0,
                    N=rng.choice([32, 64, 128]), dtype=dtype, schedule="auto",
                    count=rng.randint(4, 24), sizes=rng.randint(0, 9999))
    if op == "host":
        return dict(op="host", matrix=matrix, M=M, K=K, mean=mean, N=rng.choice([4, 4, 16, 64]),
                    dtype="f32",
                    schedule=rng.choice(["spmm_rb_sr", "spmm_rb_pr", "spmm_eb_sr",
                                         "spmm_eb_pr", "spmm_csr_gpu_taco"]))
    if matrix == "uniform":
        schedule = rng.choice(["auto", "auto", "rb_sr", "rb_pr"])
    else:
        schedule = rng.choice(["auto", "auto", "rb_sr", "rb_pr", "eb_sr", "eb_pr", "eb_cs"])
        if schedule == "eb_cs":
            dtype = "f32"
    return dict(op="spmm", matrix=matrix, M=M, K=K, mean=mean, N=N, dtype=dtype,
                schedule=schedule)


def _products(case):
    """The (M, mean, N) of a batch's products; one product for other cases."""
    if case["op"] != "batch":
        return [(case["M"], case.get("mean", 0.0), case["N"])]
    r = random.Random(case["sizes"])
    widths = [w for w in (16, 32, 64, 128) if w <= case["N"]]
    return [(r.randint(1000, case["M"]), r.uniform(8, case["mean"]), r.choice(widths))
            for _ in range(case["count"])]


def _lengths(case, M, K, mean):
    """Entries per row (int64[M]), in an order that _csr shuffles."""
    if case["matrix"] == "banded":
        i = torch.arange(M)
        return (i + case["bw"]).clamp(max=K - 1) - (i - case["bw"]).clamp(min=0) + 1
    if case["matrix"] == "uniform":
        return torch.full((M,), int(round(mean))).clamp(max=K)
    z = torch.special.ndtri((torch.arange(M, dtype=torch.float64) + 0.5) / M)
    n = torch.exp(math.log(mean) - 0.5 * SIGMA * SIGMA + SIGMA * z).round().long()
    return n.clamp(max=min(CAP, K))


def _csr(case, M, K, mean, g):
    """(pos, crd, vals, rows) on the GPU: sorted, distinct columns in every
    row, spread evenly over [0, K); values in [-1, 1) in the storage type."""
    n = _lengths(case, M, K, mean).cuda()
    if case["matrix"] == "powerlaw":
        n = n[torch.randperm(M, generator=g, device="cuda")]
    pos = torch.zeros(M + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(n, 0, out=pos[1:])
    nnz = int(pos[-1])
    rows = torch.repeat_interleave(torch.arange(M, device="cuda"), n, output_size=nnz)
    rank = torch.arange(nnz, device="cuda") - pos[rows]
    if case["matrix"] == "banded":
        crd = (rows - case["bw"]).clamp(min=0) + rank
    else:
        # sorted draws from [0, K - n], plus their rank: distinct, below K
        span = (K - n + 1)[rows]
        u = torch.rand(nnz, generator=g, device="cuda", dtype=torch.float64)
        key = rows * K + (u * span).long().clamp(max=K - 1)
        crd = torch.sort(key).values - rows * K + rank
    vals = (torch.rand(nnz, generator=g, device="cuda") * 2 - 1).to(TORCH[case["dtype"]])
    return pos.int(), crd.int(), vals, rows


def _dense(rows, cols, case, g):
    return (torch.rand((rows, cols), generator=g, device="cuda") * 2 - 1).to(
        TORCH[case["dtype"]])


def _inputs(case, seed):
    """Per product: (pos, crd, vals, rows, B) and X for sddmm."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    out = []
    for M, mean, N in _products(case):
        K = M if case["op"] == "batch" else case["K"]
        pos, crd, vals, rows = _csr(case, M, K, mean, g)
        B = _dense(K, N, case, g)
        X = _dense(M, N, case, g) if case["op"] == "sddmm" else None
        out.append((pos, crd, vals, rows, B, X))
    return out


def prepare(case, seed):
    """Operands in device memory (host memory for `host`), the plan, the
    workspace, and the argument list of the call."""
    op, dt = case["op"], S.DTYPES[case["dtype"]]
    ins = _inputs(case, seed)
    if op == "host":
        pos, crd, vals, _, B, _ = ins[0]
        C = np.zeros((case["M"], case["N"]), dtype=np.float32)
        return dict(op=op, args=(case["schedule"], pos.cpu().numpy(), crd.cpu().numpy(),
                                 vals.cpu().numpy(), B.cpu().numpy(), case["K"], C))
    if op == "batch":
        items, keep, outs = [], [], []
        for pos, crd, vals, _, B, _ in ins:
            M, N = pos.numel() - 1, B.shape[1]
            A = S.csr_desc(M, M, crd.numel(), pos.data_ptr(), crd.data_ptr(), vals.data_ptr(),
                           dt)
            C = torch.empty((M, N), dtype=torch.float32, device="cuda")
            host = pos.cpu().numpy()
            items.append(S.batch_item(A, B.data_ptr(), N, C.data_ptr(), N, N, None, host))
            keep.append((pos, crd, vals, B, host))
            outs.append(C)
        torch.cuda.synchronize()
        batch = S.Batch(items, dt)
        batch.capture()
        return dict(op=op, batch=batch, keep=keep, out=outs)
    pos, crd, vals, _, B, X = ins[0]
    M, K, N, nnz = case["M"], case["K"], case["N"], crd.numel()
    A = S.csr_desc(M, K, nnz, pos.data_ptr(), crd.data_ptr(), vals.data_ptr(), dt)
    if op == "sddmm":
        out = torch.empty(nnz, dtype=torch.float32, device="cuda")
        nbytes = S.sddmm_workspace_bytes(A)
        ws = torch.empty(max(nbytes, 1), dtype=torch.uint8, device="cuda")
        args = (A, X.data_ptr(), N, B.data_ptr(), N, N, dt, out.data_ptr(), ws.data_ptr(),
                nbytes)
        return dict(op=op, args=args, keep=(pos, crd, vals, B, X, ws), out=out)
    if case["schedule"] == "auto":
        plan = S.tune_model(S.row_stats(pos.cpu().numpy(), K), N, dt)
    else:
        plan = S.make_plan(case["schedule"])
    C = torch.empty((M, N), dtype=torch.float32, device="cuda")
    nbytes = S.workspace_bytes(A, N, plan)
    ws = torch.empty(max(nbytes, 1), dtype=torch.uint8, device="cuda")
    if op == "prepared":
        S.spmm_prepare(A, dt, N, N, N, plan, ws.data_ptr(), nbytes)
    args = (A, B.data_ptr(), dt, N, N, C.data_ptr(), N, plan, ws.data_ptr(), nbytes)
    return dict(op=op, args=args, keep=(pos, crd, vals, B, ws), out=C)


def run(state):
    op = state["op"]
    if op == "spmm":
        S.spmm(*state["args"])
    elif op == "prepared":
        S.spmm_prepared(*state["args"])
    elif op == "sddmm":
        S.sddmm(*state["args"])
    elif op == "batch":
        state["batch"].replay()
    else:
        return S.legacy(*state["args"])[0]
    return state["out"]


def work(case):
    """Every operand read once, every result written once; of B (Y) the rows
    that the columns, drawn evenly, refer to."""
    e, nbytes, flops = ELEM[case["dtype"]], 0.0, 0.0
    for M, mean, N in _products(case):
        K = M if case["op"] == "batch" else case["K"]
        nnz = int(_lengths(case, M, K, mean).sum())
        touched = K if case["matrix"] == "banded" else K * -math.expm1(-nnz / K)
        nbytes += 4 * (M + 1) + nnz * (4 + e) + touched * N * e
        nbytes += M * N * e + 4 * nnz if case["op"] == "sddmm" else 4 * M * N
        flops += 2.0 * nnz * N
    return {"bytes": nbytes, "flops": flops}


def exact(case, seed):
    out = []
    for pos, crd, vals, rows, B, X in _inputs(case, seed):
        M, N, nnz = pos.numel() - 1, B.shape[1], crd.numel()
        B, v = B.double(), vals.double()
        step = max(1, (1 << 28) // N)  # entries per pass: 2 GiB of products
        if X is not None:
            r = torch.cat([(X[rows[a:a + step]].double() * B[crd[a:a + step]]).sum(1)
                           for a in range(0, nnz, step)]) * v
        else:
            r = torch.zeros((M, N), dtype=torch.float64, device="cuda")
            for a in range(0, nnz, step):
                r.index_add_(0, rows[a:a + step],
                             B[crd[a:a + step]] * v[a:a + step, None])
        out.append(r)
    return out if case["op"] == "batch" else out[0]
