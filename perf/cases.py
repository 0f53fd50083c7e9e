"""The performance cases: what programs have this library do, over its real range.

A case is one call, or the pair of calls a program makes per pass, through the
public functions: `ozaki_matmul`, or `split_matrix` + `cross_gemm` where the
weights' slices are kept.  Fields:

    op       "matmul": ozaki_matmul(A, B); "kept": the program holds B's slices
             (a layer's weights) and per pass splits A and multiplies
    batch    products in the call; bcast: B is one matrix shared by all of them
    M, N, K  sizes;  input, slice: dtypes;  splits: slices per operand
    pairs    "all" or "triangular"
    at, bt   A / B is the transposed view of a contiguous matrix
    dist     "normal", "uniform", "exp8" (rows of A and columns of B scaled by
             2^-8 .. 2^8) or "outliers" (1% of the entries 1e4 times larger)
"""
import math

import torch

import ozaki_triton_amd as ozk


def _case(name, op, batch, bcast, M, N, K, input, slice, splits, pairs="all", at=False, bt=False,
          dist="normal"):
    c = dict(op=op, batch=batch, bcast=bcast, M=M, N=N, K=K, input=input, slice=slice,
             splits=splits, pairs=pairs, at=at, bt=bt, dist=dist)
    return dict(c, name=name) if name else c


def listed():
    return [
        # a small product on its own: launches and latency
        _case("small_f32_f16_l2", "matmul", 1, False, 256, 256, 256, "float32", "float16", 2),
        # a batch of small products with the function's default options
        _case("batch16_f32_f16_l3", "matmul", 16, False, 512, 128, 512, "float32", "float16", 3),
        # few rows against a wide, deep matrix: a skinny fp64 product
        _case("skinny_f64_i8_l4", "matmul", 1, False, 128, 2048, 4096, "float64", "int8", 4,
              dist="exp8"),
        # fp32 accuracy from two fp16 slices at a middle size
        _case("square_f32_f16_l2", "matmul", 1, False, 4096, 4096, 4096, "float32", "float16", 2,
              dist="uniform"),
        # the headline: an fp64 product from four int8 slices
        _case("square_f64_i8_l4", "matmul", 1, False, 8192, 8192, 8192, "float64", "int8", 4,
              dist="exp8"),
        # one matrix applied to a batch
        _case("shared_f64_f16_l3", "matmul", 16, True, 1024, 1024, 2048, "float64", "float16", 3),
        # a long contraction with outliers (covariances, normal equations)
        _case("deep_f32_i8_l3", "matmul", 1, False, 1024, 1024, 65536, "float32", "int8", 3,
              dist="outliers"),
        # full fp64-level accuracy: five slices, the triangular pair set
        _case("square_f64_i8_l5_tri", "matmul", 1, False, 4096, 4096, 4096, "float64", "int8", 5,
              pairs="triangular", dist="exp8"),
        # a rank-k update of a large matrix, as in blocked factorisations
        _case("update_f64_i8_l4", "matmul", 1, False, 8192, 8192, 256, "float64", "int8", 4),
        # sizes as meshes and data sets give them: no dimension a round number
        _case("ragged_f64_i8_l4", "matmul", 1, False, 2049, 3000, 2047, "float64", "int8", 4,
              dist="exp8"),
        # the same in fp32, batched, rows that are not whole 16-byte pieces
        _case("ragged_f32_f16_l3", "matmul", 3, False, 257, 1000, 4100, "float32", "float16", 3),
        # a linear layer y = x W^T in bf16 with W's slices kept: split x, multiply
        _case("kept_bf16_i8_l2", "kept", 1, True, 512, 4096, 4096, "bfloat16", "int8", 2),
    ]


def _pairs(case):
    L = case["splits"]
    return L * (L + 1) // 2 if case["pairs"] == "triangular" else L * L


def _size(dtype):
    return {"float64": 8, "float32": 4, "float16": 2, "bfloat16": 2, "int8": 1}[dtype]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _extent(rng, lo, hi):
    """A size of lo .. hi, uniform in its logarithm: half of them multiples of
    64, a tenth of 4, the others any whole number."""
    n, kind = _log_uniform(rng, lo, hi), rng.random()
    step = 64 if kind < 0.5 else 4 if kind < 0.6 else 1
    return max(lo, min(hi, (n + step // 2) // step * step))


def draw(rng):
    while True:
        op = "kept" if rng.random() < 0.15 else "matmul"
        input = rng.choice(["float64"] * 8 + ["float32"] * 8 + ["bfloat16"] * 2 + ["float16"] * 2)
        slice = rng.choice(["int8"] * 10 + ["float16"] * 6 + ["bfloat16"] * 3 + ["float32"])
        batch = 1 if rng.random() < 0.65 else rng.randint(2, 16)
        bcast = op == "kept" or (batch > 1 and rng.random() < 0.4)
        M, N = _extent(rng, 64, 8192), _extent(rng, 64, 8192)
        K = _extent(rng, 64, 65536 if rng.random() < 0.15 else 8192)
        splits = rng.choice([1, 2, 2, 3, 3, 4, 4, 4, 5])
        if splits == 1 and K > 1024:       # one slice of few bits: no use that deep
            continue
        if splits == 5 and (slice == "float32" or op == "kept"):
            splits = 4
        tri = splits >= 2 and rng.random() < (0.5 if splits == 5 else 0.1)
        at, bt = rng.random() < 0.15, op == "matmul" and rng.random() < 0.3
        dist = rng.choice(["normal", "uniform", "exp8"])
        if dist == "exp8" and input == "float16":   # the products leave fp16's range
            dist = "normal"
        case = _case(None, op, batch, bcast, M, N, K, input, slice, splits,
                     "triangular" if tri else "all", at, bt, dist)
        # no dearer than the largest listed case: products, and operands
        cost = work(case)["flops"] * {"int8": 1, "float32": 32}.get(slice, 2)
        words = batch * M * K + (1 if bcast else batch) * N * K
        if cost <= 4e12 and words <= 1 << 24 and batch * M * N <= 1 << 26:
            return case


def _matrix(g, batch, rows, cols, case, scale_dim):
    dt, dev = getattr(torch, case["input"]), "cuda"
    wide = torch.float64 if case["input"] == "float64" else torch.float32
    if case["dist"] in ("uniform", "outliers"):
        X = torch.rand(batch, rows, cols, generator=g, device=dev, dtype=wide) * 2 - 1
    else:
        X = torch.randn(batch, rows, cols, generator=g, device=dev, dtype=wide)
    if case["dist"] == "outliers":
        hit = torch.rand(batch, rows, cols, generator=g, device=dev) < 0.01
        X = torch.where(hit, X * 1e4, X)
    elif case["dist"] == "exp8":
        n = rows if scale_dim == 1 else cols
        e = torch.randint(-8, 9, (batch, n), generator=g, device=dev).to(wide)
        X = X * torch.exp2(e).unsqueeze(2 if scale_dim == 1 else 1)
    return X.to(dt)


def _inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    batch = case["batch"]
    A = _matrix(g, batch, case["M"], case["K"], case, 1)
    B = _matrix(g, 1 if case["bcast"] else batch, case["K"], case["N"], case, 2)
    if case["at"]:
        A = A.mT.contiguous().mT
    if case["bt"]:
        B = B.mT.contiguous().mT
    if case["op"] == "matmul" and batch == 1:
        return A[0], B[0]
    if case["bcast"]:
        return A, B[0]
    return A, B


def prepare(case, seed):
    A, B = _inputs(case, seed)
    slice = getattr(torch, case["slice"])
    state = dict(case=case, A=A, slice=slice)
    if case["op"] == "kept":
        # a linear layer's weights are stored [N, K]; their slices are made once
        state["alpha"] = ozk.compute_split_bits(
            case["K"], slice, torch.int32 if slice == torch.int8 else torch.float32)
        W = B.mT.contiguous().unsqueeze(0)
        state["W_slices"], state["W_scales"] = ozk.split_matrix(W, case["splits"], state["alpha"],
                                                                slice)
    else:
        state["B"] = B
    return state


def run(state):
    case = state["case"]
    L = case["splits"]
    if case["op"] == "kept":
        x_slices, x_scales = ozk.split_matrix(state["A"], L, state["alpha"], state["slice"])
        C = ozk.cross_gemm(x_slices, state["W_slices"].transpose(-1, -2), x_scales,
                           state["W_scales"], L, state["A"].dtype, pairs=case["pairs"])
        return x_slices, x_scales, C
    return ozk.ozaki_matmul(state["A"], state["B"], L, state["slice"], max_splits=max(4, L),
                            pairs=case["pairs"])


def exact(case, seed):
    A, B = _inputs(case, seed)
    C = torch.matmul(A.double().contiguous(), B.double().contiguous())
    return (None, None, C) if case["op"] == "kept" else C


def work(case):
    b, M, N, K, L = (case[k] for k in ("batch", "M", "N", "K", "splits"))
    x, s = _size(case["input"]), _size(case["slice"])
    nb = 1 if case["bcast"] else b
    if case["op"] == "kept":
        data = b * M * K * x + b * L * M * (K * s + 4) + nb * L * N * (K * s + 4)
    else:
        data = b * M * K * x + nb * N * K * x
    return {"bytes": data + b * M * N * x, "flops": 2.0 * _pairs(case) * b * M * N * K}


def tolerance(case):
    # int8 slices: integer products, exact sums and one defined order of the
    # scaled terms, so every correct implementation gives the same bits
    if case["slice"] == "int8":
        return "exact"
    # float slices: the fp32 sums over K in another order.  Measured between
    # two kernels that order them differently: 1.3e-7 at K = 300, 1.8e-6 at
    # K = 65536 (largest difference 6 times that); stated here: four times it
    rel = max(5e-7, 2.8e-8 * math.sqrt(case["K"]))
    if case["input"] in ("float64", "float32"):
        return {"rel": rel, "max": 8 * rel}
    # 16-bit results: a value moved across a rounding boundary is one unit in
    # the last place off, and few are
    return {"float16": {"rel": 4e-4, "max": 4e-3},
            "bfloat16": {"rel": 2e-3, "max": 3e-2}}[case["input"]]
