"""Performance cases of the matrix-multiplication path: what a program built on the C ABI of
include/sapphire_hip.h has it do, from one sample through a small network to the largest products.

Operands live in device memory that the caller owns (torch tensors here), the calls are enqueued
on the calling thread's stream, and nothing is read back inside a pass.  The kinds of work:

  mlp_forward   a stack of fully connected layers, bias and ReLU fused, one call per layer
  mlp_train     the same stack: forward, backward and the optimizer's step of every layer
  gemm_f32      one (batched) fp32 product, any size, storage order and out mode
  gemm_f16      the same with fp16 operands and fp32 accumulation
  spmm          CSR x dense
  csr           dense -> CSR -> dense
  spgemm        CSR x CSR -> CSR
"""
import math

import torch

from sapphire_amd import capi

DEVICE = "cuda"


def listed():
    return [
        # one request at a time through a small trained network (784 inputs, two hidden layers):
        # serving, where the latency of three dependent launches counts
        {"name": "mlp_forward_8", "kind": "mlp_forward", "batch": 8, "inputs": 784, "hidden": 1024,
         "outputs": 10},
        # the network of the three-layer benchmark configuration on its batch of 1024
        {"name": "mlp_forward_1024", "kind": "mlp_forward", "batch": 1024, "inputs": 784,
         "hidden": 1024, "outputs": 10},
        # the training step of that network: products with either operand transposed, column
        # sums, weight updates
        {"name": "mlp_train_1024", "kind": "mlp_train", "batch": 1024, "inputs": 784,
         "hidden": 1024, "outputs": 10},
        # the batched benchmark configuration: 16 matrices times one shared matrix, y += a b
        {"name": "gemm_f32_batch_16x512", "kind": "gemm_f32", "M": 512, "N": 512, "K": 512,
         "batch": 16, "shared_b": True, "trans_a": False, "trans_b": False, "overwrite": False},
        # the largest square fp32 product of the benchmark's table, y += a b
        {"name": "gemm_f32_4096", "kind": "gemm_f32", "M": 4096, "N": 4096, "K": 4096, "batch": 1,
         "shared_b": False, "trans_a": False, "trans_b": False, "overwrite": False},
        # nothing is a multiple of anything, and B is stored N x K: dx += dy W^T of an odd layer
        {"name": "gemm_f32_odd", "kind": "gemm_f32", "M": 1501, "N": 1203, "K": 1001, "batch": 1,
         "shared_b": False, "trans_a": False, "trans_b": True, "overwrite": False},
        # the headline benchmark: fp16 operands, a fresh y
        {"name": "gemm_f16_4096", "kind": "gemm_f16", "M": 4096, "N": 4096, "K": 4096, "batch": 1,
         "shared_b": False, "trans_a": False, "trans_b": False, "overwrite": True},
        # an odd fp16 product with B stored N x K, adding into y
        {"name": "gemm_f16_odd", "kind": "gemm_f16", "M": 2049, "N": 1500, "K": 1001, "batch": 1,
         "shared_b": False, "trans_a": False, "trans_b": True, "overwrite": False},
        # the sparse benchmark configuration: an 8192 x 8192 weight at 1 % times 256 columns
        {"name": "spmm_8192_256", "kind": "spmm", "M": 8192, "K": 8192, "N": 256,
         "density": 0.01},
        # a pruned 8192 x 8192 weight turned into CSR, and back
        {"name": "csr_8192", "kind": "csr", "M": 8192, "N": 8192, "density": 0.01},
        # sparse times sparse at the benchmark's size: 8 entries per row on both sides
        {"name": "spgemm_8192", "kind": "spgemm", "n": 8192, "per_row": 8},
        # the same on a wide matrix (a graph of 65536 nodes)
        {"name": "spgemm_65536", "kind": "spgemm", "n": 65536, "per_row": 8},
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["mlp_forward", "mlp_train", "gemm_f32", "gemm_f32", "gemm_f16", "gemm_f16",
                       "spmm", "csr", "spgemm"])
    if kind in ("mlp_forward", "mlp_train"):
        return {"kind": kind,
                "batch": _log_int(rng, 1, 4096) if kind == "mlp_forward" else _log_int(rng, 32, 2048),
                "inputs": _log_int(rng, 64, 1024), "hidden": _log_int(rng, 128, 2048),
                "outputs": _log_int(rng, 2, 256)}
    if kind in ("gemm_f32", "gemm_f16"):
        batch = rng.choice([1, 1, 1, _log_int(rng, 2, 16)])
        high = 4096 if batch == 1 else 1024
        return {"kind": kind, "M": _log_int(rng, 128, high), "N": _log_int(rng, 128, high),
                "K": _log_int(rng, 128, high), "batch": batch, "shared_b": rng.random() < 0.5,
                "trans_a": rng.random() < 0.3, "trans_b": rng.random() < 0.3,
                "overwrite": rng.random() < 0.5}
    if kind == "spmm":
        return {"kind": kind, "M": _log_int(rng, 512, 8192), "K": _log_int(rng, 512, 8192),
                "N": _log_int(rng, 16, 512),
                "density": math.exp(rng.uniform(math.log(0.002), math.log(0.02)))}
    if kind == "csr":
        return {"kind": kind, "M": _log_int(rng, 256, 8192), "N": _log_int(rng, 256, 8192),
                "density": math.exp(rng.uniform(math.log(0.001), math.log(0.1)))}
    n = _log_int(rng, 1024, 65536)
    # at most as many products as the widest listed case
    most = min(32, int(math.sqrt(65536 * 64 / n)))
    return {"kind": kind, "n": n, "per_row": _log_int(rng, 2, most)}


# ---- inputs ---------------------------------------------------------------------------------

def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    return g


def _uniform(g, shape, low, high):
    return torch.rand(shape, generator=g, device=DEVICE) * (high - low) + low


def _random_csr(g, rows, cols, entries):
    """CSR arrays of a rows x cols matrix with about `entries` entries at uniformly random places
    (distinct columns, ascending within a row), values U(-1, 1)."""
    keys = torch.unique(torch.randint(rows * cols, (entries,), generator=g, device=DEVICE))
    row = torch.zeros(rows + 1, dtype=torch.int64, device=DEVICE)
    row[1:] = torch.cumsum(torch.bincount(keys // cols, minlength=rows), 0)
    return {"V": _uniform(g, (keys.numel(),), -1.0, 1.0), "COL": (keys % cols).to(torch.int32),
            "ROW": row.to(torch.int32)}


def _prepare_gemm(case, g):
    half = case["kind"] == "gemm_f16"
    M, N, K, batch = case["M"], case["N"], case["K"], case["batch"]
    batch_b = 1 if case["shared_b"] else batch
    if half:
        # N(0, 1/sqrt(K)), the benchmark's fp16 operands
        a = (torch.randn((batch, M * K), generator=g, device=DEVICE) * K ** -0.5).half()
        b = (torch.randn((batch_b, K * N), generator=g, device=DEVICE) * K ** -0.5).half()
    else:
        a = _uniform(g, (batch, M * K), -1.0, 1.0)
        b = _uniform(g, (batch_b, K * N), -1.0, 1.0)
    flags = ((capi.SPH_GEMM_TRANS_A if case["trans_a"] else 0) |
             (capi.SPH_GEMM_TRANS_B if case["trans_b"] else 0) |
             (capi.SPH_GEMM_OVERWRITE if case["overwrite"] else 0))
    out = _uniform(g, (batch, M, N), -1.0, 1.0)
    return {"a": a, "b": b, "out": out,
            "entry": "sph_gemm_f16f32" if half else "sph_gemm_f32_ex",
            "args": (out.data_ptr(), a.data_ptr(), b.data_ptr(), M, N, K, batch, M * N, M * K,
                     0 if case["shared_b"] else K * N, flags)}


def _prepare_mlp(case, g):
    batch = case["batch"]
    sizes = [case["inputs"], case["hidden"], case["hidden"], case["outputs"]]
    state = {"batch": batch, "sizes": sizes, "x": _uniform(g, (batch, sizes[0]), 0.0, 1.0)}
    bound = [math.sqrt(6.0 / (i + o)) for i, o in zip(sizes, sizes[1:])]
    state["W"] = [_uniform(g, (i, o), -r, r) for i, o, r in zip(sizes, sizes[1:], bound)]
    state["b"] = [_uniform(g, (o,), -0.1, 0.1) for o in sizes[1:]]
    state["y"] = [torch.zeros((batch, o), device=DEVICE) for o in sizes[1:]]
    if case["kind"] == "mlp_train":
        state["target"] = _uniform(g, (batch, sizes[3]), -1.0, 1.0)
        state["dy"] = [torch.zeros((batch, o), device=DEVICE) for o in sizes[1:]]
        state["dx"] = [torch.zeros((batch, i), device=DEVICE) for i in sizes[:3]]
        state["ones"] = torch.ones(batch, device=DEVICE)
        # the reference's weight gradient is a sum over the batch; small enough that a long run
        # on one batch stays bounded
        state["rate"] = 0.1 / (batch * max(sizes))
    return state


def _prepare_spmm(case, g):
    M, K, N = case["M"], case["K"], case["N"]
    state = _random_csr(g, M, K, max(1, int(case["density"] * M * K)))
    state["B"] = _uniform(g, (K, N), -1.0, 1.0)
    state["out"] = torch.zeros((M, N), device=DEVICE)
    state["args"] = (state["out"].data_ptr(), state["V"].data_ptr(), state["COL"].data_ptr(),
                     state["ROW"].data_ptr(), M, K, N, state["B"].data_ptr(), 0)
    return state


def _prepare_csr(case, g):
    M, N = case["M"], case["N"]
    dense = _uniform(g, (M, N), -1.0, 1.0)
    # pruned: all but `density` of the weights set to zero, so a bound on their number is known
    dense = dense * (torch.rand((M, N), generator=g, device=DEVICE) < case["density"])
    mean = case["density"] * M * N
    count = min(M * N, int(mean + 8 * math.sqrt(mean)) + 16)
    state = {"dense": dense, "again": torch.zeros((M, N), device=DEVICE),
             "V": torch.zeros(count, device=DEVICE),
             "COL": torch.zeros(count, dtype=torch.int32, device=DEVICE),
             "ROW": torch.zeros(M + 1, dtype=torch.int32, device=DEVICE)}
    v, col, row = (state[k].data_ptr() for k in ("V", "COL", "ROW"))
    state["to_csr"] = (v, col, row, count, dense.data_ptr(), M, N, N, None)
    state["to_dense"] = (state["again"].data_ptr(), N, v, col, row, M, N)
    return state


def _prepare_spgemm(case, g):
    n = case["n"]
    a = _random_csr(g, n, n, n * case["per_row"])
    b = _random_csr(g, n, n, n * case["per_row"])
    # the bound a caller takes for the entries of the result: the number of products
    capacity = int(1.05 * n * case["per_row"] ** 2) + 1024
    state = {"a": a, "b": b, "V": torch.zeros(capacity, device=DEVICE),
             "COL": torch.zeros(capacity, dtype=torch.int32, device=DEVICE),
             "ROW": torch.zeros(n + 1, dtype=torch.int32, device=DEVICE)}
    state["args"] = (state["V"].data_ptr(), state["COL"].data_ptr(), state["ROW"].data_ptr(),
                     capacity, a["V"].data_ptr(), a["COL"].data_ptr(), a["ROW"].data_ptr(),
                     b["V"].data_ptr(), b["COL"].data_ptr(), b["ROW"].data_ptr(), n, n, n, None)
    return state


_PREPARE = {"mlp_forward": _prepare_mlp, "mlp_train": _prepare_mlp, "gemm_f32": _prepare_gemm,
            "gemm_f16": _prepare_gemm, "spmm": _prepare_spmm, "csr": _prepare_csr,
            "spgemm": _prepare_spgemm}


def prepare(case, seed):
    state = _PREPARE[case["kind"]](case, _generator(seed))
    state["kind"] = case["kind"]
    torch.cuda.synchronize()  # the library's stream does not wait for torch's
    return state


# ---- one pass -------------------------------------------------------------------------------

def _forward(s):
    x = s["x"]
    for l in range(3):
        capi.call("sph_linear_forward_f32", s["y"][l].data_ptr(), x.data_ptr(),
                  s["W"][l].data_ptr(), s["b"][l].data_ptr(), s["batch"], s["sizes"][l],
                  s["sizes"][l + 1], capi.SPH_LINEAR_RELU if l < 2 else 0)
        x = s["y"][l]


def _train(s):
    _forward(s)
    batch, sizes, rate = s["batch"], s["sizes"], s["rate"]
    # the squared error's gradient at the output
    capi.call("sph_sub_f32", s["dy"][2].data_ptr(), s["y"][2].data_ptr(), s["target"].data_ptr(),
              batch * sizes[3], 0, 0, 0)
    for l in (2, 1, 0):
        n_in, n_out = sizes[l], sizes[l + 1]
        x = s["y"][l - 1] if l > 0 else s["x"]
        dy, dx, W = s["dy"][l], s["dx"][l], s["W"][l]
        capi.call("sph_gemm_f32_ex", dx.data_ptr(), dy.data_ptr(), W.data_ptr(), batch, n_in,
                  n_out, 1, batch * n_in, batch * n_out, n_in * n_out,
                  capi.SPH_GEMM_TRANS_B | capi.SPH_GEMM_OVERWRITE)
        capi.call("sph_gemm_f32_sgd", W.data_ptr(), x.data_ptr(), dy.data_ptr(), n_in, n_out,
                  batch, 1.0, rate, capi.SPH_GEMM_TRANS_A)
        capi.call("sph_gemm_f32_sgd", s["b"][l].data_ptr(), s["ones"].data_ptr(), dy.data_ptr(), 1,
                  n_out, batch, 1.0 / batch, rate, 0)
        if l > 0:
            below = s["dy"][l - 1]
            capi.call("sph_fill_f32", below.data_ptr(), 0.0, batch * n_in)
            capi.call("sph_relu_backward_f32", below.data_ptr(), dx.data_ptr(), x.data_ptr(),
                      batch * n_in)


def run(state):
    kind = state["kind"]
    if kind == "mlp_forward":
        _forward(state)
        return state["y"]
    if kind == "mlp_train":
        _train(state)
        return {k: state[k] for k in ("y", "dx", "W", "b")}
    if kind in ("gemm_f32", "gemm_f16"):
        capi.call(state["entry"], *state["args"])
        return state["out"]
    if kind == "spmm":
        capi.call("sph_spmm_csr_f32", *state["args"])
        return state["out"]
    if kind == "csr":
        capi.call("sph_csr_from_dense_f32", *state["to_csr"])
        capi.call("sph_csr_to_dense_f32", *state["to_dense"])
        return {k: state[k] for k in ("V", "COL", "ROW", "again")}
    capi.call("sph_spgemm_f32", *state["args"])
    return {k: state[k] for k in ("V", "COL", "ROW")}


# ---- what a pass cannot do without ----------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind in ("gemm_f32", "gemm_f16"):
        M, N, K, batch = case["M"], case["N"], case["K"], case["batch"]
        size = 2 if kind == "gemm_f16" else 4
        batch_b = 1 if case["shared_b"] else batch
        return {"bytes": size * K * (batch * M + batch_b * N) +
                4 * batch * M * N * (1 if case["overwrite"] else 2),
                "flops": 2.0 * batch * M * N * K}
    if kind in ("mlp_forward", "mlp_train"):
        batch = case["batch"]
        sizes = [case["inputs"], case["hidden"], case["hidden"], case["outputs"]]
        weights = sum(i * o + o for i, o in zip(sizes, sizes[1:]))
        products = 2.0 * batch * sum(i * o for i, o in zip(sizes, sizes[1:]))
        if kind == "mlp_forward":
            # x and the parameters once, every layer's output once
            return {"bytes": 4 * (weights + batch * sum(sizes)), "flops": products}
        # parameters read and written; x, target in; y and dx of three layers out
        return {"bytes": 4 * (2 * weights + batch * (sizes[0] + sizes[3] + sum(sizes[1:]) +
                                                     sum(sizes[:3]))),
                "flops": 3 * products}
    if kind == "spmm":
        nnz = case["density"] * case["M"] * case["K"]
        return {"bytes": 8 * nnz + 4 * (case["M"] + 1) + 4 * case["N"] * (case["M"] + case["K"]),
                "flops": 2.0 * nnz * case["N"]}
    if kind == "csr":
        nnz = case["density"] * case["M"] * case["N"]
        # dense in, CSR out; CSR in, dense out
        return {"bytes": 8 * case["M"] * case["N"] + 2 * (8 * nnz + 4 * (case["M"] + 1)),
                "flops": 0.0}
    n, per_row = case["n"], case["per_row"]
    entries = n * n * -math.expm1(-per_row * per_row / n)  # distinct columns of a row's products
    return {"bytes": 8 * (2 * n * per_row + entries) + 12 * (n + 1),
            "flops": 2.0 * n * per_row * per_row}


def tolerance(case):
    # Exact or once-rounded products summed in fp32: what another order of the sums changes.
    # Measured against the same pass in fp64, over the listed and thirty drawn cases (relative
    # 2-norm, largest difference): fp32 up to 1.2e-6 and 1.1e-5 (4096^3), fp16 operands up to
    # 4.1e-7 and 3.5e-6; stated are four times these.  The sparse paths define the order of their
    # sums, so their values are the same bits.
    kind = case["kind"]
    if kind in ("gemm_f32", "mlp_forward"):
        return {"rel": 5e-6, "max": 5e-5}
    if kind == "gemm_f16":
        return {"rel": 2e-6, "max": 1.5e-5}
    if kind == "mlp_train":
        # about one hidden value in a million lies within a rounding of zero, and the gradient of
        # its ReLU is then one value or none: measured 4.6e-4 and 2.5e-2 on dx where that happened
        # (1e-6 and 1e-5 elsewhere); the largest difference grows as the layers get narrower
        return {"rel": 2e-3, "max": 0.5}
    return "exact"
