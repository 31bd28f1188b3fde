"""The workloads that the library's speed is measured on, and how one pass of
each is made, run and judged.

A pass is one call of a launcher of kernels.so on tensors that are resident
on the GPU, on torch's current stream: what a program that keeps its latents
and its K and V on the device does per layer (O = softmax(Q K^T / sqrt(768)) V,
single head, dim 768).  The split-K launchers take their scratch from the
caller, who keeps it between calls, and the number of splits that the split-K
drivers take by default (choose_num_splits at the device's CU count).
"""

import ctypes
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "fast-cuda-cross-attention_amd"))
import cuda_wrappers as cw  # noqa: E402

D = 768
# type of Q, K and V -> (torch type, bytes per value)
TYPES = {"fp32": (torch.float32, 4), "fp16": (torch.float16, 2), "bf16": (torch.bfloat16, 2)}
# (type, splits given by the caller) -> launcher
ENTRY = {
    ("fp32", False): "launch_optimized_kernel",
    ("fp16", False): "launch_wmma_kernel",
    ("bf16", False): "launch_wmma_bf16_kernel",
    ("fp32", True): "launch_splitk_kernel",
    ("fp16", True): "launch_wmma_splitk_kernel",
    ("bf16", True): "launch_wmma_splitk_bf16_kernel",
}
# Costliest listed case, in (batch, latent, key) units: 32 x 1024 x 784 in
# fp32; a 16-bit unit costs about a fifth of that.
MOST_UNITS = 32 * 1024 * 784


def _case(name, dtype, batch, n_latent, n_input, splitk=False):
    case = {"dtype": dtype, "batch": batch, "n_latent": n_latent, "n_input": n_input,
            "splitk": splitk}
    if name:
        case["name"] = name
    return case


def listed():
    return [
        # One image's 28 x 28 grid into the smallest latent bank: the smallest
        # call, where launches and latency count.
        _case("fp32-b1-nl64-ni784", "fp32", 1, 64, 784),
        # The single-batch sweep over the size of the latent bank, at its middle.
        _case("fp32-b1-nl512-ni784", "fp32", 1, 512, 784),
        # The batched grid, at its middle.
        _case("fp32-b8-nl512-ni784", "fp32", 8, 512, 784),
        # The batched grid's largest point, the benchmark's headline.
        _case("fp32-b32-nl1024-ni784", "fp32", 32, 1024, 784),
        # A pixel array of 224 x 224 as the input of one latent bank.
        _case("fp32-b1-nl256-ni50176", "fp32", 1, 256, 50176),
        # The key-parallel launcher on a middling long input.
        _case("fp32-splitk-b1-nl256-ni4096", "fp32", 1, 256, 4096, True),
        # Sizes that are multiples of nothing.
        _case("fp32-b3-nl197-ni1025", "fp32", 3, 197, 1025),
        # The smallest call in 16 bits.
        _case("fp16-b1-nl64-ni784", "fp16", 1, 64, 784),
        # The reduced-precision configuration, in the training type.
        _case("bf16-b16-nl512-ni784", "bf16", 16, 512, 784),
        # The headline's shape in 16 bits: the largest 16-bit call.
        _case("bf16-b32-nl1024-ni784", "bf16", 32, 1024, 784),
        # A long input through the 16-bit key-parallel launcher.
        _case("fp16-splitk-b1-nl256-ni16384", "fp16", 1, 256, 16384, True),
        # A ragged batch of middling size in 16 bits.
        _case("bf16-b5-nl333-ni2047", "bf16", 5, 333, 2047),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """Batch 1 to 32, 32 to 1,024 latents, 196 to 50,176 keys, in the three
    types, a quarter of the cases through the split-K launchers; one size in
    three is rounded to a multiple of 16, as grids and latent banks often are."""
    while True:
        sizes = [_log_int(rng, 1, 32), _log_int(rng, 32, 1024), _log_int(rng, 196, 50176)]
        for i in (1, 2):
            if rng.random() < 1 / 3:
                sizes[i] = max(16, sizes[i] // 16 * 16)
        if sizes[0] * sizes[1] * sizes[2] <= MOST_UNITS:
            break
    return _case(None, rng.choice(["fp32", "fp16", "bf16"]), *sizes, rng.random() < 0.25)


def _inputs(case, seed):
    """Q, K, V of the case's type: standard normal; latents of a long-input
    layer are at their initial scale (0.02).  The 16-bit launchers take Q
    scaled by 1/sqrt(768)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype, _ = TYPES[case["dtype"]]

    def normal(rows):
        return torch.randn(case["batch"], rows, D, generator=gen, device="cuda")

    q, k, v = normal(case["n_latent"]), normal(case["n_input"]), normal(case["n_input"])
    if case["n_input"] >= 4096:
        q *= 0.02
    if dtype != torch.float32:
        q /= math.sqrt(D)
    return q.to(dtype), k.to(dtype), v.to(dtype)


def prepare(case, seed):
    q, k, v = _inputs(case, seed)
    batch, nl, ni = case["batch"], case["n_latent"], case["n_input"]
    out = torch.empty(batch, nl, D, device="cuda")
    fn = getattr(cw.lib, ENTRY[case["dtype"], case["splitk"]])
    tensors, tail = [q, k, v, out], [batch, nl, ni, D]
    if case["splitk"]:
        cu, _ = cw.device_info(torch.cuda.current_device())
        splits = cw.choose_num_splits(nl, ni, batch, sm_count=cu,
                                      latents_per_block=4 if case["dtype"] == "fp32" else 16)
        tensors += [torch.empty(batch, nl, splits, D, device="cuda"),
                    torch.empty(batch, nl, splits, device="cuda"),
                    torch.empty(batch, nl, splits, device="cuda")]
        tail.append(splits)
    args = [ctypes.cast(t.data_ptr(), kind) for t, kind in zip(tensors, fn.argtypes)]
    return {"launch": fn, "args": args + tail, "tensors": tensors, "out": out}


def run(state):
    state["launch"](*state["args"], torch.cuda.current_stream().cuda_stream)
    return state["out"]


def work(case):
    batch, nl, ni = case["batch"], case["n_latent"], case["n_input"]
    _, size = TYPES[case["dtype"]]
    return {"bytes": batch * ((nl + 2 * ni) * D * size + nl * D * 4),
            "flops": 4 * batch * nl * ni * D}


def tolerance(case):
    """fp32: sums of up to 50,176 products in another order.  16 bits: each
    softmax weight is rounded to the type against a reference that an
    implementation is free to choose.  About four times what two such
    evaluations differ by."""
    return TOLERANCE[case["dtype"]]


TOLERANCE = {"fp32": {"rel": 5e-6, "max": 5e-5},
             "fp16": {"rel": 8e-4, "max": 4e-3},
             "bf16": {"rel": 8e-3, "max": 6e-2}}


def exact(case, seed):
    q, k, v = _inputs(case, seed)
    scale = 1.0 if case["dtype"] != "fp32" else 1.0 / math.sqrt(D)
    out = torch.empty(case["batch"], case["n_latent"], D, dtype=torch.float64, device="cuda")
    for b in range(case["batch"]):
        scores = q[b].double() @ k[b].double().t().contiguous() * scale
        out[b] = torch.softmax(scores, dim=-1) @ v[b].double()
    return out
