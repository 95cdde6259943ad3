"""The workloads on which this package's speed is measured: what users of a fused SwiGLU run, through the public entry
points, from one decoded token to the largest training step.

A case is a dict:
  api        "function": FusedSwiGLU.apply / FastAccumFusedSwiGLU.apply on weights [d, i];
             "swiglu":   the SwiGLU module;   "mlp": the SwiGLUMLP module (SwiGLU and the down projection behind it)
  train      True: forward and backward, with every gradient;   False: forward only, under no_grad
  batch, seq, d, i   x is [batch, seq, d], d_intermediate is i
  dtype      "bf16" or "fp16"
  linear     (modules) the weights are stored like nn.Linear's, [out, in]
  packed     (modules) gate and up weights are one parameter
  recompute  (modules, train) no pre-activations are kept between forward and backward
"""
import math

import torch

from fusedswiglu_amd import FastAccumFusedSwiGLU, FusedSwiGLU, SwiGLU, SwiGLUMLP

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
FUNCTIONS = {"bf16": FusedSwiGLU, "fp16": FastAccumFusedSwiGLU}


def _case(name, api, train, batch, seq, d, i, dtype="bf16", linear=False, packed=False, recompute=False):
    c = dict(api=api, train=train, batch=batch, seq=seq, d=d, i=i, dtype=dtype, linear=linear, packed=packed,
             recompute=recompute)
    return dict(c, name=name) if name else c


def listed():
    return [
        # a few sequences decoded on a small model: launches and host time count
        _case("decode_8_small", "function", False, 8, 1, 1024, 3072),
        # one token through a whole gated MLP block that adopted a checkpoint's nn.Linear weights
        _case("decode_1_mlp", "mlp", False, 1, 1, 4096, 11008, linear=True),
        # batched decoding on the largest weights of the benchmark: weight streaming
        _case("decode_16_large", "function", False, 16, 1, 8192, 28672),
        # a large decode batch or a short prompt: between weight streaming and matrix-core bound
        _case("prompt_256_large", "function", False, 1, 256, 8192, 28672),
        # one prompt of odd length through an MLP block
        _case("prompt_777_mlp", "mlp", False, 1, 777, 4096, 11008, dtype="fp16", linear=True),
        # training steps of the reference's published sweep (batch 4, sequence 2048, i = 3 d): its smallest width ...
        _case("step_256", "function", True, 4, 2048, 256, 768),
        # ... a small model's ...
        _case("step_1024", "function", True, 4, 2048, 1024, 3072),
        # ... and its largest: the headline benchmark
        _case("step_4096", "function", True, 4, 2048, 4096, 12288),
        # fp16 with a ragged intermediate dimension, as in the benchmark
        _case("step_4096_fp16", "function", True, 2, 4096, 4096, 11008, dtype="fp16"),
        # i = int(8 d / 3) without rounding it up, as many small models have it: rows that are not 16-byte aligned
        _case("step_unaligned", "function", True, 2, 1024, 1024, 2730),
        # fine-tuning a whole MLP block on packed nn.Linear weights, pre-activations recomputed to save memory
        _case("step_mlp_recompute", "mlp", True, 1, 4096, 2048, 5632, linear=True, packed=True, recompute=True),
        # the largest training step of the benchmark
        _case("step_8192", "function", True, 8, 4096, 8192, 28672),
    ]


def _log(rng, low, high):
    return math.exp(rng.uniform(math.log(low), math.log(high)))


def draw(rng):
    """Another workload of the same ranges: decoding 1-128 tokens, prompts of 129-4096, training steps of 256-32768;
    d 256-8192 (1024 up for inference), i 2-4 times d; one in six with dimensions that are not multiples of 8."""
    kind = rng.choice(["decode", "prompt", "train", "train"])
    unaligned = rng.random() < 1 / 6
    most_flops = 6e11 if unaligned else (2.5e13 if kind == "train" else 4e12)
    while True:
        low_t, high_t = {"decode": (1, 128), "prompt": (129, 4096), "train": (256, 32768)}[kind]
        tokens = round(_log(rng, low_t, high_t))
        multiple = rng.choice([1, 2]) if unaligned else rng.choice([128, 64, 8])
        d = max(multiple, round(_log(rng, 256 if kind == "train" else 1024, 8192) / multiple) * multiple)
        i = max(multiple, round(d * rng.uniform(2, 4) / multiple) * multiple)
        api = rng.choice(["function", "function", "swiglu", "mlp"])
        if (12 if kind == "train" else 4) * tokens * d * i * (1.5 if api == "mlp" else 1) <= most_flops and i <= 28672:
            break
    batch = 1
    if kind == "decode":
        batch = tokens
    elif kind == "train":
        batch = rng.choice([1, 2, 4])
    seq = max(1, tokens // batch)
    module = api != "function"
    return _case(None, api, kind == "train", batch, seq, d, i, dtype=rng.choice(["bf16", "bf16", "fp16"]),
                 linear=module and rng.random() < 0.7, packed=module and rng.random() < 0.4,
                 recompute=module and kind == "train" and rng.random() < 0.3)


def prepare(case, seed):
    """x and the upstream gradient ~ N(0, 1), weights ~ N(0, 1 / fan_in), on the GPU."""
    dtype, d, i = DTYPES[case["dtype"]], case["d"], case["i"]
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape, std=1.0):
        return torch.empty(shape, device="cuda", dtype=dtype).normal_(0.0, std, generator=gen)

    x = normal(case["batch"], case["seq"], d)
    if case["api"] == "function":
        weights = [normal(d, i, std=d ** -0.5), normal(d, i, std=d ** -0.5)]
        fn, call = FUNCTIONS[case["dtype"]], None
    else:
        kind = SwiGLU if case["api"] == "swiglu" else SwiGLUMLP
        call = kind(d, i, dtype=dtype, device="cuda", packed=case["packed"], recompute=case["recompute"],
                    weights_out_in=case["linear"])
        weights, fn = list(call.parameters()), None
        with torch.no_grad():
            for name, w in call.named_parameters():
                w.normal_(0.0, (i if name == "w_down" else d) ** -0.5, generator=gen)
    state = dict(x=x, weights=weights, fn=fn, call=call, grad=None)
    if case["train"]:
        state["grad"] = normal(case["batch"], case["seq"], d if case["api"] == "mlp" else i)
        x.requires_grad_(True)
        for w in weights:
            w.requires_grad_(True)
    return state


def _forward(state):
    if state["call"] is not None:
        return state["call"](state["x"])
    return state["fn"].apply(state["x"], *state["weights"])


def run(state):
    """The output; for a training step the gradients of x and of every weight as well."""
    if state["grad"] is None:
        with torch.no_grad():
            return _forward(state)
    out = _forward(state)
    return [out.detach(), *torch.autograd.grad(out, [state["x"], *state["weights"]], state["grad"])]


def work(case):
    """Inputs read once, outputs written once; 2*t*d*i per matrix product.  Recomputing the two forward products is part
    of a step that keeps no pre-activations."""
    t, d, i = case["batch"] * case["seq"], case["d"], case["i"]
    mlp = case["api"] == "mlp"
    weights = (3 if mlp else 2) * d * i
    x, out = t * d, t * (d if mlp else i)
    products = 3 if mlp else 2
    if not case["train"]:
        return {"bytes": 2 * (x + weights + out), "flops": 2 * t * d * i * products}
    return {"bytes": 2 * (2 * x + 2 * weights + 2 * out),
            "flops": 2 * t * d * i * (3 * products + (2 if case["recompute"] else 0))}


def tolerance(case):
    """About four times the error seen against the same formula in float64 on the same inputs (bf16: 1.7e-3 to 3.1e-3, the
    largest single difference 1.5e-2; fp16: 2e-4 to 4.3e-4 and 2.7e-3)."""
    return {"rel": 1e-2, "max": 0.06} if case["dtype"] == "bf16" else {"rel": 1.5e-3, "max": 0.011}
