"""The work that users of this layer have it do, as cases that can be timed and compared.

Every case is one forward pass of the MoE layer through the `flashMoeLauncher` extension
(`MoeKernelLauncher.create` once, `launch` per pass), on weights ~ N(0, 0.02) and token rows
~ N(0, 1) as in `synth.CONFIGS`, with inputs and outputs resident in device memory.

A case is a dict of
  T, H, E, k, I   tokens of the pass, hidden size, experts, top-k, expert intermediate size
  dtype           "bf16" or "f32": weights, tokens and output
  weights         how the launcher is given the expert weights: "in_place" (packed where they
                  lie, FLAG_WEIGHTS_PREPACKED), "copy" (the default of `create`: the launcher
                  keeps a packed copy) or "row_major" (flags = 0)
  edges           True: RMSNorm in front of the layer and the residual behind it
  hot             experts whose router logit carries a fixed +3.0 bias (0: no router bias)
  max_tokens      the batch the launcher is sized for
"""
import torch

import flashMoeLauncher

HOT_BIAS = 3.0
SIGMA_W = 0.02
NORM_EPS = 1e-6

# Layer shapes of synth.CONFIGS
QWEN3_30B = dict(H=2048, E=128, k=8, I=768)
QWEN3_235B = dict(H=4096, E=128, k=8, I=1536)
TINY = dict(H=256, E=8, k=2, I=128)


def _case(T, shape, dtype="bf16", weights="in_place", edges=False, hot=0, max_tokens=None):
    return dict(T=T, dtype=dtype, weights=weights, edges=edges, hot=hot,
                max_tokens=max_tokens or T, **shape)


def listed():
    named = [
        # the layer of the CPU comparison and of the first test anyone runs: launch latency only
        ("tiny_f32_16", _case(16, TINY, dtype="f32", weights="copy")),
        # one sequence being decoded: the latency of a single token, eight experts
        ("decode_1", _case(1, QWEN3_30B, weights="copy", max_tokens=256)),
        # a handful of sequences, about half of the experts in use
        ("decode_11", _case(11, QWEN3_30B, max_tokens=256)),
        # the decode batch the headline number is quoted on
        ("decode_64", _case(64, QWEN3_30B)),
        # a decode batch of a caller that leaves its tensors as they are
        ("decode_48_row_major", _case(48, QWEN3_30B, weights="row_major", max_tokens=256)),
        # a busy decode batch, the layer as the whole MoE half of a pre-norm block
        ("decode_200_block", _case(200, QWEN3_30B, edges=True, max_tokens=256)),
        # a short prompt, or decode mixed with a chunk of a prompt
        ("chunk_600", _case(600, QWEN3_30B, weights="copy")),
        # chunked prefill on the caller's tensors
        ("chunk_2048_row_major", _case(2048, QWEN3_30B, weights="row_major")),
        # long prefill
        ("prefill_8192", _case(8192, QWEN3_30B)),
        # the large model's layer: chunked prefill
        ("large_4096", _case(4096, QWEN3_235B)),
        # prefill with four experts that draw half of all rows
        ("imbalance_16384", _case(16384, QWEN3_30B, hot=4)),
        # the dtype of the reference-shaped entry point, with its packed copy
        ("f32_1024", _case(1024, QWEN3_30B, dtype="f32", weights="copy")),
    ]
    return [dict(name=name, **case) for name, case in named]


# No drawn case may ask for more than the largest listed ones: 1.25 TFLOP in bf16
# (imbalance_16384), 78 GFLOP in float32 (f32_1024), 2.42 G expert weights (large_4096).
_MAX_FLOPS = {"bf16": 1.24e12, "f32": 7.7e10}
_MAX_WEIGHTS = 3 * 128 * 4096 * 1536


def _flops(case):
    return case["T"] * case["k"] * 6 * case["H"] * case["I"] + 2 * case["T"] * case["H"] * case["E"]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    while True:
        family = rng.choice(["30b", "30b", "30b", "235b", "f32", "other"])
        dtype = "bf16"
        weights = rng.choice(["in_place", "copy", "row_major"])
        hot = rng.choice([0, 0, 0, 4])
        if family == "30b":
            shape, T = dict(QWEN3_30B), _log_int(rng, 1, 16384)
        elif family == "235b":
            shape, T = dict(QWEN3_235B), _log_int(rng, 1, 4096)
        elif family == "f32":
            shape, T, dtype = dict(QWEN3_30B), _log_int(rng, 1, 1024), "f32"
        else:
            # any admitted shape: H a multiple of 64, I of 32, any number of experts
            E = _log_int(rng, 8, 256)
            shape = dict(H=64 * rng.randint(4, 64), E=E, k=rng.randint(1, min(E, 10)), I=32 * rng.randint(4, 64))
            T = _log_int(rng, 1, 8192)
            dtype = rng.choice(["bf16", "bf16", "bf16", "f32"])
        case = _case(T, shape, dtype=dtype, weights=weights, edges=rng.random() < 0.25, hot=hot,
                     max_tokens=max(T, 256) if rng.random() < 0.5 else T)
        if _flops(case) <= _MAX_FLOPS[dtype] and 3 * shape["E"] * shape["H"] * shape["I"] <= _MAX_WEIGHTS:
            return case


def _dtype(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float32


def prepare(case, seed):
    dev, dt = torch.device("cuda:0"), _dtype(case)
    gen = torch.Generator(device=dev)
    gen.manual_seed(int(seed))

    def normal(sigma, *shape):
        return torch.empty(shape, dtype=dt, device=dev).normal_(0.0, sigma, generator=gen)

    T, H, E, k, I = case["T"], case["H"], case["E"], case["k"], case["I"]
    gate = normal(SIGMA_W, E, H)
    ffn1 = normal(SIGMA_W, E, 2 * I, H)
    ffn2 = normal(SIGMA_W, E, H, I)
    tokens = normal(1.0, T, H)
    bias = norm_weight = None
    if case["hot"]:
        chosen = torch.randperm(E, generator=torch.Generator().manual_seed(int(seed)))[:case["hot"]]
        bias = torch.zeros(E, dtype=torch.float32)
        bias[chosen] = HOT_BIAS
        bias = bias.to(dev)
    flags = {"in_place": flashMoeLauncher.FLAG_WEIGHTS_PREPACKED,
             "copy": flashMoeLauncher.FLAG_PACK_WEIGHTS,
             "row_major": 0}[case["weights"]]
    if case["edges"]:
        flags |= flashMoeLauncher.FLAG_RMSNORM | flashMoeLauncher.FLAG_RESIDUAL
        norm_weight = (1.0 + normal(0.1, H).float()).to(dt)
    if case["weights"] == "in_place":
        flashMoeLauncher.pack_weights_in_place(ffn1, ffn2)
    launcher = flashMoeLauncher.MoeKernelLauncher()
    launcher.create(gate, ffn1, ffn2, case["max_tokens"], launcher.getDistributedUniqueId(empty=True), 0, 1,
                    top_k=k, router_bias=bias, flags=flags, norm_weight=norm_weight, norm_eps=NORM_EPS)
    return dict(launcher=launcher, tokens=tokens, output=torch.empty_like(tokens))


def run(state):
    state["launcher"].launch(state["tokens"], state["output"])
    return state["output"]


def work(case):
    """Each weight of the experts that are expected to be in use read once, the router's weights
    and the token rows read once, the output rows written once."""
    T, H, E, k, I = case["T"], case["H"], case["E"], case["k"], case["I"]
    size = 2 if case["dtype"] == "bf16" else 4
    used = E * (1.0 - (1.0 - k / E) ** T)
    return {"bytes": (used * 3 * H * I + E * H + 2 * T * H) * size, "flops": float(_flops(case))}


def tolerance(case):
    # Against the layer in float64 on the same routing: bf16 2.9e-3 / 1.6e-2 (h, the slots' rows
    # and the output are rounded to bf16), float32 1.8e-6 / 1.2e-5; four times that.
    return {"rel": 1.1e-2, "max": 6e-2} if case["dtype"] == "bf16" else {"rel": 7e-6, "max": 5e-5}
