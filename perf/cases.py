"""Performance cases of the fused FFN operator, through its public entry points.

A case is one FFN: X [m, k] (or a permuted view of more dims), hidden width h, output width n,
storage type, activation, biases, down-projection, and the way a program calls it:

* entry 'prepared': the plan and the padded operands are made once (`prepare_ffn` /
  `prepare_eagle_ffn`) and a pass is one `run()`; weights and buffers are the program's to keep.
* entry 'call': a pass is one `ffn()` / `eagle_ffn_linear()` call on the caller's tensors, as a
  program does whose activations are new at every step.

Values are those of a trained layer's neighbourhood: X ~ N(0, 1), W1 ~ N(0, 1/k), W2 ~ N(0, 1/h),
biases ~ N(0, 0.1^2).
"""
from __future__ import annotations

import torch

from ffn_optim_amd import eagle_ffn_linear, ffn, prepare_eagle_ffn, prepare_ffn
from ffn_optim_amd.host.dispatch import NotApplicable

MAX_FLOPS = 4 * 8192 * 3072 * 12288


def _case(name, m, k, h, n, dtype, down="basic", act="gelu", gelu="erf", bias=False, entry="prepared",
          permuted=False):
    return {"name": name, "m": m, "k": k, "h": h, "n": n, "dtype": dtype, "down": down, "act": act, "gelu": gelu,
            "bias": bias, "entry": entry, "permuted": permuted}


def listed():
    return [
        # a small layer, where launches and latency are everything (the smoke workload)
        _case("smoke_fp16", 128, 256, 1024, 256, "float16"),
        # odd widths and a permuted 4-D activation, one-shot call: staging copies and all
        _case("call_ragged_fp16", 1005, 1000, 3001, 999, "float16", entry="call", permuted=True),
        # one decode step of a serving loop: new activations each step, weights read in place
        _case("call_decode_bf16", 16, 5120, 13824, 5120, "bfloat16", entry="call"),
        # the same layer prepared, Stream-K down: streams 283 MB of weights
        _case("decode_bf16", 16, 5120, 13824, 5120, "bfloat16", down="streamk"),
        # one GPU's share of that layer when H is split over eight
        _case("decode_shard_bf16", 16, 5120, 1728, 5120, "bfloat16"),
        # batched decode or a short prompt: 128 rows against wide weights
        _case("batch_bf16", 128, 4096, 16384, 4096, "bfloat16"),
        # a prompt chunk through a narrow layer with biases, Stream-K down
        _case("chunk_fp16", 512, 1024, 4096, 1024, "float16", down="streamk", bias=True),
        # odd widths again, prepared, the rational GELU option
        _case("ragged_fp16", 1005, 1000, 3001, 999, "float16", gelu="rational", permuted=True),
        # a mid-size transformer layer, everything aligned
        _case("aligned_bf16", 4096, 1024, 4096, 1024, "bfloat16"),
        # a gated (SwiGLU) layer with biases on a 2048-token prompt
        _case("swiglu_bf16", 2048, 3072, 8192, 3072, "bfloat16", act="swiglu", bias=True),
        # one GPU's share of a diffusion transformer's layer when H is split over eight
        _case("dit_shard_bf16", 8192, 3072, 1536, 3072, "bfloat16"),
        # the whole layer: the largest work
        _case("dit_bf16", 8192, 3072, 12288, 3072, "bfloat16", down="streamk"),
    ]


def _width(rng, lo, hi):
    """A width spread over its logarithm: half of them multiples of 256, a quarter of 8, the rest any."""
    v = lo * (hi / lo) ** rng.random()
    u = rng.random()
    unit = 256 if u < 0.5 else 8 if u < 0.75 else 1
    return max(unit, int(round(v / unit)) * unit)


def draw(rng):
    while True:
        m = max(1, int(round(8192 ** rng.random())))
        if rng.random() < 0.5:
            m = max(16, (m + 15) // 16 * 16)
        k, h = _width(rng, 256, 8192), _width(rng, 512, 16384)
        n = k if rng.random() < 0.75 else _width(rng, 256, 8192)
        act = rng.choice(("gelu", "gelu", "gelu", "silu", "swiglu"))
        entry = "call" if rng.random() < 0.2 else "prepared"
        case = _case("", m, k, h, n, rng.choice(("float16", "bfloat16", "bfloat16")),
                     down="streamk" if entry == "prepared" and rng.random() < 0.4 else "basic", act=act,
                     gelu=rng.choice(("erf", "erf", "rational")) if act == "gelu" else "erf",
                     bias=rng.random() < 0.3, entry=entry, permuted=m % 4 == 0 and rng.random() < 0.2)
        del case["name"]
        if work(case)["flops"] <= MAX_FLOPS:
            return case


def _inputs(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    dtype = getattr(torch, case["dtype"])

    def normal(shape, std):
        return (torch.randn(shape, generator=g, device="cuda") * std).to(dtype)

    m, k, h, n = case["m"], case["k"], case["h"], case["n"]
    u = 2 * h if case["act"] == "swiglu" else h
    if not case["permuted"]:
        x = normal((m, k), 1.0)
    elif m == 1005:
        x = normal((3, 67, 5, k), 1.0).transpose(1, 2)
    else:
        x = normal((m // 4, 4, k), 1.0).transpose(0, 1)
    w1, w2 = normal((u, k), k ** -0.5), normal((n, h), h ** -0.5)
    b1, b2 = (normal((u,), 0.1), normal((n,), 0.1)) if case["bias"] else (None, None)
    return x, w1, w2, b1, b2


def prepare(case, seed):
    x, w1, w2, b1, b2 = _inputs(case, seed)
    eagle = case["bias"] or case["act"] != "gelu"
    options = {} if case["gelu"] == "erf" else {"gelu": case["gelu"]}
    if case["entry"] == "call":
        return {"x": x, "w1": w1, "w2": w2, "b1": b1, "b2": b2, "act": case["act"] if eagle else None,
                "options": options}

    def make(down):
        if eagle:
            return prepare_eagle_ffn(x, w1, w2, b1, b2, activation=case["act"], down_impl=down, **options)
        return prepare_ffn(x, w1, w2, down_impl=down, **options)

    try:
        return {"prepared": make(case["down"])}
    except NotApplicable:  # Stream-K refuses outputs whose tiles divide the grid: Basic serves them
        return {"prepared": make("basic")}


def run(state):
    if "prepared" in state:
        return state["prepared"].run()
    if state["act"] is None:
        return ffn(state["x"], state["w1"], state["w2"], **state["options"])
    return eagle_ffn_linear(state["x"], state["w1"], state["w2"], state["b1"], state["b2"], state["act"],
                            **state["options"])


def work(case):
    m, k, h, n = case["m"], case["k"], case["h"], case["n"]
    u = 2 * h if case["act"] == "swiglu" else h
    biases = u + n if case["bias"] else 0
    return {"bytes": 2 * (m * k + u * k + n * h + m * n + biases), "flops": 2 * m * (u * k + h * n)}


def tolerance(case):
    # The hidden activation and the output are rounded to the storage type once each; two correct
    # kernels differ where a sum lands on the other side of a rounding boundary.  Four times what
    # whole, split and K-sliced sums of these cases differ by: rel 3.0e-4 and max 7.8e-3 (bf16),
    # 1.4e-4 and 9.8e-4 (fp16).
    if case["dtype"] == "bfloat16":
        return {"rel": 1.2e-3, "max": 3.2e-2}
    return {"rel": 6e-4, "max": 4e-3}


def _gelu_rational(z):
    t = (z * 0.5 ** 0.5).clamp(-3.92, 3.92)
    t2 = t * t
    p = q = None
    for c in (0.053443748819, 7.5517016694, 101.62808918, 1393.8061484, 5063.7915060, 29639.384698):
        p = torch.full_like(t2, c) if p is None else p * t2 + c
    for c in (1.0, 31.212858877, 398.56963806, 3023.1248150, 13243.365831, 26267.224157):
        q = torch.full_like(t2, c) if q is None else q * t2 + c
    return 0.5 * z * (1.0 + t * p / q)


def exact(case, seed):
    x, w1, w2, b1, b2 = _inputs(case, seed)
    x, w1, w2 = x.double(), w1.double(), w2.double()
    z = x.reshape(-1, case["k"]) @ w1.t()
    if b1 is not None:
        z = z + b1.double()
    if case["act"] == "swiglu":
        hidden = torch.nn.functional.silu(z[:, :case["h"]]) * z[:, case["h"]:]
    elif case["act"] == "silu":
        hidden = torch.nn.functional.silu(z)
    elif case["gelu"] == "rational":
        hidden = _gelu_rational(z)
    else:
        hidden = 0.5 * z * torch.special.erfc(-z * 0.5 ** 0.5)
    y = hidden @ w2.t()
    if b2 is not None:
        y = y + b2.double()
    return y.reshape(*x.shape[:-1], case["n"])
