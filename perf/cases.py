"""Performance cases: what programs that use this library have it do, at the sizes they have.

listed() is a fixed selection, draw() gives further cases of the same ranges, prepare() makes what a
program has in hand before the call, run() is one pass through the public entry points.  A case is a
dict of plain values:

  kind     which program (see run)
  experts, rows (over all experts, after top-k routing), hidden_in, hidden_out
  dtype    element type of activations and weights
  trans_b  weights stored (experts, hidden_out, hidden_in)
  zipf     skew of the routing: expert popularity falls with rank ** -zipf (0: every expert alike);
           the row counts are drawn from it, so they are ragged in every case
  empty    experts that no row is routed to
  host     batch_sizes in host memory instead of on the device
  top_k    kinds that permute: rows per token
"""
import math

import numpy as np
import torch

from grouped_gemm_amd import backend, ops

_DTYPES = {"bfloat16": torch.bfloat16, "float16": torch.float16, "float8_e4m3fn": torch.float8_e4m3fn}


def _case(kind, experts, rows, hidden_in, hidden_out, dtype="bfloat16", trans_b=False, zipf=0.0, empty=0, host=False,
          top_k=1, name=None):
    case = dict(kind=kind, experts=experts, rows=rows, hidden_in=hidden_in, hidden_out=hidden_out, dtype=dtype,
                trans_b=trans_b, zipf=zipf, empty=empty, host=host, top_k=top_k)
    if name is not None:
        case["name"] = name
    return case


def listed():
    return [
        # The smallest layer the operator's own tests train: three launches, all latency, row counts
        # in host memory as a router that runs on the host leaves them.
        _case("train", 8, 1024, 128, 128, host=True, name="train tiny"),
        # A small expert layer in mixed-precision fp16, a few thousand rows per device (fine-tuning,
        # small micro-batches): less than one tile per compute unit.
        _case("train", 32, 4096, 768, 2048, dtype="float16", trans_b=True, name="train small fp16"),
        # The headline workload: Mixtral-8x7B w1, 16384 tokens top-2, forward and both gradients.
        _case("train", 8, 32768, 4096, 14336, name="train mixtral w1"),
        # Fine-grained ragged experts: 8192 tokens top-6 with Zipf popularity and idle experts.
        _case("train", 64, 49152, 2048, 1408, zipf=1.2, empty=4, name="train ragged"),
        # A DeepSeek-V3-style share of one device: many experts of about 256 rows each, weights
        # stored transposed, most of the time spent moving weights and weight gradients.
        _case("train", 256, 65536, 7168, 2048, trans_b=True, name="train many experts"),
        # Gradient accumulation of a trainer that keeps fp32 main gradients.
        _case("accumulate", 8, 32768, 4096, 14336, name="accumulate fp32 gradient"),
        # An expert layer that hands its token permutation to the library: gather in the first
        # product's loads, scatter in the second's stores, with all gradients.
        _case("permuted", 64, 49152, 2048, 1408, top_k=6, name="train gather scatter"),
        # A gated (SwiGLU) expert layer in training: both products and all gradients.
        _case("gated", 16, 16384, 2048, 4096, name="train gated"),
        # Hidden sizes that are odd numbers (any size is allowed): a training step at a middling size.
        _case("train", 8, 8192, 2047, 5461, name="train odd sizes"),
        # Token generation, a batch of 64 at top-2 over few large experts: the gated expert layer
        # with the permutation fused, a handful of rows per expert, all weights read.
        _case("serve gated", 8, 128, 4096, 14336, top_k=2, name="decode gated"),
        # Token generation over many experts, two rows each, weights stored transposed.
        _case("forward", 256, 512, 7168, 2048, trans_b=True, name="decode many experts"),
        # Prefill with fp8 weights and activations, stored depth-contiguous as the matrix units take them.
        _case("forward", 8, 32768, 4096, 14336, dtype="float8_e4m3fn", trans_b=True, name="prefill fp8"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _hidden(rng, lo, hi, kind, dtype):
    """A hidden size: usually a multiple of 64 or 8, for the plain two-byte products also any even or odd one."""
    n = _log_uniform(rng, lo, hi)
    if dtype == "float8_e4m3fn":
        return max(16, n // 16 * 16)
    pick = rng.random()
    if pick < 0.5:
        return max(64, n // 64 * 64)
    if pick < 0.75 or kind not in ("train", "forward"):
        return max(8, n // 8 * 8)
    return max(8, n // 2 * 2) if pick < 0.88 else max(9, n // 2 * 2 + 1)


def _seconds(case):
    """A rough cost, to keep drawn cases below the listed ones."""
    w = work(case)
    return w["bytes"] / 4e12 + w["flops"] / 1e15


def draw(rng):
    most = {key: max(work(c)[key] for c in listed()) for key in ("bytes", "flops")}
    most_seconds = max(_seconds(c) for c in listed())
    while True:
        kind = rng.choice(["train", "train", "train", "forward", "forward", "accumulate", "permuted", "gated", "serve gated"])
        dtype = "float16" if rng.random() < 0.2 else "bfloat16"
        if kind == "forward" and rng.random() < 0.4:
            dtype = "float8_e4m3fn"
        top_k = rng.choice([1, 2, 4, 6, 8]) if kind in ("permuted", "serve gated") else 1
        experts = _log_uniform(rng, 4, 256)
        lo, hi = {"forward": (32, 65536), "serve gated": (16, 8192)}.get(kind, (512, 65536))
        rows = max(1, _log_uniform(rng, lo, hi) // top_k) * top_k
        trans_b = rng.random() < 0.5
        case = _case(kind, experts, rows, _hidden(rng, 128, 7168, kind, dtype), _hidden(rng, 128, 14336, kind, dtype),
                     dtype=dtype, trans_b=trans_b and kind != "accumulate", zipf=rng.choice([0.0, 0.0, 0.6, 1.2]),
                     empty=rng.choice([0, 0, experts // 16]), host=rng.random() < 0.25, top_k=top_k)
        w = work(case)
        if w["bytes"] <= most["bytes"] and w["flops"] <= most["flops"] and _seconds(case) <= most_seconds:
            return case


# ------------------------------------------------------------------------------- inputs


def _row_counts(case, rng):
    experts = case["experts"]
    p = np.arange(1, experts + 1, dtype=np.float64) ** -case["zipf"]
    p[experts - case["empty"]:] = 0.0
    p = p[rng.permutation(experts)]
    return torch.from_numpy(rng.multinomial(case["rows"], p / p.sum()).astype(np.int64))


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]
    experts, rows, hin, hout = case["experts"], case["rows"], case["hidden_in"], case["hidden_out"]
    kind, trans_b = case["kind"], case["trans_b"]
    train = kind in ("train", "permuted", "gated")

    def randn(*shape, scale=1.0, grad=False):
        made = torch.float16 if dtype == torch.float16 else torch.bfloat16
        t = torch.randn(shape, dtype=made, device="cuda", generator=gen).mul_(scale).to(dtype)
        return t.requires_grad_(grad)

    def weights(k, n, grad=False):
        # products keep about the size of their inputs; fp8 weights fill their format's range, as
        # weights with a scale per tensor do
        scale = 1.0 if dtype == torch.float8_e4m3fn else k ** -0.5
        return randn(*((experts, n, k) if trans_b else (experts, k, n)), scale=scale, grad=grad)

    counts = _row_counts(case, rng)
    s = {"kind": kind, "trans_b": trans_b, "sizes": counts if case["host"] else counts.cuda()}
    if kind == "train":
        s.update(a=randn(rows, hin, grad=True), b=weights(hin, hout, True), upstream=randn(rows, hout, scale=0.1))
    elif kind == "forward":
        s.update(a=randn(rows, hin), b=weights(hin, hout))
    elif kind == "accumulate":
        s.update(a=randn(rows, hin), upstream=randn(rows, hout, scale=0.1),
                 main_grad=torch.randn(experts, hin, hout, device="cuda", generator=gen))
    elif kind == "gated":
        s.update(x=randn(rows, hin, grad=True), w13=weights(hin, 2 * hout, True), w2=weights(hout, hin, True),
                 upstream=randn(rows, hin, scale=0.1))
    else:
        # token t holds the routed rows t * top_k .. + top_k - 1; `order` lists them by expert
        expert_of = torch.repeat_interleave(torch.arange(experts), counts)[torch.from_numpy(rng.permutation(rows))]
        order = torch.argsort(expert_of, stable=True).to("cuda", torch.int32)
        s.update(order=order, token_of=order // case["top_k"], rows=rows)
        tokens = rows // case["top_k"]
        first = hout if kind == "permuted" else 2 * hout
        s.update(x=randn(tokens, hin, grad=train), w13=weights(hin, first, train), w2=weights(hout, hin, train))
        if train:
            s["upstream"] = randn(rows, hin, scale=0.1)
    return s


# ------------------------------------------------------------------------------- passes


def run(s):
    kind, sizes, trans_b = s["kind"], s["sizes"], s["trans_b"]
    if kind == "train":
        out = ops.gmm(s["a"], s["b"], sizes, trans_b)
        return (out, *torch.autograd.grad(out, (s["a"], s["b"]), s["upstream"]))
    if kind == "forward":
        with torch.no_grad():
            return ops.gmm(s["a"], s["b"], sizes, trans_b)
    if kind == "accumulate":
        return backend.accumulate_weight_gradient(s["a"], s["upstream"], sizes, s["main_grad"])
    if kind == "gated":
        h = ops.gmm_swiglu(s["x"], s["w13"], sizes, trans_b)
        out = ops.gmm(h, s["w2"], sizes, trans_b)
        return (out, *torch.autograd.grad(out, (s["x"], s["w13"], s["w2"]), s["upstream"]))
    if kind == "permuted":
        h = ops.gmm_gather(s["x"], s["w13"], sizes, s["token_of"], trans_b)
        h = torch.nn.functional.gelu(h, approximate="tanh")
        out = ops.gmm_scatter(h, s["w2"], sizes, s["order"], trans_b)
        return (out, *torch.autograd.grad(out, (s["x"], s["w13"], s["w2"]), s["upstream"]))
    if kind == "serve gated":
        h = backend.gmm_swiglu(s["x"], s["w13"], sizes, trans_b=trans_b, a_rows=s["token_of"])
        out = torch.empty(s["rows"], s["x"].shape[1], dtype=h.dtype, device=h.device)
        return backend.gmm_indexed(h, s["w2"], sizes, trans_b=trans_b, c=out, c_rows=s["order"])
    raise ValueError("unknown kind of case: %r" % kind)


# ------------------------------------------------------------------------------- bounds


def work(case):
    e, r, k, n = case["experts"], case["rows"], case["hidden_in"], case["hidden_out"]
    kind, tokens = case["kind"], case["rows"] // case["top_k"]
    size = 1 if case["dtype"] == "float8_e4m3fn" else 2
    # experts that rows are routed to (their weights are read): the expectation for even routing
    busy = (e - case["empty"]) * (1.0 - (1.0 - 1.0 / max(1, e - case["empty"])) ** r)
    if kind == "train":      # a, upstream and b in; the product and both gradients out
        return {"flops": 6.0 * r * k * n, "bytes": 2.0 * (2 * r * k + 2 * r * n + (busy + e) * k * n)}
    if kind == "forward":
        return {"flops": 2.0 * r * k * n, "bytes": size * (r * k + busy * k * n) + 2.0 * r * n}
    if kind == "accumulate":   # the fp32 gradient is read and written
        return {"flops": 2.0 * r * k * n, "bytes": 2.0 * (r * k + r * n) + 8.0 * busy * k * n}
    if kind == "gated":
        return {"flops": 18.0 * r * k * n, "bytes": 2.0 * (4 * r * k + 3 * (busy + e) * k * n)}
    if kind == "permuted":
        return {"flops": 12.0 * r * k * n, "bytes": 2.0 * (2 * tokens * k + 2 * r * k + 2 * (busy + e) * k * n) + 8.0 * r}
    return {"flops": 6.0 * r * k * n, "bytes": 2.0 * (tokens * k + r * k + 3 * busy * k * n) + 8.0 * r}


def tolerance(case):
    """About four times the distance from a float64 computation (rounding where the path rounds is
    not repeated there), measured at 256 to 2048 deep products: bf16 rel 1.7e-3 and max 3.9e-3 for
    one rounding of fp32 sums, up to 3.4e-3 and 2.4e-2 for a chain of products whose intermediate
    results are rounded; fp16 an eighth of that; fp32 accumulation rel 3.8e-7 at 4000 rows."""
    if case["kind"] == "accumulate":   # fp32 sums in another order, over up to 65536 rows
        return {"rel": 1e-5, "max": 5e-5}
    chain = case["kind"] in ("gated", "permuted", "serve gated")
    if case["dtype"] == "float16":
        return {"rel": 1.7e-3, "max": 1.2e-2} if chain else {"rel": 1e-3, "max": 2e-3}
    return {"rel": 1.3e-2, "max": 0.1} if chain else {"rel": 7e-3, "max": 1.6e-2}
