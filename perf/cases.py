"""Performance cases of the fused sequence+depth attention operators: the calls that models built on them make.

Every case goes through the package's public entry points as a model does -- ``parallel_moda`` and its chunk-visible
and depth-only variants, ``parallel_attn``, ``DepthStream``, ``MoDAStack`` -- forward and backward through autograd
where the model trains, forward alone where it serves.  A case is a dict of plain values:

  path    moda | chunk | fda | attn | stream | stack   (which entry point)
  grad    forward + backward, or forward alone
  dtype   bf16 | fp16 | fp32
  B, T    batch size, tokens per sequence;  lens: comma-separated sequence lengths of a packed batch (B = 1)
  H, G    key/value heads, query heads per key/value head
  D, L    head dim, depth slots per token (stream, stack: layers)
  causal  False for the vision models

Inputs are 0.5 * N(0, 1) and the upstream gradient N(0, 1), as in the benchmark configurations.
"""
import math

import torch

import moda_amd

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_SIZES = {"bf16": 2, "fp16": 2, "fp32": 4}
# relative error (2-norm) that another correct implementation at the same precision shows: results rounded to 8 or 11
# bits of mantissa from P and dS rounded alike; fp32 sums in another order
_REL = {"bf16": 1e-2, "fp16": 2e-3, "fp32": 1e-5}

_PACKED_LENGTHS = [16384] + [8192] * 2 + [4096] * 4 + [2048] * 8


def _case(path, B, T, H, G, D, L, causal=True, dtype="bf16", grad=True, lens=""):
    return {"path": path, "B": B, "T": T, "H": H, "G": G, "D": D, "L": L, "causal": causal, "dtype": dtype,
            "grad": grad, "lens": lens}


def listed():
    cases = {
        # the smallest calls: a unit-test-sized ragged shape of the reference's own test matrix; launches and host
        # time are all of it
        "small-fp16-train": _case("moda", 2, 95, 4, 2, 64, 8, dtype="fp16"),
        # the fp32 configuration (gradient checks, CPU comparisons, fp32 fine-tuning of small models)
        "fp32-train": _case("moda", 1, 256, 4, 1, 64, 4, dtype="fp32"),
        # language-model training step at an ordinary context length, GQA 4
        "lm-4k-train": _case("moda", 2, 4096, 4, 4, 128, 8),
        # chunk-visible variant, 24-layer-deep depth stream, 64-row chunks
        "chunk-16k-train": _case("chunk", 1, 16384, 4, 4, 128, 24),
        # the long-context headline
        "lm-64k-train": _case("moda", 1, 65536, 4, 4, 128, 24),
        # vision transformer layer (196 patches + class token), non-causal, one query head per key/value head
        "vision-train": _case("moda", 64, 197, 6, 1, 64, 12, causal=False),
        # depth-only attention on the same tensors
        "vision-depth-only-train": _case("fda", 64, 197, 6, 1, 64, 12, causal=False),
        # the reference's published benchmark row: head dim 64, 64 query heads on 8, 64 depth slots, 16K tokens
        "lm-d64-16k-train": _case("moda", 1, 16384, 8, 8, 64, 64),
        # documents of different lengths packed on one token axis
        "packed-64k-train": _case("moda", 1, sum(_PACKED_LENGTHS), 4, 4, 128, 24, lens=",".join(map(str, _PACKED_LENGTHS))),
        # plain causal attention with head-dim GQA, the layers of a model that carry no depth stream
        "plain-16k-train": _case("attn", 1, 16384, 4, 4, 128, 0),
        # the twelve layers of the smallest vision model chained through one depth stream, training
        "vision-stream-train": _case("stream", 64, 197, 1, 4, 64, 12, causal=False),
        # the same model's blocks (attention + MLP) serving: forward alone, depth cache filled in place
        "vision-stack-infer": _case("stack", 64, 197, 1, 4, 64, 12, causal=False, grad=False),
    }
    return [dict(c, name=n) for n, c in cases.items()]


def _between(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm, odd as often as even."""
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    top = next(c for c in listed() if c["name"] == "lm-64k-train")
    limit = work(top)
    while True:
        c = _draw_any(rng)
        w = work(c)
        # wide heads and small launches run at a lower rate than the largest listed case: leave room for that
        if w["flops"] <= limit["flops"] / 4 and w["bytes"] <= limit["bytes"] / 2:
            return c


def _draw_any(rng):
    kind = rng.choice(["small", "fp32", "lm", "lm", "chunk", "vision", "fda", "packed", "attn", "stream", "stack"])
    half = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "small":
        return _case("moda", rng.randint(1, 6), _between(rng, 32, 256), rng.randint(1, 8), rng.choice([1, 2, 4, 8]), 64,
                     rng.randint(0, 16), dtype=half)
    if kind == "fp32":
        return _case("moda", rng.randint(1, 2), _between(rng, 64, 1024), rng.randint(2, 8), rng.choice([1, 2, 4]),
                     rng.choice([64, 128]), rng.randint(0, 12), causal=rng.random() < 0.7, dtype="fp32",
                     grad=rng.random() < 0.8)
    if kind == "lm":
        return _case("moda", rng.randint(1, 4), _between(rng, 512, 49152), rng.choice([2, 4, 8]), rng.choice([1, 2, 4, 8]),
                     rng.choice([64, 64, 96, 128, 128, 256]), rng.choice([0, 4, 8, 12, 16, 24, 32, 64]), dtype=half,
                     grad=rng.random() < 0.8)
    if kind == "chunk":
        return _case("chunk", rng.randint(1, 2), _between(rng, 512, 24576), rng.choice([2, 4, 8]), rng.choice([1, 2, 4, 8]),
                     rng.choice([64, 128, 128]), rng.choice([4, 8, 12, 24]), dtype=half, grad=rng.random() < 0.8)
    if kind in ("vision", "fda"):
        return _case("moda" if kind == "vision" else "fda", _between(rng, 4, 128), rng.choice([50, 145, 197, 257, 401, 577]),
                     rng.choice([1, 2, 3, 6]), rng.choice([1, 2, 4]), 64, rng.randint(1, 24), causal=False, dtype=half,
                     grad=rng.random() < 0.8)
    if kind == "packed":
        lens = [_between(rng, 64, 8192) for _ in range(rng.randint(2, 16))]
        return _case("moda", 1, sum(lens), rng.choice([2, 4, 8]), rng.choice([1, 2, 4]), rng.choice([64, 128, 128]),
                     rng.choice([4, 8, 12, 24]), dtype=half, grad=rng.random() < 0.8, lens=",".join(map(str, lens)))
    if kind == "attn":
        return _case("attn", rng.randint(1, 4), _between(rng, 512, 32768), rng.choice([2, 4, 8]), rng.choice([1, 2, 4, 8]),
                     rng.choice([64, 128, 128]), 0, dtype=half, grad=rng.random() < 0.8)
    return _case(kind, _between(rng, 4, 64), rng.choice([50, 145, 197, 257]), rng.choice([1, 2]), rng.choice([2, 4]), 64,
                 rng.randint(6, 12), causal=False, grad=kind == "stream")


def _randn(gen, dtype, std, *shape):
    x = torch.empty(shape, dtype=dtype, device="cuda")
    flat, step = x.view(-1), 1 << 26  # in pieces, which bounds the fp32 temporaries
    for i in range(0, flat.numel(), step):
        n = min(step, flat.numel() - i)
        flat[i:i + n] = torch.randn(n, generator=gen, device="cuda") * std
    return x


def prepare(case, seed):
    B, T, H, G, D, L = (case[n] for n in ("B", "T", "H", "G", "D", "L"))
    dt, grad, path = _DTYPES[case["dtype"]], case["grad"], case["path"]
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def given(*shape, std=0.5):
        return _randn(gen, dt, std, *shape).requires_grad_(grad)

    if path == "stack":
        dim = H * G * D
        torch.manual_seed(seed)
        with torch.device("cuda"):
            model = moda_amd.MoDAStack(dim, L, H * G, H).to(dt)
        return {"case": case, "model": model.eval(), "x": _randn(gen, dt, 0.5, B, T, dim)}
    if path == "stream":
        layers = [(given(B, T * G, H, D), given(B, T, H, D), given(B, T, H, D)) for _ in range(L)]
        return {"case": case, "layers": layers, "do": [_randn(gen, dt, 1.0, B, T * G, H, D) for _ in range(L)]}
    rows, heads = (T, H * G) if path == "attn" else (T * G, H)
    s = {"case": case, "q": given(B, rows, heads, D), "scale": None, "cu": None}
    if case["dtype"] == "fp32":  # unit inputs, the scale folded into q
        s["q"] = given(B, rows, heads, D, std=D ** -0.5)
        s["scale"] = 1.0
    std = 1.0 if case["dtype"] == "fp32" else 0.5
    s["k"] = s["v"] = s["kd"] = s["vd"] = None
    if path != "fda":
        s["k"], s["v"] = given(B, T, H, D, std=std), given(B, T, H, D, std=std)
    if L:
        s["kd"], s["vd"] = given(B, T * L, H, D, std=std), given(B, T * L, H, D, std=std)
    if case["lens"]:
        ends = [0]
        for n in case["lens"].split(","):
            ends.append(ends[-1] + int(n))
        s["cu"] = torch.tensor(ends, dtype=torch.int32, device="cuda")
    if grad:
        s["do"] = _randn(gen, dt, 1.0, B, rows, heads, D)
    return s


def run(state):
    case = state["case"]
    path, G = case["path"], case["G"]
    if path == "stack":
        with torch.no_grad():
            return state["model"](state["x"])
    if path == "stream":
        stream = moda_amd.DepthStream(case["L"])
        outs = []
        for q, k, v in state["layers"]:
            outs.append(stream.attend(q, k, v, moda_group_num=G, is_causal=case["causal"]))
            stream.push(k, v)
        return outs, torch.autograd.grad(outs, [x for layer in state["layers"] for x in layer], state["do"])
    q, k, v, kd, vd = (state[n] for n in ("q", "k", "v", "kd", "vd"))
    if path == "attn":
        out = o = moda_amd.parallel_attn(q, k, v, scale=state["scale"])
    else:
        common = dict(cached_k=kd, cached_v=vd, scale=state["scale"], moda_group_num=G, need_lse=True, warn_shape=False)
        if path == "fda":
            out = moda_amd.parallel_fda(q, **common)
        elif path == "chunk":
            out = moda_amd.parallel_moda_chunk_visible(q, k, v, **common)
        else:
            out = moda_amd.parallel_moda(q, k, v, cu_seqlens=state["cu"], is_causal=case["causal"], **common)
        o = out[0]
    if not case["grad"]:
        return out
    return out, torch.autograd.grad(o, [x for x in (q, k, v, kd, vd) if x is not None], state["do"])


def _pairs(case):
    """(query token, key) pairs of one head: sequence keys, then depth slots."""
    T, L, path = case["T"], case["L"], case["path"]
    lens = [int(n) for n in case["lens"].split(",")] if case["lens"] else [T]
    seq = 0 if path == "fda" else sum(n * (n + 1) // 2 if case["causal"] or path == "attn" else n * n for n in lens)
    if path == "chunk":
        full, rem = divmod(T, 64 // case["G"])
        cb = 64 // case["G"]
        return seq, L * (full * cb * (cb + 1) // 2 + rem * (rem + 1) // 2)
    return seq, T * L


def work(case):
    """Operations: two products of every visible pair forward, five backward.  Bytes: inputs and outputs once."""
    B, T, H, G, D, L, e = (*(case[n] for n in ("B", "T", "H", "G", "D", "L")), _SIZES[case["dtype"]])
    units = 7 if case["grad"] else 2
    rows, keys = B * T * G * H * D * e, B * T * H * D * e
    seq, dep = _pairs(case)
    if case["path"] == "stack":
        dim, tokens = H * G * D, B * T
        weights = L * (dim * (2 * dim + 2 * H * D) + 8 * dim * dim)
        seen = L * T * T + T * (L * (L - 1) // 2)
        return {"bytes": 2 * tokens * dim * e + weights * e, "flops": 2 * tokens * weights + 4 * D * B * H * G * seen}
    if case["path"] == "stream":
        seen = L * seq + T * (L * (L - 1) // 2)
        return {"bytes": L * (4 * rows + 4 * keys), "flops": 2 * D * B * H * G * units * seen}
    with_keys, with_depth = case["path"] != "fda", L > 0
    moved = 2 * rows + 2 * keys * with_keys + 2 * L * keys * with_depth + 4 * B * T * G * H
    if case["grad"]:
        moved += 2 * rows + 2 * keys * with_keys + 2 * L * keys * with_depth
    return {"bytes": moved, "flops": 2 * D * B * H * G * units * (seq + dep)}


def tolerance(case):
    return {"rel": _REL[case["dtype"]]}
