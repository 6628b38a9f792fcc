"""Performance cases of the fused FP8 MoE layer and of the activation quantiser before it.

One case is one call of a public entry point on resident inputs, as a serving or prefill loop
makes it for every MoE layer of a model: H=7168, I=2048, 32 local of 256 experts, top-8. The
token count is the only size that varies in use; the routing (even or skewed), the rank's
expert window, the router bias and output types and the entry point vary with the program.
Inputs follow the layer's own workload generator: N(0,1) hidden states quantised per token and
128 columns, N(0,0.02) weights quantised per 128x128 block, N(0,1) logits, N(0,0.1) bias.

  entry "run"         run(): a Python program's call. Up to 256 tokens it streams the packed copy
                      of the weight set that its first call with the set builds and keeps.
  entry "run_packed"  run() with a packed copy that the program made itself and keeps.
  entry "abi"         moe_fp8_run of the C ABI on the row-major weights, with the argument struct
                      and the workspace that a native program keeps: also what run() launches
                      above 256 tokens and for weight sets beyond those it keeps copies of.
  entry "quantise"    quantize_hidden(): hidden states to the layer's fp8 activations and scales.
"""
import math

import torch

import __graft_entry__

pkg = __graft_entry__.load_package()
from mlsys26_flashinfer_moe_amd import _lib, inputs  # noqa: E402

HIDDEN, INTER, EXPERTS, LOCAL, TOP_K, GROUPS, KEPT_GROUPS = 7168, 2048, 256, 32, 8, 8, 4
SCALING = 2.5
BOOSTED = (3, 11, 19, 27)   # local experts whose bias is raised to +3.0 in a skewed batch
MAX_TOKENS = 14107
MAX_SKEWED_TOKENS = 4096

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _layer(name, tokens, offset=0, skew=False, bias="bf16", out="bf16", entry="run"):
    return dict(name=name, entry=entry, tokens=tokens, offset=offset, skew=skew, bias=bias, out=out)


def listed():
    return [
        # one sequence being decoded: a handful of experts, latency and launches decide
        _layer("decode_1", 1),
        # a few sequences decoded together (or one with speculative tokens), on a later rank
        _layer("decode_7", 7, offset=96),
        # small decode batches: the weights of ten to twenty-odd experts stream from HBM
        _layer("decode_16", 16),
        _layer("decode_64", 64),
        # the same batch from a native program on the row-major weights (the layers of a deep
        # model that have no packed copy), float32 bias
        _layer("decode_64_rowmajor", 64, bias="f32", entry="abi"),
        # an odd batch above 64 tokens, nearly every local expert touched, float32 output
        _layer("decode_80_f32", 80, offset=32, out="f32", entry="run_packed"),
        # a chunked-prefill step of ragged size on a middle rank, fp16 bias
        _layer("chunk_901", 901, offset=64, bias="f16"),
        # a round prefill chunk
        _layer("chunk_2048", 2048, offset=128, entry="abi"),
        # four hot experts that take most of the assignments
        _layer("prefill_4096_skew", 4096, skew=True),
        # ordinary and long prefill
        _layer("prefill_8192", 8192),
        _layer("prefill_14107", 14107, offset=224),
        # the step before the layer for a prefill batch
        dict(name="quantise_8192", entry="quantise", tokens=8192, hidden="bf16"),
    ]


def _log_tokens(rng, top):
    return min(top, int(round(math.exp(rng.uniform(0.0, math.log(top + 0.49))))))


def draw(rng):
    kind = rng.random()
    if kind < 0.1:
        return dict(entry="quantise", tokens=_log_tokens(rng, MAX_TOKENS), hidden=rng.choice(("bf16", "bf16", "f16", "f32")))
    skew = kind > 0.85
    tokens = _log_tokens(rng, MAX_SKEWED_TOKENS if skew else MAX_TOKENS)
    entry = rng.choice(("run", "run", "run", "abi", "run_packed"))
    return dict(entry=entry, tokens=tokens, offset=LOCAL * rng.randrange(EXPERTS // LOCAL), skew=skew,
                bias=rng.choice(("bf16", "bf16", "f32", "f16")), out=rng.choice(("bf16", "bf16", "bf16", "f32")))


def _local(case, logits, bias):
    """The local expert of every assignment that falls on this rank."""
    local = _route(logits, bias)[0] - case["offset"]
    return local[(local >= 0) & (local < LOCAL)]


def _activations(case, seed, device):
    # a batch that gives this rank something to do (a batch of a few tokens often does not): the
    # first such of the seed's batches
    for batch in range(64):
        logits, bias, hq, hs = inputs.make_activations(case["tokens"], 2 * seed + 1 + (batch << 32), device,
                                                       case["offset"], BOOSTED if case["skew"] else ())
        bias = bias.to(DTYPES[case["bias"]])
        if _local(case, logits, bias).numel():
            break
    return logits, bias, hq, hs


def _hidden(case, seed, device):
    gen = torch.Generator(device=device)
    gen.manual_seed(2 * seed + 1)
    x = torch.randn((case["tokens"], HIDDEN), generator=gen, device=device, dtype=torch.float32)
    return x.to(DTYPES[case["hidden"]])


def prepare(case, seed):
    device = torch.device("cuda")
    T = case["tokens"]
    if case["entry"] == "quantise":
        return dict(entry="quantise", x=_hidden(case, seed, device),
                    q=torch.empty((T, HIDDEN), dtype=torch.float8_e4m3fn, device=device),
                    scale=torch.empty((HIDDEN // 128, T), dtype=torch.float32, device=device))
    logits, bias, hq, hs = _activations(case, seed, device)
    w13, s13, w2, s2 = inputs.make_weights(2 * seed, device)
    out = torch.empty((T, HIDDEN), dtype=DTYPES[case["out"]], device=device)
    args = (logits, bias, hq, hs, w13, s13, w2, s2, case["offset"], SCALING, out)
    state = dict(entry=case["entry"], args=args, out=out)
    if case["entry"] == "run_packed":
        state["packed"] = pkg.pack_weights(w13, w2)
    elif case["entry"] == "abi":
        state["struct"] = pkg.make_args(*args)
        state["workspace"] = pkg.Workspace(T, device)
    return state


def run(state):
    entry = state["entry"]
    if entry == "quantise":
        return pkg.quantize_hidden(state["x"], out=state["q"], out_scale=state["scale"])
    if entry == "run":
        pkg.run(*state["args"])
    elif entry == "run_packed":
        pkg.run_packed(*state["args"], packed_weights=state["packed"])
    else:
        ws = state["workspace"]
        _lib.check(_lib.load().moe_fp8_run(state["struct"], ws.ptr, ws.nbytes, torch.cuda.current_stream().cuda_stream),
                   "moe_fp8_run")
    return state["out"]


def _route(logits, bias):
    """(ids, weights) [T, 8] of the grouped top-8 routing, in 64 bits."""
    T = logits.shape[0]
    score = torch.sigmoid(logits.double())
    biased = score + bias.double()
    group = biased.view(T, GROUPS, EXPERTS // GROUPS).topk(2, dim=-1).values.sum(-1)
    kept = torch.zeros_like(group, dtype=torch.bool).scatter_(1, group.topk(KEPT_GROUPS, dim=-1).indices, True)
    masked = biased.masked_fill(~kept.repeat_interleave(EXPERTS // GROUPS, dim=1), float("-inf"))
    ids = masked.topk(TOP_K, dim=-1).indices
    w = score.gather(1, ids)
    return ids, w / (w.sum(-1, keepdim=True) + 1e-20) * SCALING


def work(case):
    T = case["tokens"]
    if case["entry"] == "quantise":
        read = T * HIDDEN * DTYPES[case["hidden"]].itemsize
        return {"bytes": read + T * HIDDEN + T * (HIDDEN // 128) * 4, "flops": 0}
    # the experts that a batch touches and its local assignments follow from its routing: the
    # mean over four batches of the same distribution
    touched = rows = batches = 0
    for seed in range(256):
        gen = torch.Generator().manual_seed(seed)
        logits = torch.randn((T, EXPERTS), generator=gen)
        bias = torch.randn((EXPERTS,), generator=gen) * 0.1
        if case["skew"]:
            for e in BOOSTED:
                bias[case["offset"] + e] = 3.0
        local = _local(case, logits, bias)
        if local.numel():
            touched += local.unique().numel()
            rows += local.numel()
            batches += 1
        if batches == 4:
            break
    expert = 3 * INTER * HIDDEN + 4 * 3 * (INTER // 128) * (HIDDEN // 128)   # W13, W2 and their block scales
    token = 4 * EXPERTS + HIDDEN + 4 * (HIDDEN // 128) + HIDDEN * DTYPES[case["out"]].itemsize
    return {"bytes": touched / batches * expert + T * token + EXPERTS * DTYPES[case["bias"]].itemsize,
            "flops": rows / batches * 2 * 3 * INTER * HIDDEN}


def tolerance(case):
    # the quantiser's scale and rounding are defined bit by bit
    if case["entry"] == "quantise":
        return "exact"
    # against the same algorithm with its sums in 64 bits: up to 0.0033 and 0.07 over all cases,
    # where a sum at the edge of two fp8 codes of the requantised intermediate takes the other
    return {"rel": 0.012, "max": 0.28}


def _expert(w, s, e):
    """Expert e's weights in 64 bits: the fp8 values times their 128x128 block scales."""
    v = w[e].float().double()
    R, C = v.shape
    return (v.view(R // 128, 128, C // 128, 128) * s[e].double()[:, None, :, None]).view(R, C)


def exact(case, seed):
    device = torch.device("cuda") if torch.cuda.is_available() else torch.device("cpu")
    if case["entry"] == "quantise":
        x = _hidden(case, seed, device).double().view(case["tokens"], HIDDEN // 128, 128)
        scale = (x.abs().amax(-1) / 448.0).clamp_min(1e-12)
        q = (x / scale[..., None]).float().to(torch.float8_e4m3fn).double()
        return q.view(case["tokens"], HIDDEN), scale.t().contiguous()
    logits, bias, hq, hs = _activations(case, seed, device)
    w13, s13, w2, s2 = inputs.make_weights(2 * seed, device)
    ids, weights = _route(logits, bias)
    T = case["tokens"]
    x = (hq.float().double().view(T, HIDDEN // 128, 128) * hs.double().t()[..., None]).view(T, HIDDEN)
    out = torch.zeros((T, HIDDEN), dtype=torch.float64, device=device)
    for e in range(LOCAL):
        token, slot = (ids == case["offset"] + e).nonzero(as_tuple=True)
        if token.numel():
            h = x[token] @ _expert(w13, s13, e).t()
            act = torch.nn.functional.silu(h[:, INTER:]) * h[:, :INTER]
            out.index_add_(0, token, (act @ _expert(w2, s2, e).t()) * weights[token, slot][:, None])
    return out
