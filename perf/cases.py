"""The work that users of the fused FP8 MoE layer have it do, as timed cases.

One case is one call of the layer on one expert-parallel shard, through
``flashinfer_amd.kernel.run`` (FP8 activations with their block scales) or
``flashinfer_amd.kernel.run_bf16`` (bf16 activations, quantised by the call).
The sizes run from one decode token to the largest prefill batch of the
repository's benchmark; the layers are the definitions the repository builds.

A case holds

* ``layer``: one of ``LAYERS``;
* ``entry``: ``run`` or ``run_bf16``;
* ``T``: tokens of the batch;
* ``offset``: first global expert of the shard;
* ``spread``: how tokens choose experts. ``even``: independent N(0,1) logits
  with a small per-expert bias. ``same``: every token chooses the shard's
  first experts (a shard that holds the hot experts, the repository's skewed
  workload). ``owned``: as ``even``, and each token surely chooses ``owned``
  of the shard's experts (a batch of a few tokens that was sent to this shard
  because it holds their experts);
* ``owned``: see above, 0 otherwise.
"""
from __future__ import annotations

import torch

from flashinfer_amd import kernel

# H, I, experts of the shard, all experts, groups, groups kept, experts per token
LAYERS = {
    "h7168_i2048": (7168, 2048, 32, 256, 8, 4, 8),
    "h7168_i2048_e64": (7168, 2048, 64, 256, 8, 4, 8),
    "h4096_i1536": (4096, 1536, 32, 256, 8, 4, 8),
    "h4096_i1536_e16_g128": (4096, 1536, 16, 128, 8, 3, 6),
}
MAX_T = 14000
BLOCK = 128
SCALING = 2.5
FP8 = torch.float8_e4m3fn


def _case(name, T, layer="h7168_i2048", entry="run", offset=0, spread="even", owned=0):
    return {"name": name, "layer": layer, "entry": entry, "T": T, "offset": offset,
            "spread": spread, "owned": owned}


def listed():
    return [
        # one decoding user: one token, two of its experts on this shard
        _case("decode_1", 1, spread="owned", owned=2),
        # a handful of decoding users
        _case("decode_4", 4, spread="owned", owned=1),
        # small serving batches, on shards other than the first too
        _case("decode_16", 16, offset=32),
        _case("decode_64", 64),
        # a decode batch whose requests all want the same experts
        _case("decode_64_same", 64, spread="same"),
        # the smaller layer of another family, an odd batch
        _case("decode_37_g128", 37, layer="h4096_i1536_e16_g128", offset=16),
        # the layer over 4 GPUs instead of 8, activations still in bf16
        _case("decode_130_e64_bf16", 130, layer="h7168_i2048_e64", entry="run_bf16", offset=64),
        # a large decode batch / a short prompt
        _case("mixed_256", 256),
        # a prefill chunk with an odd number of tokens, on an inner shard
        _case("chunk_1000", 1000, offset=64),
        # a long ragged prompt on the smaller hidden size
        _case("prefill_3001_h4096", 3001, layer="h4096_i1536", offset=96),
        # full prefill batch
        _case("prefill_8192", 8192),
        # the largest: a prefill batch that all goes to this shard's experts
        _case("prefill_14000_same", 14000, spread="same"),
    ]


def draw(rng):
    layer = rng.choice(sorted(LAYERS))
    el, eg = LAYERS[layer][2:4]
    T = int(round(MAX_T ** rng.random()))
    spread = "same" if rng.random() < 0.2 else "even"
    owned = 0
    if spread == "even" and T <= 8:
        spread, owned = "owned", rng.randint(1, 2)
    return {"layer": layer, "entry": "run_bf16" if rng.random() < 0.2 else "run", "T": T,
            "offset": el * rng.randrange(eg // el), "spread": spread, "owned": owned}


def _logits(case, g, device):
    _, _, el, eg, _, _, _ = LAYERS[case["layer"]]
    T, off = case["T"], case["offset"]
    logits = torch.randn(T, eg, generator=g, device=device)
    bias = torch.randn(eg, generator=g, device=device) * 0.1
    if case["spread"] == "same":
        bias[off:off + 8] = 3.0
    if case["owned"]:
        own = torch.rand(T, el, generator=g, device=device).argsort(dim=1)[:, :case["owned"]]
        logits.scatter_add_(1, off + own, torch.full_like(own, 4, dtype=logits.dtype))
    return logits, bias.to(torch.bfloat16)


def _fp8(shape, g, device):
    return torch.randn(shape, generator=g, device=device).to(FP8)


def _inputs(case, seed, device):
    H, I, el, _, _, _, _ = LAYERS[case["layer"]]
    g = torch.Generator(device=device).manual_seed(seed)
    logits, bias = _logits(case, g, device)

    def scales(*shape, lo, hi):
        return torch.empty(shape, device=device).uniform_(lo, hi, generator=g)

    if case["entry"] == "run_bf16":
        acts = (torch.randn(case["T"], H, generator=g, device=device).to(torch.bfloat16),)
    else:
        acts = (_fp8((case["T"], H), g, device), scales(H // BLOCK, case["T"], lo=0.01, hi=0.1))
    w1 = torch.empty(el, 2 * I, H, dtype=FP8, device=device)
    w2 = torch.empty(el, H, I, dtype=FP8, device=device)
    for e in range(el):
        w1[e] = _fp8((2 * I, H), g, device)
        w2[e] = _fp8((H, I), g, device)
    w1s = scales(el, 2 * I // BLOCK, H // BLOCK, lo=0.001, hi=0.01)
    w2s = scales(el, H // BLOCK, I // BLOCK, lo=0.001, hi=0.01)
    return (logits, bias, *acts, w1, w1s, w2, w2s)


def prepare(case, seed):
    H = LAYERS[case["layer"]][0]
    args = _inputs(case, seed, "cuda")
    out = torch.empty(case["T"], H, dtype=torch.bfloat16, device="cuda")
    return {"entry": case["entry"], "out": out, "args": (*args, case["offset"], SCALING, out)}


def run(state):
    if state["entry"] == "run_bf16":
        q, s = kernel.run_bf16(*state["args"])
        return [state["out"], q, s]
    kernel.run(*state["args"])
    return [state["out"]]


def _route(case, logits, bias, dtype):
    """Expert ids [T, k] chosen in fp32, as the layer is defined, and their weights in `dtype`."""
    _, _, _, eg, n_group, kept, k = LAYERS[case["layer"]]
    T = logits.shape[0]
    choice = torch.sigmoid(logits) + bias.float()
    grouped = choice.view(T, n_group, eg // n_group)
    score = grouped.topk(2, dim=-1).values.sum(dim=-1)
    keep = torch.zeros_like(score, dtype=torch.bool).scatter_(1, score.topk(kept, dim=1).indices, True)
    masked = grouped.masked_fill(~keep[:, :, None], float("-inf")).view(T, eg)
    ids = masked.topk(k, dim=1).indices
    s = torch.sigmoid(logits.to(dtype)).gather(1, ids)
    return ids, s * SCALING / (s.sum(dim=1, keepdim=True) + 1e-20)


def work(case):
    """Inputs read once (the weights of the experts that have tokens), output written once,
    and the multiply-adds of the rows of those experts, for one typical batch."""
    H, I, el, eg, _, _, _ = LAYERS[case["layer"]]
    logits, bias = _logits(case, torch.Generator().manual_seed(1), "cpu")
    ids, _ = _route(case, logits, bias, torch.float32)
    local = ids[(ids >= case["offset"]) & (ids < case["offset"] + el)]
    experts, rows = local.unique().numel(), local.numel()
    act = 2 * H + H + 4 * H // BLOCK if case["entry"] == "run_bf16" else H + 4 * H // BLOCK
    per_token = 4 * eg + act + 2 * H
    per_expert = 3 * I * H + 4 * 3 * (I // BLOCK) * (H // BLOCK)
    return {"bytes": case["T"] * per_token + 2 * eg + experts * per_expert,
            "flops": 2 * 3 * I * H * rows}


def tolerance(case):
    # bf16 output of a product whose inner activation is bf16 as well: 1.7e-3
    # to 2.9e-3 from 64 bits over all cases
    return {"rel": 0.01, "max": 0.1}


def exact(case, seed):
    H, I, el, _, _, _, _ = LAYERS[case["layer"]]
    args = _inputs(case, seed, "cuda")
    logits, bias, (w1, w1s, w2, w2s) = args[0], args[1], args[-4:]
    T, f64 = case["T"], torch.float64
    quantised = []
    if case["entry"] == "run_bf16":
        # quotients in 64 bits, rounded once to the fp32 ones of the definition
        x = args[2].to(f64).view(T, H // BLOCK, BLOCK)
        s = (x.abs().amax(dim=-1).clamp_min(1e-10) / 448.0).float()
        q = (x / s[:, :, None].to(f64)).float().clamp(-448.0, 448.0).to(FP8).view(T, H)
        s = s.t().contiguous()
        quantised = [q.to(f64), s.to(f64)]
    else:
        q, s = args[2], args[3]

    def blocks(w, scale):
        return (w.to(f64).view(w.shape[0] // BLOCK, BLOCK, w.shape[1] // BLOCK, BLOCK)
                * scale.to(f64)[:, None, :, None]).view(w.shape)

    ids, weights = _route(case, logits, bias, f64)
    out = torch.zeros(T, H, dtype=f64, device="cuda")
    for e in range(el):
        tok, place = (ids == case["offset"] + e).nonzero(as_tuple=True)
        if not tok.numel():
            continue
        x = (q[tok].to(f64).view(-1, H // BLOCK, BLOCK) * s.t()[tok].to(f64)[:, :, None]).view(-1, H)
        y = x @ blocks(w1[e], w1s[e]).t()
        y = y[:, I:] * torch.sigmoid(y[:, I:]) * y[:, :I]
        y = y @ blocks(w2[e], w2s[e]).t()
        out.index_add_(0, tok, y * weights[tok, place][:, None])
    return [out, *quantised]
