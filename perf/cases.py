"""The work that a user of this package has it do, as cases to be timed and compared.

Three kinds of call, each through the package's public entry points:

  linear   one BitStackLinear.forward on a [1, tokens, in_features] input, as any model that holds the module
           calls it: single decode tokens, a handful of sequences, prompts.  `level` is the module's fused_level.
  step     one SyntheticLlamaDecoder.step_fused(): a decode step of `batch` sequences at position `pos`, called
           directly or (`graph`) replayed from a HIP graph that was captured once.
  prompt   one SyntheticLlamaDecoder.prefill(): a prompt of `length` tokens for `batch` sequences in one pass.

A decoder here has a few layers and a small vocabulary: its layers are alike, and more of them only repeat the work.
"""
import math

import torch

from bitstack_amd import BitStackLinear
from bitstack_amd.utils.llama_decode import PROJ, LlamaShape, SyntheticLlamaDecoder

DEVICE = "cuda"
VOCAB = 32000
HEAD_DIM = 128


def _linear(out_features, in_features, blocks, tokens, rank=16, bias=False, level=5):
    return {"kind": "linear", "out_features": out_features, "in_features": in_features, "blocks": blocks, "tokens": tokens,
            "rank": rank, "bias": bias, "level": level}


def _decoder(kind, hidden, intermediate, kv_heads, layers, lo, hi, batch, **more):
    return {"kind": kind, "hidden": hidden, "intermediate": intermediate, "kv_heads": kv_heads, "layers": layers,
            "blocks_lo": lo, "blocks_hi": hi, "batch": batch, **more}


def listed():
    cases = [
        # the smallest matrix of an 8B-shape layer (k_proj) for one new token: what counts is the cost of a call
        ("kv_one_token", _linear(1024, 4096, 3, 1)),
        # its largest matrices (gate, up) with a generous memory budget: streaming sign bytes
        ("mlp_one_token", _linear(14336, 4096, 8, 1)),
        # an intermediate size that is a multiple of 128 but not of 512, with a bias: many models have one
        ("uneven_one_token", _linear(4096, 11008, 4, 1, bias=True)),
        # four sequences, or four drafted tokens of one, through the widest matrix (down)
        ("four_tokens", _linear(4096, 14336, 4, 4)),
        # a batch of several dozen sequences; neither rows nor tokens fill whole tiles
        ("ragged_37_tokens", _linear(5000, 4096, 6, 37, bias=True)),
        # a short prompt
        ("short_prompt", _linear(14336, 4096, 5, 100)),
        # a prompt of about 512 tokens
        ("prompt_509", _linear(4096, 14336, 8, 509)),
        # eight prompts of 2048 tokens through the largest matrix of a 70B-shape layer
        ("prompts_16384", _linear(28672, 8192, 3, 16384)),
        # the level that rebuilds the weight and leaves the product to torch
        ("level3_300_tokens", _linear(4096, 4096, 8, 300, level=3)),
        # a decode loop as it is usually written: one step_fused() per token, one sequence, 8B-shape layers
        ("step_one_sequence", _decoder("step", 4096, 14336, 8, 8, 2, 5, 1, pos=384, max_len=1024, graph=False)),
        # a serving loop: eight sequences in lock step behind long prompts, 70B-shape layers, the step replayed from a graph
        ("step_eight_sequences", _decoder("step", 8192, 28672, 8, 2, 1, 5, 8, pos=2100, max_len=2304, graph=True)),
        # two prompts through 8B-shape layers: the linears and everything between them
        ("prompt_pass", _decoder("prompt", 4096, 14336, 8, 2, 2, 6, 2, length=700)),
    ]
    return [dict(case, name=name) for name, case in cases]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    pick = rng.random()
    if pick < 0.64:
        # linears: any number of rows; the columns are nearly always a multiple of 128 in real models
        rank = 16 if rng.random() < 0.8 else rng.randint(4, 15)
        level = 5 if rng.random() < 0.8 else rng.choice((2, 3, 4))
        tokens = _log_int(rng, 1, 4096) if rng.random() < 0.7 else rng.randint(1, 8)
        bias = rng.random() < 0.3
        if rng.random() < 0.12:
            # ... and only a multiple of 8 in some small ones
            return _linear(_log_int(rng, 192, 6144), 8 * _log_int(rng, 24, 768), rng.randint(1, 8), tokens, rank, bias, level)
        in_features = 128 * _log_int(rng, 4, 224)
        out_features = _log_int(rng, 512, min(28672, 28672 * 8192 // in_features))
        return _linear(out_features, in_features, rng.randint(1, 6) if rng.random() < 0.7 else rng.randint(7, 16), tokens, rank,
                       bias, level)
    heads = 4 * rng.randint(2, 16)
    hidden = HEAD_DIM * heads
    intermediate = 512 * max(2, round(hidden * rng.uniform(2.5, 3.6) / 512))
    kv_heads = heads // rng.choice((1, 2, 4))
    lo = rng.randint(1, 3)
    hi = lo + rng.randint(1, 4)
    if pick < 0.84:
        pos = _log_int(rng, 16, 4000)
        return _decoder("step", hidden, intermediate, kv_heads, rng.randint(2, 6), lo, hi,
                        1 if rng.random() < 0.4 else _log_int(rng, 2, 32), pos=pos, max_len=pos + rng.randint(32, 512),
                        graph=rng.random() < 0.5)
    return _decoder("prompt", hidden, intermediate, kv_heads, 2, lo, hi, rng.randint(1, 4), length=_log_int(rng, 16, 1500))


# ------------------------------------------------------------------------------------------------- inputs
def _factors(M, N, blocks, k, gen):
    """u [blocks, M, k] and vt [blocks, k, N] as the decomposition of a Gaussian weight leaves them: the first rank of
    |residual| is its positive mean, the others carry the bulk (both signs, about a fiftieth of it each), and every
    block's residual is about 0.6 of the last one's."""
    decay = 0.6 ** torch.arange(blocks, device=DEVICE, dtype=torch.float32).view(blocks, 1, 1)
    u = torch.randn(blocks, M, k, device=DEVICE, generator=gen)
    vt = torch.randn(blocks, k, N, device=DEVICE, generator=gen)
    bulk = math.sqrt(0.012 * (M ** -0.5 + N ** -0.5))
    mean = math.sqrt(0.016)
    u[:, :, 1:] *= bulk
    vt[:, 1:, :] *= bulk
    u[:, :, 0] = mean * (1.0 + 0.1 * u[:, :, 0])
    vt[:, 0, :] = mean * (1.0 + 0.1 * vt[:, 0, :])
    root = decay.sqrt()
    return (u * root).half(), (vt * root).half()


def _activations(tokens, N, gen):
    """N(0, 1) with a few channels eight times larger, as the inputs of decoder linears have them."""
    x = torch.randn(1, tokens, N, device=DEVICE, generator=gen)
    loud = torch.rand(N, device=DEVICE, generator=gen) < 0.005
    return torch.where(loud, 8.0 * x, x).half()


def _prepare_linear(c, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    M, N, blocks, k = c["out_features"], c["in_features"], c["blocks"], c["rank"]
    with torch.device(DEVICE):
        mod = BitStackLinear(blocks, N, M, k, c["bias"], False, DEVICE, fused_level=c["level"])
    u, vt = _factors(M, N, blocks, k, gen)
    for i in range(blocks):
        getattr(mod, f"qweight_{i}").random_(0, 256, generator=gen)
        getattr(mod, f"u_{i}").copy_(u[i])
        getattr(mod, f"vt_{i}").copy_(vt[i])
    mod.stack_blocks()
    if c["bias"]:
        mod.bias.normal_(0.0, 0.1, generator=gen)
    return {"kind": "linear", "mod": mod, "x": _activations(c["tokens"], N, gen)}


def _prepare_decoder(c, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    shape = LlamaShape(layers=c["layers"], hidden=c["hidden"], intermediate=c["intermediate"], heads=c["hidden"] // HEAD_DIM,
                       kv_heads=c["kv_heads"], vocab=VOCAB)
    config = {f"layer.{L}.{p}": b for (L, p), b in _blocks(c).items()}
    max_len = c["max_len"] if c["kind"] == "step" else c["length"]
    dec = SyntheticLlamaDecoder(shape, config, max_len, DEVICE, seed=seed, batch=c["batch"])
    if c["kind"] == "prompt":
        return {"kind": "prompt", "dec": dec,
                "prompt": torch.randint(0, VOCAB, (c["batch"], c["length"]), device=DEVICE, generator=gen)}
    # a cache that holds `pos` earlier positions
    for cache in (dec.kcache, dec.vcache):
        cache[:, :, :, :c["pos"]].normal_(0.0, 0.07, generator=gen)
    state = {"kind": "step", "dec": dec, "graph": None, "pos": torch.full_like(dec.pos, c["pos"]),
             "token": torch.randint(0, VOCAB, (c["batch"],), device=DEVICE, generator=gen)}
    if c["graph"]:
        _start(state)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            dec.step_fused()                     # once outside of the capture: workspaces, argument blocks
        torch.cuda.current_stream().wait_stream(side)
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            dec.step_fused()
    return state


def prepare(case, seed):
    return (_prepare_linear if case["kind"] == "linear" else _prepare_decoder)(case, seed)


# ------------------------------------------------------------------------------------------------- one pass
def _start(state):
    """The tokens and the position that a step takes up (a step writes both)."""
    state["dec"].pos.copy_(state["pos"])
    state["dec"].token.copy_(state["token"])


def run(state):
    if state["kind"] == "linear":
        return state["mod"](state["x"])
    dec = state["dec"]
    if state["kind"] == "prompt":
        dec.prefill(state["prompt"])
    else:
        _start(state)
        if state["graph"] is None:
            dec.step_fused()
        else:
            state["graph"].replay()
    # (the greedy token is the argmax of the logits: two equally good logits may come out in either order, so it is not compared)
    return {"logits": dec.logits, "kcache": dec.kcache, "vcache": dec.vcache, "pos": dec.pos}


# ------------------------------------------------------------------------------------------------- what a pass needs
def _blocks(c):
    """Blocks per linear of a decoder case: lo..hi in turn, so that neighbours differ."""
    span = c["blocks_hi"] - c["blocks_lo"] + 1
    names = [(L, p) for L in range(c["layers"]) for p in PROJ]
    return {name: c["blocks_lo"] + (3 * j + j // 7) % span for j, name in enumerate(names)}


def _linear_work(M, N, blocks, k, tokens):
    """(bytes of the weight, flops) of one linear: signs, u and vt once; either the signs contracted with vt * x for every
    token, or the weight put together once and multiplied."""
    weight = blocks * (M * N // 8 + 2 * k * (M + N))
    rebuild = 2.0 * k * blocks * M * N
    return weight, min(rebuild * tokens, rebuild + 2.0 * M * N * tokens)


def work(case):
    c = case
    if c["kind"] == "linear":
        M, N, T = c["out_features"], c["in_features"], c["tokens"]
        weight, flops = _linear_work(M, N, c["blocks"], c["rank"], T)
        return {"bytes": weight + 2 * T * (M + N) + (2 * M if c["bias"] else 0), "flops": flops}
    shape = LlamaShape(layers=c["layers"], hidden=c["hidden"], intermediate=c["intermediate"], heads=c["hidden"] // HEAD_DIM,
                       kv_heads=c["kv_heads"], vocab=VOCAB)
    B, H = c["batch"], c["hidden"]
    tokens = B if c["kind"] == "step" else B * c["length"]
    nbytes = 2 * VOCAB * H + 2 * B * VOCAB + 2 * tokens * H      # lm_head, logits, embeddings of the tokens
    flops = 2.0 * B * VOCAB * H
    for (_, p), blocks in _blocks(c).items():
        M, N = shape.proj_shape(p)
        weight, f = _linear_work(M, N, blocks, shape.k, tokens)
        nbytes += weight
        flops += f
    kv_row = 2 * c["layers"] * B * c["kv_heads"] * HEAD_DIM * 2  # k and v of one position, all layers
    if c["kind"] == "step":
        nbytes += kv_row * (c["pos"] + 1)
        flops += 4.0 * B * H * (c["pos"] + 1) * c["layers"]
    else:
        nbytes += kv_row * c["length"]
        flops += 2.0 * B * H * c["length"] * (c["length"] + 1) * c["layers"]
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # one linear: fp16 in and out, fp32 sums; another order of the roundings (x * vt, the rebuilt weight, y) moves it by a few 1e-4.
    # Levels 2 to 4 round the same weight to fp16 once and multiply it in fp32.
    if case["kind"] == "linear":
        return {"rel": 1e-3}
    # a few decoder layers in fp16, each with a dozen roundings
    return {"rel": 5e-3}
