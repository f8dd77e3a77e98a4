"""A minimal Llama-architecture decode loop around BitStackLinear, for measuring
end-to-end decode throughput on random-init weights (no checkpoints, no tokenizer).

Every decoder linear (q, k, v, o, gate, up, down) is a BitStackLinear at
fused_level 5 with a per-layer block count taken from a compression_config in the
reference's format, {"layer.{L}.self_attn.q_proj": n_blocks, ...}
(bitstack/utils/decompose.py:14, bitstack/utils/model_utils.py:53-66); embed_tokens
and lm_head stay dense fp16, as in the reference (only the decoder layers are
walked, bitstack/utils/scale_utils.py:212-221).  Everything around the linears
(RMSNorm, RoPE, attention over a static KV cache, SiLU gate) is plain torch in
step() and the library's decode-step kernels in step_fused().  One decode step has
static shapes and reads its position from a device tensor, so it can be captured in
a HIP graph and replayed.
"""
from __future__ import annotations

import ctypes
import math
from dataclasses import dataclass

import torch
import torch.nn.functional as F

from bitstack_amd import _lib
from bitstack_amd._lib import EPI_NONE, EPI_RESIDUAL, EPI_SWIGLU
from bitstack_amd.modules.BitStackLinear import BitStackLinear
from bitstack_amd.utils.inference_utils import MatrixGroup, add_rmsnorm_hip, argmax_hip, attention_prefill_hip, forward_cat_hip, linear_f16_hip, plainly_called, rmsnorm_hip, rope_store_hip, silu_mul_hip

PROJ = ("self_attn.q_proj", "self_attn.k_proj", "self_attn.v_proj", "self_attn.o_proj",
        "mlp.gate_proj", "mlp.up_proj", "mlp.down_proj")


@dataclass
class LlamaShape:
    layers: int = 32
    hidden: int = 4096
    intermediate: int = 14336
    heads: int = 32
    kv_heads: int = 8
    vocab: int = 128256
    rope_theta: float = 500000.0
    rms_eps: float = 1e-5
    k: int = 16
    # Hugging Face `rope_scaling` / `rope_parameters` dictionary (None: plain RoPE); see rope_inv_freq
    rope_scaling: dict | None = None

    @property
    def head_dim(self):
        return self.hidden // self.heads

    def proj_shape(self, name):
        kv = self.kv_heads * self.head_dim
        return {"self_attn.q_proj": (self.hidden, self.hidden), "self_attn.k_proj": (kv, self.hidden),
                "self_attn.v_proj": (kv, self.hidden), "self_attn.o_proj": (self.hidden, self.hidden),
                "mlp.gate_proj": (self.intermediate, self.hidden), "mlp.up_proj": (self.intermediate, self.hidden),
                "mlp.down_proj": (self.hidden, self.intermediate)}[name]

    def block_bytes(self, name):
        m, n = self.proj_shape(name)
        return m * n // 8 + 2 * self.k * (m + n)          # BitStackLinear.memory_per_bit

    def dense_bytes(self):
        return 2 * 2 * self.vocab * self.hidden            # embed_tokens + lm_head, fp16


def rope_inv_freq(head_dim: int, theta: float, scaling: dict | None = None) -> torch.Tensor:
    """Inverse RoPE frequencies [head_dim / 2] (float32, CPU) for a Hugging Face rope configuration.

    None / "default": theta^(-2j/d).  "linear": those divided by `factor`.  "llama3" (the released
    Llama-3.1 / 3.2 checkpoints the reference evaluates): wavelengths above
    original_max_position_embeddings / low_freq_factor are divided by `factor`, those below
    original / high_freq_factor are kept, and the band between is blended linearly in
    original / wavelength.  Any other type raises: the tables would silently be wrong."""
    import math
    inv = 1.0 / (theta ** (torch.arange(0, head_dim, 2, dtype=torch.float32) / head_dim))
    kind = (scaling or {}).get("rope_type", (scaling or {}).get("type", "default")) or "default"
    if kind == "default":
        return inv
    if kind == "linear":
        return inv / float(scaling["factor"])
    if kind != "llama3":
        raise ValueError(f"rope scaling type {kind!r} is not supported (default, linear, llama3 are)")
    factor, lo_f, hi_f = float(scaling["factor"]), float(scaling["low_freq_factor"]), float(scaling["high_freq_factor"])
    old_len = float(scaling["original_max_position_embeddings"])
    wavelen = 2 * math.pi / inv
    smooth = (old_len / wavelen - lo_f) / (hi_f - lo_f)
    blended = (1 - smooth) * inv / factor + smooth * inv
    out = torch.where(wavelen > old_len / lo_f, inv / factor, inv)
    mid = (wavelen <= old_len / lo_f) & (wavelen >= old_len / hi_f)
    return torch.where(mid, blended, out)


LLAMA_8B = LlamaShape()
LLAMA_70B = LlamaShape(layers=80, hidden=8192, intermediate=28672, heads=64, kv_heads=8)


def synthetic_compression_config(shape: LlamaShape, target_bytes: float, lo=2, hi=12, seed=0):
    """Seeded per-layer block counts in [lo, hi], nudged until the total
    (dense part + sum of blocks) is as close to `target_bytes` as one block allows."""
    g = torch.Generator().manual_seed(seed)
    names = [f"layer.{L}.{p}" for L in range(shape.layers) for p in PROJ]
    counts = torch.randint(lo, hi + 1, (len(names),), generator=g).tolist()
    cost = [shape.block_bytes(n.split(".", 2)[2]) for n in names]
    total = shape.dense_bytes() + sum(c * b for c, b in zip(counts, cost))
    order = torch.randperm(len(names), generator=g).tolist()
    changed = True
    while changed:
        changed = False
        for j in order:
            if total > target_bytes and counts[j] > lo:
                counts[j] -= 1
                total -= cost[j]
                changed = True
            elif total + cost[j] <= target_bytes and counts[j] < hi:
                counts[j] += 1
                total += cost[j]
                changed = True
    return dict(zip(names, counts)), total


def _synthetic_bitstack(m, n, blocks, k, dev, gen, name):
    mod = BitStackLinear(0, n, m, k, False, False, dev, fused_level=5)
    mod.name = name
    mod.w_bit = blocks
    # written straight into the stacked layout stack_blocks() would produce
    mod.qweight = torch.randint(0, 256, (blocks, m * n // 8), dtype=torch.uint8, device=dev, generator=gen)
    scale = (0.01 / torch.arange(1, blocks + 1, device=dev, dtype=torch.float32)).view(blocks, 1, 1)
    mod.u = (torch.randn(blocks, m, k, device=dev, generator=gen).abs() * scale).half()
    mod.vt = (torch.randn(blocks, k, n, device=dev, generator=gen).abs() * scale).half()
    return mod


class SyntheticLlamaDecoder:
    """Greedy decode of `batch` sequences in lock step (all at the same position)
    with a static KV cache of `max_len` positions.

    step()        every op around the linears is a torch op, one BitStackLinear
                  call per projection (the structure the reference runs);
    step_fused()  four launch pairs per layer for the seven linears (q/k/v in one,
                  o with the residual add, gate/up with the SiLU product, down with
                  the residual add; the two RMSNorms ride on the q/k/v and gate/up
                  launches) and one attention kernel, all from the library."""

    def __init__(self, shape: LlamaShape, config: dict, max_len: int, device, seed=0, batch=1):
        dev = torch.device(device)
        g = torch.Generator(device=dev).manual_seed(seed)
        h = shape.hidden
        embed = (torch.randn(shape.vocab, h, device=dev, generator=g) * 0.02).half()
        lm_head = (torch.randn(shape.vocab, h, device=dev, generator=g) * 0.02).half()
        norm_w = torch.ones(shape.layers, 2, h, device=dev, dtype=torch.float16)
        final_norm = torch.ones(h, device=dev, dtype=torch.float16)
        lin = []
        for L in range(shape.layers):
            row = {}
            for p in PROJ:
                m, n = shape.proj_shape(p)
                row[p] = _synthetic_bitstack(m, n, config[f"layer.{L}.{p}"], shape.k, dev, g, f"layer.{L}.{p}")
            lin.append(row)
        self._setup(shape, lin, embed, lm_head, norm_w, final_norm, max_len, dev, batch)

    def _setup(self, shape, lin, embed, lm_head, norm_w, final_norm, max_len, dev, batch):
        self.s, self.dev, self.max_len, self.batch = shape, dev, max_len, batch
        self.lin, self.embed, self.lm_head, self.norm_w, self.final_norm = lin, embed, lm_head, norm_w, final_norm
        d = shape.head_dim
        self.kcache = torch.zeros(shape.layers, batch, shape.kv_heads, max_len, d, device=self.dev, dtype=torch.float16)
        self.vcache = torch.zeros_like(self.kcache)
        inv = rope_inv_freq(d, shape.rope_theta, shape.rope_scaling).to(self.dev)
        ang = torch.arange(max_len, device=self.dev, dtype=torch.float32)[:, None] * inv[None, :]
        self.cos, self.sin = ang.cos().half().contiguous(), ang.sin().half().contiguous()   # [max_len, d/2]
        self.pos = torch.zeros(1, device=self.dev, dtype=torch.long)       # next position to write
        self.token = torch.zeros(batch, device=self.dev, dtype=torch.long)
        self.span = torch.arange(max_len, device=self.dev)
        self.logits = None
        self._groups = None
        self._steps = None                                                 # (what it was made for, (launch list, last norm in it, its tensors))

    @classmethod
    def from_checkpoint(cls, path, max_len, device, compression_config=None, niter=None, max_memory_MB=None, batch=1):
        """A decoder over a compressed checkpoint in the reference's layout on local disk
        (bitstack_amd/utils/checkpoint.py): `config.json` supplies the Llama dimensions
        (Hugging Face keys), `compression_config.json` + max_memory_MB pick the blocks per
        layer as the reference's --max_memory_MB does (bitstack/main.py:85-91), or pass a
        compression_config / niter directly.  Token ids in, token ids out: no tokenizer."""
        import json
        import os
        from bitstack_amd.utils import checkpoint as ck
        with open(os.path.join(path, "config.json"), "r") as f:
            hf = json.load(f)
        rope_par = hf.get("rope_parameters") or {}
        rope = hf.get("rope_theta") or rope_par.get("rope_theta", 10000.0)
        scaling = hf.get("rope_scaling") or (rope_par if rope_par.get("rope_type", "default") != "default" else None)
        rope_inv_freq(2, float(rope), scaling)              # raises here, before any weight is read, if unsupported
        shape = LlamaShape(rope_scaling=scaling, layers=hf["num_hidden_layers"], hidden=hf["hidden_size"], intermediate=hf["intermediate_size"],
                           heads=hf["num_attention_heads"], kv_heads=hf.get("num_key_value_heads", hf["num_attention_heads"]),
                           vocab=hf["vocab_size"], rope_theta=float(rope), rms_eps=float(hf.get("rms_norm_eps", 1e-5)))
        if hf.get("head_dim", shape.head_dim) != shape.head_dim:
            raise ValueError("head_dim other than hidden_size / num_attention_heads is not supported")
        if max_memory_MB is not None:
            compression_config = ck.retrieve_compression_config(ck.read_compression_configs(path), max_memory_MB)
        dev = torch.device(device)
        linears, other = ck.load_bitstack_checkpoint(path, compression_config=compression_config, niter=niter,
                                                     device=dev, fused_level=5)
        lin = [{p: linears[f"layer.{L}.{p}"] for p in PROJ} for L in range(shape.layers)]
        shape.k = lin[0][PROJ[0]].k
        f16 = lambda t: t.to(dev, torch.float16).contiguous()
        norm_w = torch.stack([torch.stack([f16(other[f"model.layers.{L}.input_layernorm.weight"]),
                                           f16(other[f"model.layers.{L}.post_attention_layernorm.weight"])])
                              for L in range(shape.layers)])
        embed = f16(other["model.embed_tokens.weight"])
        lm_head = f16(other["lm_head.weight"]) if "lm_head.weight" in other else embed      # tied embeddings
        self = cls.__new__(cls)
        self._setup(shape, lin, embed, lm_head, norm_w, f16(other["model.norm.weight"]), max_len, dev, batch)
        return self

    @classmethod
    def from_dense(cls, shape: LlamaShape, weights: dict, niter: int, max_len: int, device, k=16, batch=1):
        """Compress a dense Llama: every decoder linear becomes a BitStackLinear with `niter`
        residual blocks of rank `k`, decomposed on the device one linear at a time (what
        bitstack/utils/decompose.py:8-31 does to the Hugging Face model with
        BitStackLinear.from_linear; names layer.{L}.{proj} as there).  `weights` uses the
        Hugging Face keys: model.layers.{L}.{proj}.weight, the two layer norms per layer,
        model.embed_tokens.weight, model.norm.weight and lm_head.weight (optional: tied)."""
        import dataclasses
        dev = torch.device(device)
        shape = dataclasses.replace(shape, k=k)
        f16 = lambda t: torch.as_tensor(t).to(dev, torch.float16).contiguous()
        lin = []
        for L in range(shape.layers):
            row = {}
            for p in PROJ:
                w = torch.as_tensor(weights[f"model.layers.{L}.{p}.weight"]).to(dev, torch.float32)
                m, n = shape.proj_shape(p)
                if tuple(w.shape) != (m, n):
                    raise ValueError(f"model.layers.{L}.{p}.weight is {tuple(w.shape)}, expected {(m, n)}")
                dense = torch.nn.Linear(n, m, bias=False, device=dev, dtype=torch.float16)
                with torch.no_grad():
                    dense.weight.copy_(w)
                    mod = BitStackLinear.from_linear(dense, w_bit=niter, k=k, bias=False, fused_level=5, name=f"layer.{L}.{p}")
                mod.stack_blocks()
                row[p] = mod
                del dense, w
            lin.append(row)
        norm_w = torch.stack([torch.stack([f16(weights[f"model.layers.{L}.input_layernorm.weight"]),
                                           f16(weights[f"model.layers.{L}.post_attention_layernorm.weight"])])
                              for L in range(shape.layers)])
        embed = f16(weights["model.embed_tokens.weight"])
        lm_head = f16(weights["lm_head.weight"]) if "lm_head.weight" in weights else embed
        self = cls.__new__(cls)
        self._setup(shape, lin, embed, lm_head, norm_w, f16(weights["model.norm.weight"]), max_len, dev, batch)
        return self

    def save_checkpoint(self, path, compression_configs=None, max_shard_bytes=None):
        """Writes this decoder in the same layout (config.json included)."""
        import json
        import os
        from bitstack_amd.utils import checkpoint as ck
        s = self.s
        linears = {f"layer.{L}.{p}": self.lin[L][p] for L in range(s.layers) for p in PROJ}
        other = {"model.embed_tokens.weight": self.embed, "lm_head.weight": self.lm_head, "model.norm.weight": self.final_norm}
        for L in range(s.layers):
            other[f"model.layers.{L}.input_layernorm.weight"] = self.norm_w[L, 0]
            other[f"model.layers.{L}.post_attention_layernorm.weight"] = self.norm_w[L, 1]
        ck.save_bitstack_checkpoint(path, linears, other, compression_configs, max_shard_bytes)
        with open(os.path.join(path, "config.json"), "w") as f:
            json.dump({"architectures": ["LlamaForCausalLM"], "model_type": "llama", "num_hidden_layers": s.layers,
                       "hidden_size": s.hidden, "intermediate_size": s.intermediate, "num_attention_heads": s.heads,
                       "num_key_value_heads": s.kv_heads, "vocab_size": s.vocab, "rope_theta": s.rope_theta,
                       "rms_norm_eps": s.rms_eps, "tie_word_embeddings": False}, f)

    def weight_bytes(self):
        b = self.embed.numel() * 2 + self.lm_head.numel() * 2
        for row in self.lin:
            for m in row.values():
                b += m.qweight.numel() + 2 * (m.u.numel() + m.vt.numel())
        return b

    def set_bits(self, bits):
        """Blocks in use per linear from now on: one count for all, or {"layer.{L}.{proj}": count}
        (BitStackLinear.set_bit on each; the grouped launches' argument blocks are rebuilt)."""
        for L, row in enumerate(self.lin):
            for p, m in row.items():
                b = bits if isinstance(bits, int) else bits[f"layer.{L}.{p}"]
                if not 1 <= b <= m.u.shape[0]:
                    raise ValueError(f"layer.{L}.{p}: {b} blocks asked, {m.u.shape[0]} loaded")
                m.set_bit(b)
        self._groups = None

    def set_memory_budget(self, path, max_memory_MB=None, compression_config=None):
        """Move the loaded decoder to another size of the same checkpoint while it runs: the
        config that fits max_memory_MB (bitstack/utils/model_utils.py:179-187) or the one given;
        linears that get fewer blocks free the surplus, those that get more read only the
        missing blocks from `path` (checkpoint.apply_compression_config).  The KV cache and
        the position stay as they are.  Returns (bytes_freed, bytes_loaded)."""
        from bitstack_amd.utils import checkpoint as ck
        if compression_config is None:
            compression_config = ck.retrieve_compression_config(ck.read_compression_configs(path), max_memory_MB)
        linears = {f"layer.{L}.{p}": m for L, row in enumerate(self.lin) for p, m in row.items()}
        moved = ck.apply_compression_config(path, linears, compression_config)
        self._groups = None
        return moved

    def reset(self):
        self.pos.zero_()
        self.kcache.zero_()
        self.vcache.zero_()

    def _rms(self, x, w):
        v = x.float()
        return (v * torch.rsqrt(v.pow(2).mean(-1, keepdim=True) + self.s.rms_eps)).half() * w

    def _rope(self, x, cos, sin):          # x [..., d], rotate-half convention
        d2 = x.shape[-1] // 2
        a, b = x[..., :d2], x[..., d2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)

    @torch.no_grad()
    def step(self):
        """Consume self.token at self.pos, write the greedy next token, advance."""
        s, B = self.s, self.batch
        x = self.embed.index_select(0, self.token)                       # [B, h]
        cos = self.cos.index_select(0, self.pos)
        sin = self.sin.index_select(0, self.pos)
        mask = (self.span <= self.pos).view(1, 1, 1, self.max_len)
        rep = s.heads // s.kv_heads
        for L in range(s.layers):
            lin = self.lin[L]
            hn = self._rms(x, self.norm_w[L, 0])
            q = lin["self_attn.q_proj"](hn).view(B, s.heads, s.head_dim)
            k = lin["self_attn.k_proj"](hn).view(B, s.kv_heads, s.head_dim)
            v = lin["self_attn.v_proj"](hn).view(B, s.kv_heads, s.head_dim)
            q, k = self._rope(q, cos, sin), self._rope(k, cos, sin)
            self.kcache[L].index_copy_(2, self.pos, k.unsqueeze(2))
            self.vcache[L].index_copy_(2, self.pos, v.unsqueeze(2))
            qg = q.view(B, s.kv_heads, rep, s.head_dim)
            att = torch.matmul(qg, self.kcache[L].transpose(2, 3)) / math.sqrt(s.head_dim)   # [B, kv, rep, max_len]
            att = att.masked_fill(~mask, float("-inf")).float().softmax(-1).half()
            ctx = torch.matmul(att, self.vcache[L]).reshape(B, s.hidden)
            x = x + lin["self_attn.o_proj"](ctx)
            hn = self._rms(x, self.norm_w[L, 1])
            gate = lin["mlp.gate_proj"](hn)
            up = lin["mlp.up_proj"](hn)
            x = x + lin["mlp.down_proj"](F.silu(gate) * up)
        self.logits = F.linear(self._rms(x, self.final_norm), self.lm_head)
        self.token.copy_(self.logits.argmax(-1))
        self.pos.add_(1)

    def _build_groups(self):
        """Argument blocks of the grouped launches.  The RMSNorm weight vectors in front of
        q/k/v and gate/up are folded into copies of those matrices' vt once
        (vt_i[r, n] * weight[n]); the scalar rsqrt(mean(x^2) + eps) is applied by the
        launch itself, so the fused step has no RMSNorm kernel inside a layer."""
        s, B = self.s, self.batch
        self._groups = []
        self._steps = None

        def folded(mods, weight):
            mats = []
            for m in mods:
                q, u, vt = m._stacked()
                mats.append((q, u, (vt.float() * weight.float().view(1, 1, -1)).half(), m.bias))
            return MatrixGroup(mats)

        for L in range(s.layers):
            lin = self.lin[L]
            self._groups.append({
                "qkv": folded([lin["self_attn.q_proj"], lin["self_attn.k_proj"], lin["self_attn.v_proj"]], self.norm_w[L, 0]),
                "o": MatrixGroup.from_modules([lin["self_attn.o_proj"]]),
                "gate_up": folded([lin["mlp.gate_proj"], lin["mlp.up_proj"]], self.norm_w[L, 1]),
                "down": MatrixGroup.from_modules([lin["mlp.down_proj"]]),
            })
        f16 = dict(dtype=torch.float16, device=self.dev)
        self._hn = torch.empty(B, s.hidden, **f16)
        self._qkv = torch.empty(B, (s.heads + 2 * s.kv_heads) * s.head_dim, **f16)
        self._ctx = torch.empty(B, s.hidden, **f16)
        self._act = torch.empty(B, s.intermediate, **f16)
        self._xa = torch.empty(B, s.hidden, **f16)
        self._xb = torch.empty(B, s.hidden, **f16)

    def _launches(self):
        """(the launches of step_fused() between the embedding and the last norm as one native list (host.cpp), whether that norm
        is in it, every tensor whose address it holds).  Laid out once and again whenever one of the tensors has become another one,
        by address, shape, strides or type.  Whoever runs the list holds the tensors meanwhile: other threads run too."""
        if self._groups is None:
            self._build_groups()
        held = (self.kcache, self.vcache, self.cos, self.sin, self.pos, self.final_norm)
        eps = self.s.rms_eps
        key = (eps, *((t.data_ptr(), t.shape, t.stride(), t.dtype, t.device) for t in held))
        if self._steps is not None and self._steps[0] == key:
            return self._steps[1]
        s, B, dev = self.s, self.batch, self._xa.device
        d, max_len = s.head_dim, self.kcache.shape[-2]
        for name, shape in (("kcache", (B, s.kv_heads, max_len, d)), ("vcache", (B, s.kv_heads, max_len, d)), ("cos", (max_len, d // 2)),
                            ("sin", (max_len, d // 2)), ("pos", ())):
            t = getattr(self, name)
            if name == "pos":
                ok = t.numel() == 1 and t.dtype == torch.int64
            elif len(shape) == 4:                                          # a layer is contiguous, the layers may lie apart
                ok = t.dim() == 5 and t.shape[0] >= s.layers and t.shape[1:] == shape and t.dtype == torch.float16 and t[0].is_contiguous()
            else:
                ok = t.shape == shape and t.dtype == torch.float16 and t.is_contiguous()
            if not ok or t.device != dev:
                raise ValueError(f"the decode step cannot take this {name} ({'one int64' if name == 'pos' else f'fp16 {shape}, contiguous'} on {dev} "
                                 f"is needed): {t.dtype} {tuple(t.shape)}, strides {t.stride()}, on {t.device}")
        xa, xb, qkv, ctx, act = (t.data_ptr() for t in (self._xa, self._xb, self._qkv, self._ctx, self._act))
        kcache, vcache, cos, sin, pos, norm = (t.data_ptr() for t in held)
        klayer, vlayer = 2 * self.kcache.stride(0), 2 * self.vcache.stride(0)     # bytes from a layer's cache to the next

        def group(g, x, y, epilogue, eps=None, residual=0):
            return ("group", ctypes.addressof(g.arr), g.n, g.N, g.K, x, B, eps, epilogue, residual, y)

        items = []
        for L, grp in enumerate(self._groups):
            items.append(group(grp["qkv"], xa, qkv, EPI_NONE, eps=eps))
            items.append(("attention", qkv, kcache + L * klayer, vcache + L * vlayer, cos, sin, pos, ctx, B, s.heads, s.kv_heads, d, max_len))
            items.append(group(grp["o"], ctx, xb, EPI_RESIDUAL, residual=xa))
            items.append(group(grp["gate_up"], xb, act, EPI_SWIGLU, eps=eps))
            items.append(group(grp["down"], act, xa, EPI_RESIDUAL, residual=xb))
        # a norm weight of another type or layout is converted or refused by rmsnorm_hip() in each step
        w = self.final_norm
        inside = tuple(w.shape) == (s.hidden,) and w.dtype == torch.float16 and w.is_contiguous() and w.device == dev
        if inside:
            items.append(("norm", xa, norm, self._hn.data_ptr(), B, s.hidden, eps))
        kept = (held, self._groups, self._xa, self._xb, self._qkv, self._ctx, self._act, self._hn)
        self._steps = (key, (_lib.host().make_steps(items), inside, kept))
        return self._steps[1]

    @torch.no_grad()
    def step_fused(self):
        """Same step on the library's grouped forwards and decode-step kernels: q/k/v with the RMSNorm in front, attention,
        o + residual, gate/up with the RMSNorm in front and the SiLU product, down + residual per layer."""
        launches, normed, kept = self._launches()
        xa, hn = self._xa, self._hn
        torch.index_select(self.embed, 0, self.token, out=xa)
        _lib.host().run_steps(launches, xa.device.index)
        if not normed:
            rmsnorm_hip(xa, self.final_norm, self.s.rms_eps, out=hn)
        self.logits = self._head(hn)
        if not _lib.host().argmax(self.logits, self.token, self.pos):          # both in one launch
            argmax_hip(self.logits, out=self.token)
            self.pos.add_(1)

    def _attend(self, q, k, v, kc, vc, n, stored):
        """prefill()'s attention on torch operations, for heads of other sizes or caches of another layout or type: `stored`
        means that q is rotated and k, v are in the cache.  Otherwise k and v are attended to as they are computed, whatever the
        cache keeps of them."""
        s, B, d = self.s, self.batch, self.s.head_dim
        q = q.view(B, n, s.heads, d).transpose(1, 2)
        if stored:
            k, v = kc[:, :, :n], vc[:, :, :n]
        else:
            cos, sin = self.cos[:n].view(1, 1, n, d // 2), self.sin[:n].view(1, 1, n, d // 2)
            k, v = (t.view(B, n, s.kv_heads, d).transpose(1, 2) for t in (k, v))
            q, k = self._rope(q, cos, sin), self._rope(k, cos, sin)
            kc[:, :, :n].copy_(k)
            vc[:, :, :n].copy_(v)
        ctx = torch.empty(B, n, s.hidden, dtype=torch.float16, device=self.dev)
        for b in range(B):                                                # one sequence at a time bounds the scratch
            o = F.scaled_dot_product_attention(q[b:b + 1], k[b:b + 1], v[b:b + 1], is_causal=True, enable_gqa=True)
            ctx[b].copy_(o[0].transpose(0, 1).reshape(n, s.hidden))
        return ctx.view(B * n, s.hidden)

    def _head(self, hn):
        """The logits.  Up to 8 rows on the library's kernel (32000 x 4096, one row: 56.3 us with F.linear, 48.7 with it; 8: 56.9, 49.3; on 8192
        columns both 94), which reads lm_head at the speed of memory; with 16 rows and more F.linear is level or ahead."""
        w = self.lm_head
        if (hn.shape[0] <= 8 and w.dim() == 2 and w.shape[1] == hn.shape[1] and w.shape[1] % 8 == 0 and w.dtype == hn.dtype == torch.float16
                and w.device == hn.device and w.is_contiguous() and type(w) in (torch.Tensor, torch.nn.Parameter) and w.data_ptr() % 16 == 0):
            return linear_f16_hip(hn, w)
        return F.linear(hn, w)

    @staticmethod
    def _output(module, x):
        """What the module gives for x, as a tensor that may be written over: a copy where somebody else may hold it."""
        plain = plainly_called(module)                                    # (before the call: a hook may take itself off in it)
        y = module(x)
        return y if plain else y.clone(memory_format=torch.contiguous_format)

    def _sum_norm(self, x, add, weight):
        """(x + add, its RMSNorm); the sum takes the place of `add`."""
        if add.dtype == torch.float16 and add.shape == x.shape:
            return add_rmsnorm_hip(x, add, weight, self.s.rms_eps)
        x = x + add
        return x, rmsnorm_hip(x, weight, self.s.rms_eps)

    @staticmethod
    def _silu_mul(gate, up):
        """silu(gate) * up, in gate's place."""
        if gate.dtype == up.dtype == torch.float16 and gate.shape == up.shape:
            return silu_mul_hip(gate, up)
        return F.silu(gate).mul_(up)

    @torch.no_grad()
    def prefill(self, prompt: torch.Tensor, all_logits=False, first_layer=0, hidden=None, keep=None):
        """The whole prompt [batch, len] in one pass: every linear sees batch * len tokens (the
        library's rebuild + dense path, q/k/v and small gate/up as one product), rotation, causal
        attention, norms and the SiLU product run on the library's kernels (attention of heads
        other than 128 wide and caches of another type or layout on torch operations), the KV cache
        is filled for positions 0 .. len - 1, and self.token becomes the greedy token after
        the prompt.  Decode continues from there with step() or step_fused().  With
        all_logits the logits of every position [batch, len, vocab] are returned (perplexity).
        `keep` (a list) receives the input of every decoder layer; `first_layer` with `hidden`
        (such a kept input) resumes from that layer - what a change confined to one layer needs
        to be evaluated (the KV cache of the earlier layers is then left as it is)."""
        s, B = self.s, self.batch
        prompt = prompt.view(1, -1).expand(B, -1) if prompt.dim() == 1 else prompt
        n = prompt.shape[1]
        if n < 1 or n > self.max_len:
            raise ValueError("prompt length must be in 1..max_len")
        d = s.head_dim
        if first_layer == 0:
            x = self.embed.index_select(0, prompt.reshape(-1))            # [B * n, h]
        else:
            if hidden is None or tuple(hidden.shape) != (B * n, s.hidden):
                raise ValueError("resuming needs the kept input of that layer")
            x = hidden
        # caches or tables of another layout or type, if a caller has put such in place, take the torch operations
        plain = all(t.dtype == torch.float16 and t.is_contiguous() for t in (self.kcache, self.vcache, self.cos, self.sin))
        hn = None
        for L in range(first_layer, s.layers):
            if keep is not None:
                keep.append(x)
            lin = self.lin[L]
            if hn is None:
                hn = rmsnorm_hip(x, self.norm_w[L, 0], s.rms_eps)
            wide = s.heads * d, s.kv_heads * d, s.kv_heads * d
            qkv = forward_cat_hip([lin[p] for p in PROJ[:3]], hn) if plain and d == 128 else None
            q, k, v = qkv.split(wide, 1) if qkv is not None else (self._output(lin[p], hn) for p in PROJ[:3])
            stored = plain and all(t.dtype == torch.float16 and t.shape == (B * n, w) for t, w in zip((q, k, v), wide))
            kc, vc = self.kcache[L], self.vcache[L]
            if stored:
                rope_store_hip(q, k, v, self.cos, self.sin, kc, vc, n)
            if stored and d == 128:
                ctx = attention_prefill_hip(q, kc, vc, n)
            else:
                ctx = self._attend(q, k, v, kc, vc, n, stored)
            x, hn = self._sum_norm(x, self._output(lin["self_attn.o_proj"], ctx), self.norm_w[L, 1])
            both = forward_cat_hip([lin["mlp.gate_proj"], lin["mlp.up_proj"]], hn) if s.intermediate % 8 == 0 else None
            act = self._silu_mul(*(both.chunk(2, 1) if both is not None else (self._output(lin[p], hn) for p in PROJ[4:6])))
            down = self._output(lin["mlp.down_proj"], act)
            if L + 1 < s.layers:
                x, hn = self._sum_norm(x, down, self.norm_w[L + 1, 0])
            elif all_logits:
                x, hn = self._sum_norm(x, down, self.final_norm)
            else:                                                         # the last position of each sequence
                x, down = (t.view(B, n, s.hidden)[:, -1].contiguous() for t in (x, down))
                x, hn = self._sum_norm(x, down, self.final_norm)
        if hn is None:                                                    # no layer ran: first_layer is the layer count
            x = x if all_logits else x.view(B, n, s.hidden)[:, -1].contiguous()
            hn = rmsnorm_hip(x, self.final_norm, s.rms_eps)
        if all_logits:
            full = F.linear(hn, self.lm_head).view(B, n, -1)
            self.logits = full[:, -1].contiguous()
        else:
            self.logits = self._head(hn)
        self.token.copy_(self.logits.argmax(-1))
        self.pos.fill_(n)
        return full if all_logits else None

    def prefill_positions(self, prompt: torch.Tensor, fused=False):
        """Feed a prompt token by token (the measurement is about decode).  `prompt`
        is [len] (the same for every sequence) or [batch, len]."""
        self.pos.zero_()
        prompt = prompt.view(1, -1).expand(self.batch, -1) if prompt.dim() == 1 else prompt
        for j in range(prompt.shape[1]):
            self.token.copy_(prompt[:, j])
            (self.step_fused if fused else self.step)()
