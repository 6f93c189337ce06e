"""Minimal decoder-only model runner for batched decode on one GPU, built on
the plugin's own classes.

vLLM is not installed in this image, so this module plays the part of its
model runner for the end-to-end decode measurement the reference quotes in
tokens/s (README.md:17-27, "PolarEngine v4 (Triton)": 34.2 tok/s on a 9B
model). Every linear of every layer is a ``PolarQuantLinearMethod`` layer in
vLLM's merged form (one qkv_proj, one gate_up_proj), called through
``apply`` exactly as vLLM's ``LinearBase.forward`` calls a quantization
method. Around them: token embedding, RMSNorm, rotary embedding, a static
bf16 KV cache, grouped-query attention over it, SiLU(gate) * up, a bf16
residual stream, and a bf16 lm_head (vLLM keeps embeddings and lm_head
unquantized unless a checkpoint quantizes them). Residual add + norm,
attention (with the rotary embedding and the cache write) and SiLU * up run
on the library's decode kernels where their shapes fit, else in torch. There
is no scheduler, sampler beyond argmax, paged cache or tokenizer.

One decode step (``DecodeRunner.step``) takes the batch's current tokens and
position (device tensors, so the step can be captured in a HIP graph and
replayed) and returns the logits; ``greedy_tokens_per_s`` replays it with
the argmax fed back.
"""

from __future__ import annotations

import math
from dataclasses import dataclass, field
from typing import Dict, List, Optional

import torch

from torch.autograd.graph import increment_version

from polarengine_vllm import _lib
from polarengine_vllm.linear_method import PolarQuantLinearMethod


@dataclass
class DecoderConfig:
    hidden: int = 4096
    layers: int = 36
    heads: int = 32
    kv_heads: int = 8
    head_dim: int = 128
    intermediate: int = 12288
    vocab: int = 151936
    rope_theta: float = 1.0e6
    rms_eps: float = 1e-6
    # bits per linear: the mixed assignment of one C4 decoder layer
    bits: Dict[str, int] = field(default_factory=lambda: {
        "qkv_proj": 5, "o_proj": 6, "gate_up_proj": 3, "down_proj": 4})


def qwen3_8b_shapes() -> DecoderConfig:
    """The layer shapes of Qwen3-8B (36 layers, hidden 4096, 32 query / 8 KV
    heads of 128, intermediate 12288, vocabulary 151936, RoPE theta 1e6)."""
    return DecoderConfig()


class QuantLinear(torch.nn.Module):
    """One quantized linear: the buffers create_weights registers, filled
    with codes and norms, then process_weights_after_loading's runtime
    layout; forward is PolarQuantLinearMethod.apply."""

    def __init__(self, in_f: int, out_sizes: List[int], bits: int, dev: torch.device,
                 gen: torch.Generator, codes: Optional[torch.Tensor] = None,
                 norms: Optional[torch.Tensor] = None) -> None:
        super().__init__()
        self.method = PolarQuantLinearMethod(128, bits)
        out_f = sum(out_sizes)
        self.method.create_weights(self, in_f, out_sizes, in_f, out_f, torch.bfloat16)
        self.to(dev)
        if codes is None:  # random codes and norms of a unit-variance weight
            codes = torch.randint(0, 1 << bits, self.codes.shape, generator=gen, device=dev,
                                  dtype=torch.int32).to(torch.int8)
            norms = (torch.rand(self.norms.shape, generator=gen, device=dev) * 0.4 + 0.9) \
                * math.sqrt(128.0 / in_f)
        self.codes.copy_(codes)
        self.norms.copy_(norms.to(torch.float16))
        self.method.process_weights_after_loading(self)

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        return self.method.apply(self, x)


def _rms_norm(x: torch.Tensor, w: torch.Tensor, eps: float) -> torch.Tensor:
    """bf16 in and out (fp32 statistics inside the fused kernel)."""
    return torch.nn.functional.rms_norm(x, (x.shape[-1],), w.to(x.dtype), eps)


def _kernel_operands(*tensors: Optional[torch.Tensor]) -> bool:
    """Whether the decode kernels may read these through raw pointers: contiguous
    bf16 rows, 16-byte aligned, on one GPU."""
    given = [t for t in tensors if t is not None]
    return all(t.is_cuda and t.device == given[0].device and t.dtype is torch.bfloat16
               and t.is_contiguous() and t.data_ptr() % 16 == 0 for t in given)


def _add_norm(x: torch.Tensor, r: Optional[torch.Tensor], w: torch.Tensor, eps: float):
    """x + r (x itself without r) and its RMSNorm: one launch (pe_add_rms_norm)
    for hidden sizes that are a multiple of 8; anything else in torch, which
    refuses shapes, types and devices that do not go together."""
    rows, cols = x.shape
    w = w.to(x.dtype)
    if (cols % 8 or cols > 32768 or w.shape != (cols,) or (r is not None and r.shape != x.shape)
            or not _kernel_operands(x, r, w)):
        x = x if r is None else x + r
        return x, _rms_norm(x, w, eps)
    h = torch.empty_like(x)
    x_out = x if r is None else torch.empty_like(x)
    _lib.check(_lib.lib().pe_add_rms_norm(
        x.data_ptr(), _lib.ptr(r), w.data_ptr(), rows, cols, eps, x_out.data_ptr(),
        h.data_ptr(), _lib.stream_ptr(x.device)), "pe_add_rms_norm")
    return x_out, h


def _silu_mul(gu: torch.Tensor) -> torch.Tensor:
    """silu(gate) * up of [rows, 2 I] (pe_silu_mul for I a multiple of 8, see _add_norm)."""
    rows, inter = gu.shape[0], gu.shape[1] // 2
    if inter % 8 or gu.shape[1] % 2 or not _kernel_operands(gu):
        return torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:]
    out = torch.empty(rows, inter, dtype=gu.dtype, device=gu.device)
    _lib.check(_lib.lib().pe_silu_mul(gu.data_ptr(), rows, inter, out.data_ptr(),
                                      _lib.stream_ptr(gu.device)), "pe_silu_mul")
    return out


def _lm_head(h: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """fp32 logits [rows, vocab] (pe_lm_head for the shapes that it takes, see _add_norm)."""
    rows, vocab = h.shape[0], w.shape[0]
    if (h.shape[1:] != w.shape[1:] or not _kernel_operands(h, w)
            or not _lib.lib().pe_lm_head_fits(rows, vocab, w.shape[1])):
        return torch.nn.functional.linear(h, w).float()
    out = torch.empty(rows, vocab, dtype=torch.float32, device=h.device)
    _lib.check(_lib.lib().pe_lm_head(h.data_ptr(), w.data_ptr(), rows, vocab, w.shape[1],
                                     out.data_ptr(), _lib.stream_ptr(h.device)), "pe_lm_head")
    return out


class DecodeRunner:
    """Random-weight decoder of ``cfg``'s shapes for a fixed batch and
    maximum length; the KV cache holds keys as [layer, batch, kv_head, dim,
    position] and values as [layer, batch, kv_head, position, dim], so both
    attention products take contiguous operands."""

    def __init__(self, cfg: DecoderConfig, batch: int, max_len: int, dev, seed: int = 0,
                 weights: Optional[dict] = None) -> None:
        self.cfg, self.batch, self.max_len = cfg, batch, max_len
        self.dev = torch.device(dev)
        g = torch.Generator(device=self.dev).manual_seed(seed)
        c, bf = cfg, torch.bfloat16
        q_sz, kv_sz = c.heads * c.head_dim, c.kv_heads * c.head_dim
        w = weights or {}
        self.embed = w.get("embed", torch.randn(c.vocab, c.hidden, generator=g, device=self.dev) * 0.02).to(bf)
        self.lm_head = w.get("lm_head", torch.randn(c.vocab, c.hidden, generator=g, device=self.dev)
                             / math.sqrt(c.hidden)).to(bf).contiguous()
        self.final_norm = torch.ones(c.hidden, device=self.dev, dtype=bf)
        self.layers = []
        for i in range(c.layers):
            lw = w.get("layers", [{}] * c.layers)[i]
            mk = lambda name, in_f, outs: QuantLinear(
                in_f, outs, c.bits[name], self.dev, g,
                *((lw[name]["codes"], lw[name]["norms"]) if name in lw else (None, None)))
            self.layers.append({
                "in_norm": torch.ones(c.hidden, device=self.dev, dtype=bf),
                "post_norm": torch.ones(c.hidden, device=self.dev, dtype=bf),
                "qkv_proj": mk("qkv_proj", c.hidden, [q_sz, kv_sz, kv_sz]),
                "o_proj": mk("o_proj", q_sz, [c.hidden]),
                "gate_up_proj": mk("gate_up_proj", c.hidden, [c.intermediate, c.intermediate]),
                "down_proj": mk("down_proj", c.intermediate, [c.hidden]),
            })
        self.k_cache = torch.zeros(c.layers, batch, c.kv_heads, c.head_dim, max_len, dtype=bf,
                                   device=self.dev)
        self.v_cache = torch.zeros(c.layers, batch, c.kv_heads, max_len, c.head_dim, dtype=bf,
                                   device=self.dev)
        inv = 1.0 / (c.rope_theta ** (torch.arange(0, c.head_dim, 2, device=self.dev).float()
                                      / c.head_dim))
        ang = torch.arange(max_len, device=self.dev).float()[:, None] * inv[None, :]
        self.rope = torch.cat([ang.cos(), ang.sin()], 1)  # [max_len, head_dim]
        self.positions = torch.arange(max_len, device=self.dev)

    # The rotary tables [max_len, head_dim / 2] are the halves of one table, which
    # the attention kernel reads a row of: a changed or replaced one takes effect.
    @property
    def cos(self) -> torch.Tensor:
        return self.rope[:, :self.cfg.head_dim // 2]

    @cos.setter
    def cos(self, table: torch.Tensor) -> None:
        self.rope = torch.cat([table.float(), self.sin], 1)

    @property
    def sin(self) -> torch.Tensor:
        return self.rope[:, self.cfg.head_dim // 2:]

    @sin.setter
    def sin(self, table: torch.Tensor) -> None:
        self.rope = torch.cat([self.cos, table.float()], 1)

    def step(self, tokens: torch.Tensor, pos: torch.Tensor) -> torch.Tensor:
        """One decode step for the batch: tokens [B] int64, pos [1] int64 (the
        position every sequence of the batch writes); returns fp32 logits
        [B, vocab]."""
        c = self.cfg
        x = self.embed.index_select(0, tokens)  # residual stream, bf16
        attend = self._attention(pos)
        r = None  # what the last block adds to the residual stream
        for i, ly in enumerate(self.layers):
            x, h = _add_norm(x, r, ly["in_norm"], c.rms_eps)
            o = attend(i, ly["qkv_proj"](h))
            x, h = _add_norm(x, ly["o_proj"](o), ly["post_norm"], c.rms_eps)
            r = ly["down_proj"](_silu_mul(ly["gate_up_proj"](h)))
        x, h = _add_norm(x, r, self.final_norm, c.rms_eps)
        return _lm_head(h, self.lm_head)  # [B, vocab]

    def _attention(self, pos: torch.Tensor):
        """The step's attention, as a function of (layer, qkv rows) -> [B, H * D]:
        rotary embedding, cache write and attention over positions 0 .. pos in
        one launch (pe_decode_attention) for the head sizes and groups that it
        takes; pos must lie in the cache, which the table lookup checks."""
        c, B = self.cfg, self.batch
        H, KVH, D = c.heads, c.kv_heads, c.head_dim
        ws_bytes = _lib.workspace_size("pe_decode_attention_workspace_size", B, KVH,
                                       H // KVH if H % KVH == 0 else 0, D, self.max_len)
        kc, vc = self.k_cache, self.v_cache
        if (not ws_bytes or kc.shape != (c.layers, B, KVH, D, self.max_len)
                or vc.shape != (c.layers, B, KVH, self.max_len, D) or not _kernel_operands(kc, vc)):
            return self._attention_torch(pos)
        if pos.numel() != 1 or pos.dtype != torch.int64:
            raise RuntimeError(f"pos must be one int64, got {pos.dtype} of {tuple(pos.shape)}")
        rope = self.rope.index_select(0, pos)  # [1, D]
        dev = _lib.require_device(kc, rope)
        ws = _lib.workspace(dev, ws_bytes)
        st, scale = _lib.stream_ptr(dev), 1.0 / math.sqrt(D)

        def attend(i: int, qkv: torch.Tensor) -> torch.Tensor:
            qkv = qkv.reshape(B, (H + 2 * KVH) * D).contiguous()
            if not _kernel_operands(kc, qkv):
                return self._attention_torch(pos)(i, qkv)
            out = torch.empty(B, H * D, dtype=torch.bfloat16, device=dev)
            _lib.check(_lib.lib().pe_decode_attention(
                qkv.data_ptr(), rope.data_ptr(), pos.data_ptr(), kc[i].data_ptr(), vc[i].data_ptr(),
                out.data_ptr(), B, KVH, H // KVH, D, self.max_len, scale, _lib.ptr(ws), ws_bytes, st),
                "pe_decode_attention")
            increment_version((kc, vc))  # written through raw pointers
            return out

        return attend

    def _attention_torch(self, pos: torch.Tensor):
        c, B = self.cfg, self.batch
        H, KVH, D = c.heads, c.kv_heads, c.head_dim
        grp, hd = H // KVH, D // 2
        # per step: the position's rotary factors and the attention mask
        cos = self.cos.index_select(0, pos)  # [1, D/2]
        sin = self.sin.index_select(0, pos)
        mask = torch.where(self.positions <= pos, 0.0, float("-inf")).to(torch.bfloat16)
        scale = 1.0 / math.sqrt(D)

        def attend(i: int, qkv: torch.Tensor) -> torch.Tensor:
            # rotate-half RoPE on the q and k heads together
            qk = qkv[:, :(H + KVH) * D].reshape(B, H + KVH, D).float()
            x1, x2 = qk[..., :hd], qk[..., hd:]
            qk = torch.cat([x1 * cos - x2 * sin, x2 * cos + x1 * sin], -1)
            q = (qk[:, :H] * scale).to(torch.bfloat16).reshape(B, KVH, grp, D)
            k = qk[:, H:].to(torch.bfloat16)
            v = qkv[:, (H + KVH) * D:].reshape(B, KVH, D)
            self.k_cache[i].index_copy_(3, pos, k.unsqueeze(-1))
            self.v_cache[i].index_copy_(2, pos, v.unsqueeze(2))
            # scores [B, KVH, grp, max_len] = q . K^T, positions past pos masked
            s = torch.matmul(q, self.k_cache[i]) + mask
            p = torch.softmax(s, -1, dtype=torch.float32).to(torch.bfloat16)
            return torch.matmul(p, self.v_cache[i]).reshape(B, H * D)

        return attend

    def greedy_tokens_per_s(self, start_pos: int, steps: int, warmup: int = 2) -> dict:
        """Greedy decode from ``start_pos``: the step is captured in a HIP graph
        that also writes the argmax back as the next tokens and advances the
        position, then replayed ``steps`` times between two synchronizes
        (HIP events on the replay stream). Returns tokens/s for the batch."""
        dev = self.dev
        tokens = torch.zeros(self.batch, dtype=torch.long, device=dev)
        pos = torch.tensor([start_pos], dtype=torch.long, device=dev)
        if start_pos + warmup + 1 + steps > self.max_len:
            raise ValueError("max_len too small for the requested steps")

        def advance():
            logits = self.step(tokens, pos)
            tokens.copy_(logits.argmax(-1))
            pos.add_(1)

        s = torch.cuda.Stream(device=dev)
        s.wait_stream(torch.cuda.current_stream(dev))
        with torch.cuda.stream(s):
            for _ in range(warmup):  # eager: workspaces and caches at full size
                advance()
            torch.cuda.synchronize(dev)
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=s):
                advance()
            graph.replay()  # one untimed replay
            torch.cuda.synchronize(dev)
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record(s)
            for _ in range(steps):
                graph.replay()
            e1.record(s)
        torch.cuda.synchronize(dev)
        sec = e0.elapsed_time(e1) / 1e3
        return {"tok_per_s": self.batch * steps / sec, "ms_per_step": sec / steps * 1e3,
                "batch": self.batch, "steps": steps, "context_start": start_pos}
