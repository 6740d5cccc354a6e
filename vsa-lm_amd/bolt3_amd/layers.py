"""Small modules around the Bolt-3 path, with the reference's parameter names.

``RMSNorm`` and ``RoPE`` carry the state-dict names the reference uses
(``weight``; non-persistent buffer ``inv_freq``) so checkpoints load
unchanged.  ``SoftmaxAttn``, ``MLP`` and ``HybridLM`` are the caller side of the
path (the softmax-anchor layers and the model container that
``Bolt3Decoder`` walks); they run as PyTorch ops on the device, except
``RMSNorm``, whose device forward is the library's ``bolt3_rms_norm`` (one pass
per row instead of the torch ops' six; CPU tensors keep the torch ops), and the
decoder's MLPs (``mlp_swiglu``; ``mlp_rows`` for a one-token step on request).
  RMSNorm      -- vsa_lm/surgery.py:43-53
  rope_inv_freq-- vsa_lm/surgery.py:56-72
  RoPE         -- vsa_lm/surgery.py:80-93
  MLP          -- vsa_lm/surgery.py:202-211
  SoftmaxAttn  -- vsa_lm/config/standard.py:55-122 (plain, un-gated variant)
  HybridLM     -- vsa_lm/config/standard.py:341-404 (UniversalBlock / UniversalVSALM names)
"""
from __future__ import annotations

import math

import torch
import torch.nn as nn
import torch.nn.functional as F


class RMSNorm(nn.Module):
    def __init__(self, dim: int, eps: float = 1e-5):
        super().__init__()
        self.weight = nn.Parameter(torch.ones(dim))
        self.eps = eps

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        if x.is_cuda and _hip_norm_ok(x, self.weight):
            return _rms_norm_hip(x, self.weight, self.eps)
        xf = x.float()
        xf = xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + self.eps)
        return (xf * self.weight.float()).to(x.dtype)


def _hip_norm_ok(x: torch.Tensor, w: torch.Tensor) -> bool:
    """bolt3_rms_norm takes the device forward when nothing asks for a gradient (it has no
    backward) and the shape and dtypes are its own; CPU tensors keep the torch ops."""
    needs_grad = torch.is_grad_enabled() and (x.requires_grad or w.requires_grad)
    return (not needs_grad and x.dtype in (torch.float32, torch.bfloat16) and
            w.dtype in (torch.float32, torch.bfloat16) and x.shape[-1] % 8 == 0 and x.numel() > 0)


def _rms_norm_hip(x: torch.Tensor, w: torch.Tensor, eps: float) -> torch.Tensor:
    from . import _abi as A
    D = x.shape[-1]
    x2 = x.reshape(-1, D)
    if x2.stride(-1) != 1 or (x2.stride(0) * x2.element_size()) % 16 or x2.data_ptr() % 16:
        x2 = x2.contiguous()
    y = torch.empty(x2.shape, dtype=x.dtype, device=x.device)
    wc = w.detach().contiguous()
    a = A.RmsNormArgs()
    a.dtype, a.rows, a.dim = A.dtype_code(x.dtype), x2.shape[0], D
    a.x, a.x_row_stride, a.w, a.w_dtype = x2.data_ptr(), x2.stride(0), wc.data_ptr(), A.dtype_code(wc.dtype)
    a.y, a.y_row_stride, a.eps = y.data_ptr(), y.stride(0), float(eps)
    A.call("bolt3_rms_norm", a, x.device)
    return y.view(x.shape)


def rope_inv_freq(head_dim: int, theta: float, rope_scaling: dict | None = None) -> torch.Tensor:
    """theta^(-2i/HD), with the llama3 frequency-band rescaling when requested."""
    inv = 1.0 / (theta ** (torch.arange(0, head_dim, 2, dtype=torch.int64).float() / head_dim))
    if rope_scaling and rope_scaling.get("rope_type") == "llama3":
        ctx = float(rope_scaling["original_max_position_embeddings"])
        factor = float(rope_scaling["factor"])
        lo, hi = float(rope_scaling["low_freq_factor"]), float(rope_scaling["high_freq_factor"])
        wl = 2.0 * math.pi / inv
        scaled = torch.where(wl > ctx / lo, inv / factor, inv)
        blend = (ctx / wl - lo) / (hi - lo)
        mixed = (1.0 - blend) * scaled / factor + blend * scaled
        mid = ~(wl < ctx / hi) & ~(wl > ctx / lo)
        inv = torch.where(mid, mixed, scaled)
    return inv


class RoPE(nn.Module):
    def __init__(self, head_dim: int, theta: float, rope_scaling: dict | None = None):
        super().__init__()
        self.register_buffer("inv_freq", rope_inv_freq(head_dim, theta, rope_scaling), persistent=False)

    def forward(self, x: torch.Tensor, pos_start: int = 0) -> torch.Tensor:
        t = torch.arange(pos_start, pos_start + x.shape[2], device=x.device, dtype=torch.float32)
        ang = t[:, None] * self.inv_freq.to(x.device)
        ang = torch.cat((ang, ang), dim=-1)
        half = x.shape[-1] // 2
        rot = torch.cat((-x[..., half:], x[..., :half]), dim=-1)
        return x * ang.cos().to(x.dtype)[None, None] + rot * ang.sin().to(x.dtype)[None, None]


class MLP(nn.Module):
    def __init__(self, cfg: dict):
        super().__init__()
        D, I = cfg["dim"], cfg["intermediate"]
        self.gate_proj = nn.Linear(D, I, bias=False)
        self.up_proj = nn.Linear(D, I, bias=False)
        self.down_proj = nn.Linear(I, D, bias=False)

    def forward(self, x):
        return self.down_proj(F.silu(self.gate_proj(x)) * self.up_proj(x))


def _untouched(m: nn.Module) -> bool:
    """Calling m is nothing but its class's forward: no hook of its own or of all modules, no forward set
    on the instance, not compiled.  What replaces a module's call asks for this, so that hooks and
    overrides see the calls they saw."""
    return not (m._forward_hooks or m._forward_pre_hooks or "forward" in m.__dict__ or
                m._compiled_call_impl is not None or torch.nn.modules.module._has_any_global_hook())


MLP_ROWS = 16   # rows bolt3_rows_linear takes; the library's products are the faster ones above


def _plain_linear(m: nn.Module, x: torch.Tensor) -> bool:
    """A linear layer that is nothing but its bf16 weight on x's device, rows as the kernel reads them."""
    return (type(m) is nn.Linear and m.bias is None and _untouched(m) and
            type(m.weight) in (nn.Parameter, torch.Tensor) and m.weight.dtype == torch.bfloat16 and
            m.weight.device == x.device and m.weight.is_contiguous() and m.weight.data_ptr() % 16 == 0 and
            m.in_features % 32 == 0 and m.out_features % 16 == 0)


def mlp_rows(mlp: nn.Module, h: torch.Tensor, res: torch.Tensor) -> torch.Tensor | None:
    """res + mlp(h) for the few rows of a one-token decode step, in two launches that stream the weights
    once (gate, up and SwiGLU; down and the residual), with the roundings of the module's own ops.
    None where it does not apply: gradients, autocast, hooks or overrides, other modules, dtypes or
    layouts, more than MLP_ROWS rows."""
    D = h.shape[-1]
    M = h.numel() // D if D else 0
    if (type(mlp) is not MLP or not 0 < M <= MLP_ROWS or not h.is_cuda or h.dtype != torch.bfloat16 or
            res.dtype != h.dtype or res.shape != h.shape or res.device != h.device or
            type(h) is not torch.Tensor or type(res) is not torch.Tensor or torch.is_grad_enabled() or
            torch.is_autocast_enabled(h.device.type) or not _untouched(mlp)):
        return None
    gate, up, down = mlp.gate_proj, mlp.up_proj, mlp.down_proj
    if not (_plain_linear(gate, h) and _plain_linear(up, h) and _plain_linear(down, h)):
        return None
    inner = gate.out_features
    if gate.in_features != D or up.in_features != D or up.out_features != inner or \
            down.in_features != inner or down.out_features != D:
        return None
    from . import _abi as A
    x, r = h.reshape(M, D), res.reshape(M, D)
    x = x if x.stride(1) == 1 and x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0 else x.contiguous()
    r = r if r.stride(1) == 1 and r.stride(0) % 4 == 0 and r.data_ptr() % 8 == 0 else r.contiguous()
    act = torch.empty(M, inner, dtype=h.dtype, device=h.device)
    out = torch.empty(M, D, dtype=h.dtype, device=h.device)
    a = A.RowsLinearArgs()
    a.mode, a.M, a.N, a.K = A.ROWS_SWIGLU, M, inner, D
    a.x, a.x_row_stride, a.w, a.w2 = x.data_ptr(), x.stride(0), gate.weight.data_ptr(), up.weight.data_ptr()
    a.out, a.out_row_stride = act.data_ptr(), inner
    A.call("bolt3_rows_linear", a, h.device)
    a.mode, a.N, a.K = A.ROWS_RESIDUAL, D, inner
    a.x, a.x_row_stride, a.w, a.w2 = act.data_ptr(), inner, down.weight.data_ptr(), None
    a.res, a.res_row_stride, a.out, a.out_row_stride = r.data_ptr(), r.stride(0), out.data_ptr(), D
    A.call("bolt3_rows_linear", a, h.device)
    return out.view(h.shape)


def mlp_swiglu(mlp: nn.Module, h: torch.Tensor) -> torch.Tensor | None:
    """mlp(h) with SwiGLU as one pass over the two projections' outputs instead of the module's two (the
    same roundings); None where it does not apply (gradients, autocast, hooks on the MLP or on all modules,
    an overridden forward, another MLP, not bf16)."""
    if (type(mlp) is not MLP or not h.is_cuda or h.dtype != torch.bfloat16 or type(h) is not torch.Tensor or
            torch.is_grad_enabled() or torch.is_autocast_enabled(h.device.type) or not _untouched(mlp)):
        return None
    g, u = mlp.gate_proj(h), mlp.up_proj(h)
    if (g.dtype != torch.bfloat16 or u.dtype != g.dtype or u.shape != g.shape or u.device != g.device or
            not g.is_contiguous() or not u.is_contiguous() or g.numel() % 8 or g.data_ptr() % 16 or u.data_ptr() % 16 or
            type(g) is not torch.Tensor or type(u) is not torch.Tensor):
        return mlp.down_proj(F.silu(g) * u)
    from . import _abi as A
    act = torch.empty_like(g)
    a = A.SwigluArgs()
    a.n, a.gate, a.up, a.out = g.numel(), g.data_ptr(), u.data_ptr(), act.data_ptr()
    A.call("bolt3_swiglu", a, h.device)
    return mlp.down_proj(act)


class SoftmaxAttn(nn.Module):
    """Causal softmax-anchor layer of a hybrid stack."""

    def __init__(self, cfg: dict):
        super().__init__()
        D, H, HKV = cfg["dim"], cfg["num_heads"], cfg["num_kv_heads"]
        HD = cfg.get("head_dim") or (D // H)
        bias = bool(cfg.get("qkv_bias", False))
        self.H, self.HKV, self.HD, self.G = H, HKV, HD, H // HKV
        self.q_proj = nn.Linear(D, H * HD, bias=bias)
        self.k_proj = nn.Linear(D, HKV * HD, bias=bias)
        self.v_proj = nn.Linear(D, HKV * HD, bias=bias)
        self.o_proj = nn.Linear(H * HD, D, bias=False)
        if cfg.get("qk_norm", False):
            self.q_norm, self.k_norm = RMSNorm(HD, cfg["eps"]), RMSNorm(HD, cfg["eps"])
        else:
            self.q_norm = self.k_norm = None
        self.rope = RoPE(HD, cfg["rope_theta"], cfg.get("rope_scaling"))

    def head_qkv(self, x):
        b, t, _ = x.shape
        q = self.q_proj(x).view(b, t, self.H, self.HD)
        k = self.k_proj(x).view(b, t, self.HKV, self.HD)
        v = self.v_proj(x).view(b, t, self.HKV, self.HD)
        if self.q_norm is not None:
            q, k = self.q_norm(q), self.k_norm(k)
        return q.transpose(1, 2), k.transpose(1, 2), v.transpose(1, 2)

    def forward(self, x):
        b, t, _ = x.shape
        q, k, v = self.head_qkv(x)
        q, k = self.rope(q), self.rope(k)
        y = F.scaled_dot_product_attention(q, k, v, is_causal=True, enable_gqa=self.G > 1)
        return self.o_proj(y.transpose(1, 2).reshape(b, t, self.H * self.HD))


class Block(nn.Module):
    def __init__(self, cfg: dict, kind: str):
        super().__init__()
        from .bolt3 import Bolt3Attn
        self.norm1 = RMSNorm(cfg["dim"], cfg["eps"])
        if kind == "vsa":
            self.vsa = Bolt3Attn(cfg, max_T=cfg.get("max_T", 2048), S=int(cfg.get("bolt3_S", 128)),
                                 C=int(cfg.get("bolt3_C", 128)))
        else:
            self.attn = SoftmaxAttn(cfg)
        self.norm2 = RMSNorm(cfg["dim"], cfg["eps"])
        self.mlp = MLP(cfg)

    def forward(self, x):
        attn = self.vsa if hasattr(self, "vsa") else self.attn
        x = x + attn(self.norm1(x))
        return x + self.mlp(self.norm2(x))


class HybridLM(nn.Module):
    """Hybrid Bolt-3 / softmax language model with UniversalVSALM's attribute names."""

    def __init__(self, vocab_size: int, dim: int, num_layers: int, num_heads: int, num_kv_heads: int,
                 intermediate: int, layer_types: list[str] | None = None, hybrid_every: int = 4,
                 max_T: int = 2048, rope_theta: float = 10000.0, rope_scaling: dict | None = None,
                 eps: float = 1e-5, head_dim: int | None = None, qkv_bias: bool = False,
                 tie_word_embeddings: bool = True, **extra):
        super().__init__()
        head_dim = head_dim or dim // num_heads
        if layer_types is None:
            layer_types = ["softmax" if hybrid_every > 0 and (li + 1) % hybrid_every == 0 else "vsa"
                           for li in range(num_layers)]
        self.config = dict(vocab_size=vocab_size, dim=dim, num_layers=num_layers, num_heads=num_heads,
                           num_kv_heads=num_kv_heads, intermediate=intermediate, max_T=max_T,
                           rope_theta=rope_theta, rope_scaling=rope_scaling, eps=eps, head_dim=head_dim,
                           qkv_bias=qkv_bias, tie_word_embeddings=tie_word_embeddings, layer_types=layer_types,
                           hybrid_every=hybrid_every, **extra)
        self.config.setdefault("is_bolt3", True)
        self.embed_tokens = nn.Embedding(vocab_size, dim)
        self.blocks = nn.ModuleList(Block(self.config, k) for k in layer_types)
        self.norm = RMSNorm(dim, eps)
        self.lm_head = nn.Linear(dim, vocab_size, bias=False)
        if tie_word_embeddings:
            self.lm_head.weight = self.embed_tokens.weight

    def forward(self, input_ids):
        x = self.embed_tokens(input_ids)
        for blk in self.blocks:
            x = blk(x)
        return self.norm(x)
