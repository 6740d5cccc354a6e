"""What a program has the Bolt-3 framework do, as cases that can be timed and compared.

Five kinds of work, each through the public entry points (``Bolt3Attn``, ``Bolt3Decoder``,
``DecodeGraph``, ``HybridLM``):

* ``forward``: one layer over a batch of sequences, without gradients (prompt scoring, prefill);
* ``train``:   one layer forward and backward, gradients of x and of every parameter;
* ``prefill``: a prompt through a hybrid stack (three Bolt-3 layers and a softmax layer), logits and
  the decoder state that it leaves;
* ``chunk``:   a follow-up turn of up to C tokens fed to a stack on an existing state;
* ``token``:   one token per sequence on an existing state, the captured step that generation replays.

Two layer shapes: "4b" (hidden 2560, 32 query / 8 kv heads of 128, q/k norm, theta 1e6) and "small"
(hidden 576, 9 / 3 heads of 64, no q/k norm, theta 1e4).  Parameters are a trained layer's kind: gates
with non-zero weights, kappa, gamma and norm weights that differ from head to head.
``exact`` states the same arithmetic in 64-bit torch.
"""
from __future__ import annotations

import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vsa-lm_amd"))

from bolt3_amd import Bolt3Attn, Bolt3Decoder, HybridLM  # noqa: E402
from bolt3_amd.decoder import Bolt3LayerState, DecodeGraph  # noqa: E402

DEV = "cuda"
C = S = 128
SINKS = 4
SHAPES = {
    "4b": dict(dim=2560, num_heads=32, num_kv_heads=8, head_dim=128, rope_theta=1e6, eps=1e-6, qk_norm=True),
    "small": dict(dim=576, num_heads=9, num_kv_heads=3, head_dim=64, rope_theta=1e4, eps=1e-5, qk_norm=False),
}
INTER = {"4b": 9728, "small": 1536}
VOCAB = 16384          # a stack of four layers keeps its head in proportion to a whole model's
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32, "autocast": torch.float32}


def listed():
    return [
        # a batch of long prompts through one layer, the headline workload
        dict(name="forward_4x4096", kind="forward", shape="4b", dtype="bf16", B=4, T=4096, data="random"),
        # one very long document whose keys cluster: consolidation merges, evicts and writes M_res throughout
        dict(name="forward_1x65536", kind="forward", shape="4b", dtype="bf16", B=1, T=65536, data="clustered"),
        # one chat prompt of ordinary length, not a multiple of the chunk
        dict(name="forward_1x777", kind="forward", shape="4b", dtype="bf16", B=1, T=777, data="random"),
        # a small model's layer over a few ragged documents, three query heads per kv head
        dict(name="forward_small_6x1500", kind="forward", shape="small", dtype="bf16", B=6, T=1500, data="clustered"),
        # the same layer in fp32 over one sequence, the reference's own configuration
        dict(name="forward_small_fp32", kind="forward", shape="small", dtype="fp32", B=1, T=1024, data="random"),
        # healing a converted layer: forward and backward at the headline size
        dict(name="train_4x4096", kind="train", shape="4b", dtype="bf16", B=4, T=4096, data="random"),
        # healing a small model under autocast with fp32 parameters, ragged documents
        dict(name="train_small_4x1100", kind="train", shape="small", dtype="autocast", B=4, T=1100, data="clustered"),
        # serving: the prompts of a few requests through a hybrid stack
        dict(name="prefill_2x2000", kind="prefill", shape="4b", dtype="bf16", B=2, T=2000, data="random"),
        # a follow-up turn fed to conversations that are already in memory
        dict(name="chunk_4x128", kind="chunk", shape="4b", dtype="bf16", B=4, T=128, cur=0, data="random"),
        # generation: one token for each of a full batch of requests
        dict(name="token_64", kind="token", shape="4b", dtype="bf16", B=64, T=1, cur=40, data="random"),
        # generation for a handful of requests
        dict(name="token_7", kind="token", shape="4b", dtype="bf16", B=7, T=1, cur=100, data="random"),
        # generation for one user
        dict(name="token_1", kind="token", shape="4b", dtype="bf16", B=1, T=1, cur=127, data="random"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["forward", "forward", "forward", "train", "train", "prefill", "chunk", "token", "token"])
    if kind == "forward":
        shape = rng.choice(["4b", "4b", "small"])
        dtype = "bf16" if shape == "4b" else rng.choice(["bf16", "fp32"])
        B = _log_int(rng, 1, 8)
        T = _log_int(rng, 100, min(65536, 32768 // B) if dtype == "bf16" else 4096 // B)
        return dict(kind=kind, shape=shape, dtype=dtype, B=B, T=T, data=rng.choice(["random", "clustered"]))
    if kind == "train":
        shape, dtype = rng.choice([("4b", "bf16"), ("small", "autocast"), ("small", "bf16")])
        B = _log_int(rng, 1, 4)
        return dict(kind=kind, shape=shape, dtype=dtype, B=B, T=_log_int(rng, 200, 4096),
                    data=rng.choice(["random", "clustered"]))
    if kind == "prefill":
        return dict(kind=kind, shape="4b", dtype="bf16", B=_log_int(rng, 1, 4), T=_log_int(rng, 100, 3000), data="random")
    if kind == "chunk":
        return dict(kind=kind, shape="4b", dtype="bf16", B=_log_int(rng, 1, 16), T=rng.randint(9, 128),
                    cur=rng.randint(0, 127), data="random")
    return dict(kind=kind, shape="4b", dtype="bf16", B=_log_int(rng, 1, 64), T=1, cur=rng.randint(0, 127), data="random")


# ----------------------------------------------------------------------------- inputs

def _gen(seed, what):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 1000 + what)


def _fill_layer(ly, g):
    """A trained layer's kind of parameters."""
    def u(t, lo, hi):
        t.uniform_(lo, hi, generator=g)
    for name in ("q_proj", "k_proj", "v_proj", "o_proj", "beta_proj", "eta_proj"):
        m = getattr(ly, name, None)
        if m is not None:
            m.weight.normal_(0.0, 0.02, generator=g)
    for name in ("q_norm", "k_norm"):
        if getattr(ly, name) is not None:
            u(getattr(ly, name).weight, 0.6, 1.4)
    if isinstance(ly, Bolt3Attn):
        u(ly.beta_proj.bias, -1.5, 1.0)
        u(ly.eta_proj.bias, -0.8, 0.8)
        u(ly.kappa, 0.5, 1.5)
        u(ly.log_gamma, 1.0, 4.0)
        u(ly.res_norm.weight, 0.5, 1.5)


def _inv_freq(shape):
    hd, theta = SHAPES[shape]["head_dim"], SHAPES[shape]["rope_theta"]
    return 1.0 / (theta ** (torch.arange(0, hd, 2, dtype=torch.int64).float() / hd))


def _restore_buffers(mod, shape):
    for m in mod.modules():
        if hasattr(m, "inv_freq"):
            m.inv_freq.copy_(_inv_freq(shape).to(DEV))


def _store(mod, dtype):
    """"bf16": everything but the Bolt-3 parameters (gates, kappa, gamma, res_norm), which checkpoints
    hold in fp32; otherwise fp32 throughout."""
    if dtype == "bf16":
        for name, p in mod.named_parameters():
            if not any(w in name for w in ("beta_proj", "eta_proj", "kappa", "log_gamma", "res_norm")):
                p.data = p.data.to(torch.bfloat16)
    return mod


def _layer(case, seed):
    with torch.device("meta"):
        ly = Bolt3Attn(SHAPES[case["shape"]])
    ly = ly.to_empty(device=DEV)
    with torch.no_grad():
        _restore_buffers(ly, case["shape"])
        _fill_layer(ly, _gen(seed, 1))
    return _store(ly, case["dtype"])


def _types(case):
    return ["vsa", "vsa", "vsa", "softmax"] if case["kind"] == "prefill" else ["vsa"] * 4


def _stack(case, seed):
    with torch.device("meta"):
        m = HybridLM(vocab_size=VOCAB, num_layers=4, intermediate=INTER[case["shape"]], layer_types=_types(case),
                     max_T=65536, **SHAPES[case["shape"]])
    m = m.to_empty(device=DEV)
    m.lm_head.weight = m.embed_tokens.weight
    g = _gen(seed, 2)
    with torch.no_grad():
        _restore_buffers(m, case["shape"])
        m.embed_tokens.weight.normal_(0.0, 1.0, generator=g)
        m.norm.weight.uniform_(0.6, 1.4, generator=g)
        for blk in m.blocks:
            _fill_layer(blk.vsa if hasattr(blk, "vsa") else blk.attn, g)
            for w in (blk.norm1.weight, blk.norm2.weight):
                w.uniform_(0.6, 1.4, generator=g)
            for w in (blk.mlp.gate_proj, blk.mlp.up_proj, blk.mlp.down_proj):
                w.weight.normal_(0.0, 0.02, generator=g)
    return _store(m, case["dtype"]).eval()


def _hidden(case, seed):
    """[B, T, D] around N(0, 1): independent tokens, or 512 centres (Zipf 1.1) with noise 0.15, whose
    keys and values lie close enough together for consolidation to merge them."""
    B, T, D = case["B"], case["T"], SHAPES[case["shape"]]["dim"]
    g = _gen(seed, 3)
    x = torch.randn(B, T, D, generator=g, device=DEV)
    if case["data"] == "clustered":
        centres = torch.randn(512, D, generator=g, device=DEV)
        share = torch.arange(1, 513, device=DEV, dtype=torch.float64) ** -1.1
        z = torch.multinomial((share / share.sum()).float(), B * T, replacement=True, generator=g).view(B, T)
        x = centres[z] + 0.15 * x
    return x.to(DTYPES[case["dtype"]])


def _ids(case, seed):
    return torch.randint(0, VOCAB, (case["B"], case["T"]), generator=_gen(seed, 4), device=DEV)


def _caches(case, seed):
    """The decoder state of conversations some thousands of tokens long, one dict per layer in the form
    that a program saves and loads ({key: tensor}), M_res beside it; and the next position."""
    sh = SHAPES[case["shape"]]
    B, HKV, HD, cur = case["B"], sh["num_kv_heads"], sh["head_dim"], case["cur"]
    g, dt = _gen(seed, 5), DTYPES[case["dtype"]]
    pos0 = 8192 - C                      # the previous chunk's first position
    inv = _inv_freq(case["shape"]).to(DEV)

    def n(*shape):
        return torch.randn(*shape, generator=g, device=DEV)

    def u(lo, hi, *shape):
        return torch.rand(*shape, generator=g, device=DEV) * (hi - lo) + lo

    def seg(p0, length):
        pos = torch.arange(p0, p0 + length, device=DEV, dtype=torch.float32)
        kr = n(B, HKV, length, HD).to(dt)
        return dict(kr=kr, kp=_rope(kr.double(), pos, inv).to(dt), v=n(B, HKV, length, HD).to(dt),
                    pos=pos.view(1, 1, -1), b=torch.sigmoid(n(B, HKV, length)))

    out = []
    for _ in _types(case):
        d = dict(ak=n(B * HKV, S, HD).to(dt), av=n(B * HKV, S, HD).to(dt),
                 mass=u(1.0, 6.0, B * HKV, S).floor(), util=u(0.2, 1.2, B * HKV, S),
                 pm=u(SINKS, pos0, B * HKV, S).floor(), act=torch.ones(B * HKV, S, dtype=torch.bool, device=DEV),
                 sink_v=n(B, HKV, SINKS, HD).to(dt), n_filled=S)
        sink = seg(0, SINKS)
        d["sink_k"] = sink["kp"]
        for pre, s in (("prev_", seg(pos0, C)), ("cur_", seg(pos0 + C, cur) if cur else None)):
            for k in ("kr", "kp", "v", "pos", "b"):
                d[pre + k] = None if s is None else s[k]
        out.append((d, 0.3 * n(B, HKV, HD, HD)))
    return out, pos0 + C + cur


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("forward", "train"):
        ly, x = _layer(case, seed), _hidden(case, seed)
        if kind == "forward":
            return dict(case=case, layer=ly, x=x)
        up = torch.randn(x.shape, generator=_gen(seed, 6), device=DEV).to(torch.bfloat16)
        return dict(case=case, layer=ly, x=x.requires_grad_(True), up=up)
    m = _stack(case, seed)
    dec, ids = Bolt3Decoder(m), _ids(case, seed)
    if kind == "prefill":
        return dict(case=case, model=m, dec=dec, ids=ids)
    saved, pos = _caches(case, seed)
    with torch.no_grad():
        kv = [Bolt3LayerState.from_dict(blk.vsa, d) for blk, (d, _) in zip(m.blocks, saved)]
        states = [ms.clone() for _, ms in saved]
        st = dict(case=case, model=m, dec=dec, ids=ids, kv=kv, states=states, pos=pos)
        if kind == "token":
            st["graph"] = DecodeGraph(dec, states, kv, case["B"], 65536, torch.device(DEV, 0), pos)
    return st


# ----------------------------------------------------------------------------- one pass

def _last_state(states, kv):
    """M_res of every Bolt-3 layer and the last one's newest keys and values."""
    last = max(i for i, m in enumerate(states) if m is not None)
    return dict(m_res=[m for m in states if m is not None], keys=kv[last]["cur_kp"], values=kv[last]["cur_v"])


def run(state):
    kind, case = state["case"]["kind"], state["case"]
    if kind == "forward":
        with torch.no_grad():
            return state["layer"](state["x"])
    if kind == "train":
        ly, x = state["layer"], state["x"]
        ly.zero_grad(set_to_none=True)
        x.grad = None
        if case["dtype"] == "autocast":
            with torch.autocast("cuda", dtype=torch.bfloat16):
                y = ly(x)
        else:
            y = ly(x)
        y.backward(state["up"])
        return dict(y=y.detach(), x=x.grad, grads={n: p.grad for n, p in ly.named_parameters()})
    with torch.no_grad():
        m, dec = state["model"], state["dec"]
        if kind == "prefill":
            h, states, kv = dec.prefill(state["ids"])
            return dict(logits=m.lm_head(h[:, -1]), hidden=h, **_last_state(states, kv))
        if kind == "chunk":
            h, _, _ = dec.step(state["ids"], state["pos"], state["states"], state["kv"])
            state["pos"] += state["ids"].shape[1]
            return dict(logits=m.lm_head(h[:, -1]), hidden=h, m_res=list(state["states"]))
        logits = state["graph"].step(state["ids"])
        return dict(logits=logits, **_last_state(state["states"], state["kv"]))


# ----------------------------------------------------------------------------- what a pass needs

def work(case):
    sh = SHAPES[case["shape"]]
    D, H, HKV, HD = sh["dim"], sh["num_heads"], sh["num_kv_heads"], sh["head_dim"]
    B, T, kind = case["B"], case["T"], case["kind"]
    e = 4 if case["dtype"] == "fp32" else 2
    tok = B * T
    w_layer = D * (2 * H * HD + 2 * HKV * HD + H + HKV)          # projection weights
    w_mlp = 3 * D * INTER[case["shape"]]
    chunks = -(-T // C)
    steps = max(0, chunks - 2)

    def attention(chunk, rows):          # one chunk's scores and values, and the M_res readout
        keys = min(chunk + 1, 2) * C - C // 2 + (S + SINKS if chunk >= 2 else 0)
        return 4 * B * H * rows * HD * keys + (2 * B * H * rows * HD * HD if chunk >= 2 else 0)

    attn = sum(attention(c, min(C, T - c * C)) for c in range(chunks))
    # a consolidation: scores, slot read, cosines, slot Gram, token Gram and the two delta-rule products
    cons = B * HKV * 2 * (5 * C * S * HD + 2 * C * HD * HD)
    layer = 2 * tok * w_layer + attn + steps * cons
    slots = B * HKV * (2 * S * HD * 2 + HD * HD * 4)             # slot keys and values, M_res
    if kind == "forward":
        return dict(flops=layer, bytes=e * (w_layer + 2 * tok * D))
    if kind == "train":                  # backward: two products per projection, the attention's five for its two
        pw = 4 if case["dtype"] == "autocast" else 2
        return dict(flops=3 * 2 * tok * w_layer + 3.5 * attn + 3 * steps * cons,
                    bytes=2 * pw * w_layer + (2 * pw + 4) * tok * D)
    head = VOCAB * D
    if kind == "prefill":
        soft = 2 * tok * w_layer + 2 * B * H * HD * T * T
        return dict(flops=3 * layer + soft + 4 * 2 * tok * w_mlp + 2 * B * head,
                    bytes=2 * (4 * (w_layer + w_mlp) + head + B * (VOCAB + C * D)) + 3 * slots)
    window = B * HKV * (C + case["cur"]) * 2 * HD * 2            # window keys and values
    keys = S + SINKS + C + case["cur"] + T // 2
    per = 2 * tok * (w_layer + w_mlp) + tok * H * (4 * HD * keys + 2 * HD * HD)
    cons = cons + 2 * slots if kind == "chunk" and case["cur"] + T >= C else 0
    return dict(flops=4 * (per + cons) + 2 * B * head,
                bytes=4 * (2 * (w_layer + w_mlp) + slots + window) + 2 * head + 2 * B * VOCAB)


def tolerance(case):
    """fp32: 1.3e-6 from 64 bits was measured.  A bf16 layer of up to four chunks is 0.003 from 64 bits
    and four such layers with their MLPs 0.013; one slot decision taken the other way moves a longer
    sequence's later rows by a few percent, so the layers leave room for a few of them and no more."""
    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    if case["kind"] in ("forward", "train"):
        return {"rel": 0.02, "max": 0.9}
    return {"rel": 0.03, "max": 0.9}


# ----------------------------------------------------------------------------- the same in 64 bits

def _rope(x, pos, inv_freq):
    """Rotate x [..., n, HD] by the fp32 angles pos * inv_freq."""
    ang = (pos.float().unsqueeze(-1) * inv_freq).double()
    c, s = ang.cos(), ang.sin()
    half = x.shape[-1] // 2
    a, b = x[..., :half], x[..., half:]
    return torch.cat((a * c - b * s, b * c + a * s), dim=-1)


def _order(x, k, largest):
    """The first k of the last dim in torch's own order on the host, which also decides among equal values."""
    return [t.to(x.device) for t in torch.topk(x.cpu(), k, dim=-1, largest=largest)]


def _rms(x, w, eps):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w


class _Layer64:
    """One Bolt-3 layer (or a softmax layer) with 64-bit copies of a module's parameters."""

    def __init__(self, ly, shape, grad=False):
        sh = SHAPES[shape]
        self.H, self.HKV, self.HD, self.eps = sh["num_heads"], sh["num_kv_heads"], sh["head_dim"], sh["eps"]
        self.G = self.H // self.HKV
        self.p = {n: q.detach().double().requires_grad_(grad) for n, q in ly.named_parameters()}
        self.inv = _inv_freq(shape).to(DEV)

    def project(self, x, pos):
        p, (b, t, _) = self.p, x.shape

        def heads(name, n, norm):
            y = F.linear(x, p[name + ".weight"]).view(b, t, n, self.HD)
            if norm + ".weight" in p:
                y = _rms(y, p[norm + ".weight"], self.eps)
            return y.transpose(1, 2)

        q, k, v = heads("q_proj", self.H, "q_norm"), heads("k_proj", self.HKV, "k_norm"), heads("v_proj", self.HKV, "")
        r = dict(q=q, k=k, v=v, qp=_rope(q, pos, self.inv), kp=_rope(k, pos, self.inv), pos=pos)
        if "kappa" in p:
            r["beta"] = torch.sigmoid(F.linear(x, p["beta_proj.weight"], p["beta_proj.bias"])).transpose(1, 2)
            r["eta"] = torch.tanh(F.linear(x, p["eta_proj.weight"], p["eta_proj.bias"])).transpose(1, 2).unsqueeze(-1)
        return r

    def gamma(self):
        return (0.999 * torch.sigmoid(self.p["log_gamma"])).clamp(1e-3, 0.999)

    def bias(self, st):
        return self.p["kappa"].view(1, -1, 1) * st["mass"].clamp_min(1.0).log()        # [b, hkv, S]

    def attend(self, r, lo, s0, e0, sinks, st, bias=None):
        """Chunk [s0, e0) over sinks, slots and the keys from lo on; then the M_res readout."""
        b, n = r["q"].shape[0], e0 - s0
        q = r["qp"][:, :, s0:e0].reshape(b, self.HKV, self.G * n, self.HD)
        scale = self.HD ** -0.5
        sc, vals = [], []
        if sinks is not None:
            sc.append(q @ sinks[0].transpose(-1, -2) * scale)
            vals.append(sinks[1])
        if st is not None:
            z = q @ _rope(st["ak"], st["pm"], self.inv).transpose(-1, -2) * scale + self.bias(st).unsqueeze(2)
            sc.append(z.masked_fill(~st["act"].unsqueeze(2), float("-inf")))
            vals.append(st["av"])
        seen = torch.arange(lo, e0, device=DEV)[None, :] <= torch.arange(s0, e0, device=DEV)[:, None]
        sc.append((q @ r["kp"][:, :, lo:e0].transpose(-1, -2) * scale)
                  .masked_fill(~seen.repeat(self.G, 1), float("-inf")))
        vals.append(r["v"][:, :, lo:e0])
        y = (torch.softmax(torch.cat(sc, -1), -1) @ torch.cat(vals, 2)).view(b, self.H, n, self.HD)
        if st is not None:
            u = F.normalize(r["q"][:, :, s0:e0], dim=-1).reshape(b, self.HKV, self.G * n, self.HD) @ st["m"]
            u = u * ((1.0 - self.gamma()).view(1, -1, 1, 1) * scale)
            u = _rms(u.view(b, self.H, n, self.HD), self.p["res_norm.weight"], self.eps)
            y = y + r["eta"][:, :, s0:e0] * u
        return y

    def consolidate(self, st, kr, kp, v, pos, beta):
        """The tokens of a chunk that left the window into the slots and M_res."""
        b, hkv, l, hd = kr.shape
        pos = pos.double().expand(b, hkv, l)
        if st is None:
            def z(*s):
                return torch.zeros(b, hkv, *s, device=DEV, dtype=torch.float64)
            st = dict(ak=z(S, hd), av=z(S, hd), mass=z(S) + 1, util=z(S), pm=z(S), act=z(S).bool(), m=z(hd, hd), n=0)
        st = dict(st, util=st["util"] * 0.995)

        def rows(t, i):
            return torch.gather(t, 2, i.unsqueeze(-1).expand(-1, -1, -1, hd)) if t.dim() == 4 else torch.gather(t, 2, i)

        def put(name, i, new):
            i = i.unsqueeze(-1).expand_as(new) if new.dim() == 4 else i
            st[name] = st[name].scatter(2, i, new)

        def rel_err(bias):
            z = kp @ _rope(st["ak"], st["pm"], self.inv).transpose(-1, -2) * hd ** -0.5 + bias.unsqueeze(2)
            z = z.masked_fill(~st["act"].unsqueeze(2), -1e9)
            return (v - torch.softmax(z, -1) @ st["av"]).norm(dim=-1) / (v.norm(dim=-1) + 1e-6)

        with torch.no_grad():
            cos = F.normalize(kr, dim=-1) @ F.normalize(st["ak"], dim=-1).transpose(-1, -2)
            cos = cos.masked_fill(~st["act"].unsqueeze(2), 0.0)
            best, slot = cos.max(-1)
        if st["n"] < S:
            m = min(S - st["n"], l)
            with torch.no_grad():
                if st["n"]:
                    util = rel_err(st["mass"].clamp_min(1.0).log())
                    score = util * (1.0 - best.clamp(0.0, 1.0))
                else:
                    score, util = F.normalize(v, dim=-1).var(dim=-1), torch.full_like(best, 0.15)
                tok = _order(score, m, True)[1]
            i = torch.arange(st["n"], st["n"] + m, device=DEV).expand(b, hkv, m)
            one = torch.ones(b, hkv, m, device=DEV, dtype=torch.float64)
            for name, new in (("ak", rows(kr, tok)), ("av", rows(v, tok)), ("pm", rows(pos, tok)), ("mass", one),
                              ("util", rows(util, tok)), ("act", one.bool())):
                put(name, i, new)
            st["n"] += m
            return st
        with torch.no_grad():
            rel = rel_err(self.bias(st))
            score = rel * (1.0 - best.clamp(0.0, 1.0))
            merge = (best >= 0.88) & (F.cosine_similarity(v, rows(st["av"], slot), dim=-1) >= 0.80)
            pick = (F.one_hot(slot, S).double() * merge.unsqueeze(-1)).transpose(-1, -2)      # [b, hkv, S, l]
        count = pick.sum(-1)
        hit, total = count > 0, st["mass"] + count
        for name, new in (("ak", kr), ("av", v), ("pm", pos.unsqueeze(-1))):
            old = st[name] if st[name].dim() == 4 else st[name].unsqueeze(-1)
            mean = (st["mass"].unsqueeze(-1) * old + pick @ new) / total.unsqueeze(-1)
            st[name] = torch.where(hit.unsqueeze(-1), mean, old).view(st[name].shape)
        st["mass"] = torch.where(hit, total, st["mass"])
        with torch.no_grad():
            an = F.normalize(st["ak"], dim=-1)
            pair = an @ an.transpose(-1, -2)
            pair.diagonal(dim1=-2, dim2=-1).fill_(-1.0)
            keep = st["util"] * (1.0 - pair.max(-1).values.clamp(0.0, 0.98))
            k = min(l, S)
            top, tok = _order(score.masked_fill(merge, -1e9), k, True)
            low, old = _order(keep, k, False)
            win = (top > low) & (top > -1e8)
            placed = torch.zeros_like(score).scatter(2, tok, win.double()).bool()
        for name, new in (("ak", kr), ("av", v), ("pm", pos), ("mass", torch.ones_like(score)), ("util", rel)):
            w = win.unsqueeze(-1) if st[name].dim() == 4 else win
            put(name, old, torch.where(w, rows(new, tok), rows(st[name], old)))
        kn = F.normalize(kr, dim=-1)
        w = beta * (~merge & ~placed)
        safe = w / ((kn @ kn.transpose(-1, -2)).abs() @ w.unsqueeze(-1)).squeeze(-1).clamp_min(1.0)
        err = (v - kn @ st["m"]) * safe.unsqueeze(-1)
        st["m"] = self.gamma().view(1, -1, 1, 1) * st["m"] + kn.transpose(-1, -2) @ err
        return st

    def out(self, y):
        return F.linear(y.transpose(1, 2).flatten(2), self.p["o_proj.weight"])

    def forward(self, x, last_chunk=False):
        """(layer output, the heads, the slot state).  last_chunk: a full last chunk also takes its
        predecessor out of the window, as the decoder's prefill leaves the state."""
        T = x.shape[1]
        r = self.project(x, torch.arange(T, device=DEV, dtype=torch.float32))
        st = sinks = prev = None
        ys = []
        for s0 in range(0, T, C):
            e0 = min(T, s0 + C)
            ys.append(self.attend(r, s0 if prev is None else prev, s0, e0, sinks, st))
            if e0 - s0 == C and (e0 < T or last_chunk):
                if prev is not None:
                    a = prev
                    if sinks is None:
                        sinks = (r["kp"][:, :, :SINKS], r["v"][:, :, :SINKS])
                        a = SINKS
                    st = self.consolidate(st, *(r[k][:, :, a:s0] for k in ("k", "kp", "v")), r["pos"][a:s0],
                                          r["beta"][:, :, a:s0])
                prev = s0
        return self.out(torch.cat(ys, 2)), r, st

    def step(self, x, pos, d, m_res):
        """t tokens on a saved state: (output, M_res, the current chunk's keys and values)."""
        b, t, _ = x.shape
        hk = (b, self.HKV)
        st = {k: d[k].double().view(*hk, *d[k].shape[1:]) for k in ("ak", "av", "mass", "util", "pm")}
        st.update(act=d["act"].view(*hk, S), m=m_res.double(), n=S)
        r = self.project(x, torch.arange(pos, pos + t, device=DEV, dtype=torch.float32))
        cur = {k: r[k] if d["cur_kp"] is None else torch.cat((d["cur_" + o].double(), r[k]), 2)
               for k, o in (("k", "kr"), ("kp", "kp"), ("v", "v"), ("beta", "b"))}
        whole = dict(q=r["q"], qp=r["qp"], eta=r["eta"])
        n_old = d["prev_kp"].shape[2] + cur["kp"].shape[2] - t
        pad = [torch.zeros(b, self.H, n_old, 1, device=DEV).expand(-1, -1, -1, w) for w in (self.HD, 1)]
        whole = {k: torch.cat((pad[k == "eta"].double(), a), 2) for k, a in whole.items()}
        whole["kp"] = torch.cat((d["prev_kp"].double(), cur["kp"]), 2)
        whole["v"] = torch.cat((d["prev_v"].double(), cur["v"]), 2)
        sinks = (d["sink_k"].double(), d["sink_v"].double())
        y = self.out(self.attend(whole, 0, n_old, n_old + t, sinks, st))
        if cur["kp"].shape[2] >= C:
            st = self.consolidate(st, *(d["prev_" + k].double() for k in ("kr", "kp", "v")), d["prev_pos"].view(-1),
                                  d["prev_b"].double())
            cur = dict(kp=None, v=None)
        return y, st["m"], cur["kp"], cur["v"]

    def softmax(self, x):
        T = x.shape[1]
        r = self.project(x, torch.arange(T, device=DEV, dtype=torch.float32))
        return self.out(self.attend(r, 0, 0, T, None, None))


def _stack64(m, case, x, layer):
    """Hidden states after the final norm; layer(i, module, normed x) is the attention of block i."""
    eps = SHAPES[case["shape"]]["eps"]
    for i, blk in enumerate(m.blocks):
        x = x + layer(i, blk, _rms(x, blk.norm1.weight.double(), eps))
        h = _rms(x, blk.norm2.weight.double(), eps)
        g, u, d = (getattr(blk.mlp, n).weight.double() for n in ("gate_proj", "up_proj", "down_proj"))
        x = x + F.linear(F.silu(F.linear(h, g)) * F.linear(h, u), d)
    return _rms(x, m.norm.weight.double(), eps)


def _follows(case):
    """Whether 64 bits lead to the same slots.  Which token replaces which slot is decided by comparing
    scores that lie close together, and from the first steady consolidation on (the fourth chunk) a
    comparison that 16-bit storage decides the other way leaves another state behind: a fp32 layer
    follows the 64-bit decisions, a bf16 one for the few chunks after."""
    return case["dtype"] == "fp32" or case["T"] <= (8 if case["kind"] == "forward" and case["data"] == "random" else 4) * C


def exact(case, seed):
    kind, shape = case["kind"], case["shape"]
    if not _follows(case):
        return None
    if kind in ("forward", "train"):
        ly = _layer(case, seed)
        x = _hidden(case, seed).double()
        r = _Layer64(ly, shape, grad=kind == "train")
        if kind == "forward":
            with torch.no_grad():
                return r.forward(x)[0]
        x.requires_grad_(True)
        y = r.forward(x)[0]
        up = torch.randn(x.shape, generator=_gen(seed, 6), device=DEV).to(torch.bfloat16)
        y.backward(up.double())
        return dict(y=y.detach(), x=x.grad, grads={n: p.grad for n, p in r.p.items()})
    m, ids = _stack(case, seed), _ids(case, seed)
    with torch.no_grad():
        x = m.embed_tokens.weight.double()[ids]
        left = {}
        if kind == "prefill":
            def layer(i, blk, h):
                if hasattr(blk, "attn"):
                    return _Layer64(blk.attn, shape).softmax(h)
                y, r, st = _Layer64(blk.vsa, shape).forward(h, last_chunk=True)
                n = case["T"] // C * C
                m_res = st["m"] if st is not None else torch.zeros_like(r["k"][:, :, :1].transpose(-1, -2) @ r["k"][:, :, :1])
                left[i] = (m_res, *(r[k][:, :, n:] if case["T"] > n else None for k in ("kp", "v")))
                return y

            h = _stack64(m, case, x, layer)[:, (case["T"] - 1) // C * C:]
        else:
            saved, pos = _caches(case, seed)

            def layer(i, blk, h):
                y, *left[i] = _Layer64(blk.vsa, shape).step(h, pos, *saved[i])
                return y

            h = _stack64(m, case, x, layer)
        m_res, (keys, values) = [left[i][0] for i in sorted(left)], left[max(left)][1:]
        if kind != "prefill" and case["cur"] + case["T"] >= C:
            m_res = [None] * len(m_res)          # decided in 16 bits by this call's consolidation
        out = dict(logits=F.linear(h[:, -1], m.embed_tokens.weight.double()), m_res=m_res)
        if kind != "token":
            out["hidden"] = h
        if kind != "chunk":
            out.update(keys=keys, values=values)
        return out
