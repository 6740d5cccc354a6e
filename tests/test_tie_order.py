"""torch.topk's CPU order among equal values, restated (oracle/torch_topk_order.py), against
torch.topk itself.

The reference's slot decisions are torch.topk calls (vsa_lm/config/bolt3.py:137-138, :183).
The kernel reproduces their order among exactly equal values with the wave-parallel form
(``topk_order_wave``), so both restatements are pinned here on arrays built to tie: small
integer ranges, long runs of -1e9 (merged tokens), a sorted run, NaN and -0/+0 mixed in, every
length the kernel sees (124..256) and the partial_sort path (64*k <= n).
"""
import random

import numpy as np
import pytest
import torch

from oracle.torch_topk_order import _Seq, tie_in_prefix, topk_order_levels, topk_order_seq, topk_order_wave


def _case(t: int, rng: random.Random):
    n = rng.choice([3, 4, 5, 17, 33, 100, 124, 127, 128, 129, 130, 200, 255, 256])
    k = max(1, min(n, rng.choice([1, 2, 3, 4, n // 2, n - 1, n, min(n, 128), rng.randint(1, n)])))
    r = np.random.default_rng(t)
    kind = t % 7
    if kind == 0:
        v = r.integers(0, 3, n).astype(np.float32)
    elif kind == 1:
        v = r.integers(0, 20, n).astype(np.float32)
    elif kind == 2:
        v = r.standard_normal(n).astype(np.float32)
        v[r.random(n) < 0.5] = -1e9
    elif kind == 3:
        v = np.sort(r.integers(0, 10, n)).astype(np.float32)
        v = v[::-1].copy() if t % 2 else v
    elif kind == 4:
        v = np.full(n, 0.5, np.float32)
        v[r.random(n) < 0.2] = np.nan
    elif kind == 5:
        v = r.integers(0, 4, n).astype(np.float32)
        v[r.random(n) < 0.1] = np.nan
        v[r.random(n) < 0.2] = -0.0
    else:
        v = r.standard_normal(n).astype(np.float32)
    return v, k, rng.random() < 0.5


@pytest.mark.parametrize("form", ["seq", "wave"])
def test_restatement_matches_torch_topk(form):
    rng = random.Random(7)
    bad = []
    for t in range(2500):
        v, k, largest = _case(t, rng)
        want = torch.topk(torch.from_numpy(v), k, largest=largest)[1].tolist()
        if form == "seq":
            got = topk_order_seq(v.tolist(), k, largest)
        else:
            got, limit = topk_order_wave(v.tolist(), k, largest)
            assert not limit, (t, len(v), k)
        if got != want:
            bad.append((t, len(v), k, largest))
    assert not bad, bad[:5]


def test_level_form_matches_torch_topk():
    """The form the kernel runs: every range of a level of the sort's recursion at once."""
    rng = random.Random(11)
    bad = []
    for t in range(1500):
        v, k, largest = _case(t, rng)
        got, limit = topk_order_levels(v.tolist(), k, largest)
        assert not limit, (t, len(v), k)
        if got != torch.topk(torch.from_numpy(v), k, largest=largest)[1].tolist():
            bad.append((t, len(v), k, largest))
    assert not bad, bad[:5]


class _Undecided:
    """A value whose order is fixed only when a comparison needs it, so that pivots come out extreme."""

    def __init__(self, game):
        self.v, self.game = None, game

    def __lt__(self, o):
        g = self.game
        if self.v is None and o.v is None:
            first = self if self is g["kept"] else o
            first.v, g["next"] = g["next"], g["next"] + 1
        if self.v is None or o.v is None:
            g["kept"] = self if self.v is None else o
            return self.v is not None
        return self.v < o.v


def depth_limit_values(n: int, k: int) -> list[int]:
    """A permutation of 0 .. n - 1 whose k-th smallest the median-of-three selection reaches only through
    one-sided partitions, more of them than its depth limit allows."""
    game = dict(kept=None, next=0)
    vals = [_Undecided(game) for _ in range(n)]
    _Seq(vals).nth_element(0, k - 1, n)
    for x in vals:
        if x.v is None:
            x.v, game["next"] = game["next"], game["next"] + 1
    return [x.v for x in vals]


@pytest.mark.parametrize("n,k", [(128, 100), (128, 64), (200, 128), (256, 128)])
@pytest.mark.parametrize("largest", [False, True])
def test_depth_limit_keeps_the_selection(n, k, largest):
    """Where the library falls back to a heap the order among equal values is not restated, but the k
    indices are distinct, hold the k first values and lie in their order."""
    v = [x // 2 * (-2 if largest else 2) for x in depth_limit_values(n, k)]     # pairs of equal values
    for order in (topk_order_wave, topk_order_levels):
        got, limit = order(v, k, largest)
        assert limit and len(set(got)) == k
        assert [v[i] for i in got] == sorted(v, reverse=largest)[:k]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_depth_limit_in_the_slot_order(dtype, gpu):
    """The same in a steady step of the chain: orthogonal slots, whose keep values are their utilities,
    and 100 tokens that all displace a slot."""
    from bolt3_amd import Bolt3Attn
    from bolt3_amd import _abi as A
    from oracle import bolt3_oracle as O
    from test_gpu_parity import _gpu_step
    print(f"[case] depth limit {dtype}", flush=True)
    bh, l, S, HD = 2, 100, 128, 128
    mod = Bolt3Attn(dict(dim=256, num_heads=2, num_kv_heads=2, head_dim=HD, rope_theta=1e4, eps=1e-6,
                         qk_norm=False)).to(gpu)
    g = torch.Generator().manual_seed(1)
    util = torch.tensor([1e-3 * (x // 2 + 1) for x in depth_limit_values(S, l)]).expand(bh, S).contiguous()
    st = O.SlotState(torch.eye(S).expand(bh, S, HD).contiguous().to(dtype), torch.randn(bh, S, HD, generator=g).to(dtype),
                     torch.ones(bh, S), util, torch.zeros(bh, S), torch.ones(bh, S, dtype=torch.bool),
                     torch.zeros(bh, HD, HD), S)
    kr, v = torch.randn(bh, l, HD, generator=g).to(dtype), torch.randn(bh, l, HD, generator=g).to(dtype)
    new, _, log = _gpu_step(mod, st, (kr, kr, v, torch.arange(l).float(), torch.rand(bh, l, generator=g)),
                            torch.full((2,), 0.9), 1, gpu)
    log = log.reshape(bh, A.LOG_ROWS, A.LOG_COLS)
    row = {n: log[:, i] for i, n in enumerate(A.LOG_FIELDS)}
    assert bool((row["info"][:, 0].int() & (A.TIE_BOT | A.TIE_LIMIT) == A.TIE_BOT | A.TIE_LIMIT).all())
    for r in range(bh):
        assert bool((row["win"][r, :l] == 1).all()) and sorted(row["top_tok"][r, :l].int().tolist()) == list(range(l))
        slots, keep = row["bot_slot"][r, :l].long(), row["keep"][r, :S]
        assert len(set(slots.tolist())) == l and torch.equal(keep[slots], keep.sort().values[:l])
        toks = row["top_tok"][r, :l].long()
        assert torch.equal(new["av"].view(bh, S, HD)[r, slots], v[r, toks])      # every slot one whole token


def test_slot_decision_shapes():
    """The kernel's calls: candidates (n = l tokens, k = min(l, 128), largest) and keep values
    (n = 128 slots, k = min(l, 128), smallest), with runs of equal keeps (mutual nearest slots
    of equal utility) and of -1e9 (merged tokens)."""
    for t in range(300):
        r = np.random.default_rng(1000 + t)
        l = int(r.choice([124, 128, 129, 200, 255, 256]))
        kc = min(l, 128)
        cand = r.random(l).astype(np.float32)
        cand[r.random(l) < 0.4] = -1e9
        keep = (0.15 * 0.995 ** int(r.integers(0, 20)) * (1 - np.minimum(r.random(128), 0.98))).astype(np.float32)
        pairs = r.permutation(128)[:40].reshape(20, 2)
        keep[pairs[:, 1]] = keep[pairs[:, 0]]                    # mutual nearest: equal keep
        keep[r.random(128) < 0.1] = np.float32(0.15 * 0.02)     # saturated redundancy clamp
        for vals, largest in ((cand, True), (keep, False)):
            want = torch.topk(torch.from_numpy(vals), kc, largest=largest)[1].tolist()
            assert topk_order_wave(vals.tolist(), kc, largest)[0] == want
            if t < 60:
                assert topk_order_levels(vals.tolist(), kc, largest)[0] == want


def test_tie_in_prefix():
    assert tie_in_prefix([5.0, 4.0, 4.0, 1.0], 2)
    assert not tie_in_prefix([5.0, 4.0, 3.0, 3.0], 2)
    assert tie_in_prefix([5.0, 4.0, 3.0, 3.0], 3)
    assert tie_in_prefix([0.0, -0.0, 1.0], 1)
    assert tie_in_prefix([float("nan"), float("nan"), 1.0], 1)
