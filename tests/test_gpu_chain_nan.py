"""The chain's best-slot search with NaN and infinite keys (bf16, head dims 64 and 128): it takes the
maximum of a lane's cosines first and searches for it afterwards, and a wavefront that holds a
cosine without a finite value takes the general scan instead.  torch.max's rule holds on that path
(the first NaN is the largest), and no other token's match changes, in the same wavefront (the
general scan for every lane) or in another one; equal cosines go to the lowest slot on both."""
import pytest
import torch

from bolt3_amd import _abi as A
from oracle import bolt3_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("HD", [64, 128])
def test_best_slot_with_nan_and_inf_keys(HD, gpu):
    from bolt3_amd import Bolt3Attn
    from test_gpu_parity import _gpu_step
    print(f"[case] chain NaN keys HD={HD}", flush=True)
    cfg = dict(dim=2 * HD, num_heads=2, num_kv_heads=2, head_dim=HD, rope_theta=1e4, eps=1e-6, qk_norm=False)
    mod = Bolt3Attn(cfg).to(gpu)
    g = torch.Generator().manual_seed(HD)
    bh, l, S, bf = 2, 128, 128, torch.bfloat16
    ak = torch.randn(bh, S, HD, generator=g).to(bf)
    ak[:, 77] = ak[:, 20]                                   # two equal slots: ties go to the lower one
    st = O.SlotState(ak, torch.randn(bh, S, HD, generator=g).to(bf), torch.ones(bh, S), torch.rand(bh, S, generator=g),
                     torch.zeros(bh, S), torch.ones(bh, S, dtype=torch.bool), torch.zeros(bh, HD, HD), S)
    kr = torch.randn(bh, l, HD, generator=g).to(bf)
    kr[:, 9] = ak[:, 20]
    v, pos, beta = torch.randn(bh, l, HD, generator=g).to(bf), torch.arange(l).float(), torch.rand(bh, l, generator=g)
    gam = torch.full((2,), 0.9)
    rows = [A.LOG_FIELDS.index(n) for n in ("best", "slot")]

    def run(keys):
        log = _gpu_step(mod, st, (keys, keys, v, pos, beta), gam, 1, gpu)[2]
        return log.reshape(bh, A.LOG_ROWS, A.LOG_COLS)[:, rows, :l].cpu()

    plain = run(kr)
    cos = torch.nn.functional.normalize(kr.float(), dim=-1) @ torch.nn.functional.normalize(ak.float(), dim=-1).mT
    top = cos.topk(2, dim=-1).values
    clear = top[..., 0] - top[..., 1] > 1e-4
    assert torch.equal(plain[:, 1][clear], cos.argmax(-1).float()[clear]) and bool((plain[:, 1, 9] == 20).all())
    bad = kr.clone()
    bad[:, 5, 3] = float("nan")       # beside token 9, in its wavefront
    bad[:, 100, 0] = float("inf")
    got = run(bad)
    for t in (5, 100):                # no finite norm: every cosine is NaN, the first slot holds the first
        assert bool(got[:, 0, t].isnan().all()) and bool((got[:, 1, t] == 0).all())
    keep = [t for t in range(l) if t not in (5, 100)]
    assert torch.equal(got[:, :, keep], plain[:, :, keep])
