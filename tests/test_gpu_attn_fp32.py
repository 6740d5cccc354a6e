"""The fp32 chunk attention's two widths of workgroup and two ways to load keys: a few rows of the batch
(narrow workgroups) and many (wide), aligned rows (16-byte loads) and rows at an odd float, all bit
for bit the same, and within the fp32 sums' rounding of torch in float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _run(gpu, B, G, HKV, HD, t, n_old, q, k, v, shift):
    from bolt3_amd import _abi as A
    H = G * HKV
    cap = k.shape[2]

    def at(x):      # the same values, shift floats into a buffer
        buf = torch.empty(x.numel() + 4, device=gpu)
        out = buf[shift:shift + x.numel()].view(x.shape)
        return out.copy_(x)

    q, k, v = at(q[:B]), at(k[:B]), at(v[:B])
    eta, res_w, gamma = torch.zeros(B, H, t, device=gpu), torch.ones(HD, device=gpu), torch.full((HKV,), 0.5, device=gpu)
    y = torch.full((B, t, H * HD), 7.0, device=gpu)
    a = A.AttnArgs()
    a.dtype, a.B, a.H, a.HKV, a.HD, a.S, a.C, a.n_sinks, a.mode, a.n_q, a.score_round = 0, B, H, HKV, HD, 128, 128, 4, 1, t, 0
    a.q_rope, a.q_raw, a.q_sb, a.q_sh = q.data_ptr(), q.data_ptr(), q.stride(0), q.stride(1)
    a.eta, a.e_sb, a.e_sh = eta.data_ptr(), eta.stride(0), eta.stride(1)
    a.win_k, a.win_v, a.w_sb, a.w_sh = k.data_ptr(), v.data_ptr(), k.stride(0), k.stride(1)
    a.a_start, a.a_len, a.b_start, a.b_len = 0, n_old, n_old, cap - n_old
    a.has_slots, a.n_sink_keys = 0, 0
    a.gamma, a.res_w, a.eps = gamma.data_ptr(), res_w.data_ptr(), 1e-6
    a.y, a.y_sb, a.y_st = y.data_ptr(), y.stride(0), y.stride(1)
    A.call("bolt3_chunk_attn", a, gpu)
    return y


@pytest.mark.parametrize("G,HD", [(2, 64), (3, 64), (4, 128)])
@pytest.mark.parametrize("t,n_old,extra", [(128, 37, 5), (65, 0, 0), (97, 130, 31)])
def test_fp32_widths_and_alignments(G, HD, t, n_old, extra, gpu):
    print(f"[case] fp32 attention G={G} HD={HD} t={t} old={n_old}", flush=True)
    B, HKV = 64, 2                      # 2 x 128 wide workgroups; one row of the batch: 4 x 2 narrow ones
    g = torch.Generator(device=gpu).manual_seed(t + HD)
    cap = n_old + extra + t
    q = torch.randn(B, G * HKV, t, HD, generator=g, device=gpu)
    k, v = (torch.randn(B, HKV, cap, HD, generator=g, device=gpu) for _ in range(2))
    many = _run(gpu, B, G, HKV, HD, t, n_old, q, k, v, 0)
    for shift in (0, 1):
        few = _run(gpu, 1, G, HKV, HD, t, n_old, q, k, v, shift)
        assert torch.equal(few[0], many[0])
    assert torch.equal(_run(gpu, B, G, HKV, HD, t, n_old, q, k, v, 1), many)
    kk, vv = (x[:1].double().repeat_interleave(G, dim=1) for x in (k, v))
    sc = q[:1].double() @ kk.transpose(-1, -2).contiguous() * HD ** -0.5
    pos = torch.arange(cap, device=gpu)
    sc = sc.masked_fill(pos[None, :] > n_old + extra + torch.arange(t, device=gpu)[:, None], float("-inf"))
    ref = (torch.softmax(sc, -1) @ vv).transpose(1, 2).reshape(t, -1)
    # sums of cap probabilities and HD products in fp32: about (cap + HD) 2^-24 of the values' size
    assert float((many[0] - ref).abs().max()) <= (cap + HD) * 2.0 ** -24 * float(v[0].abs().max())
