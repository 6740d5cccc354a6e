"""The decoder's chunk step (bolt3_chunk_attn mode 1, bf16) against fp32 torch on the same tensors:
every head ratio's kernel, query counts and window lengths at the edges of the 32-key tiles, with
and without sinks, slots (masked ones among them), an older window segment and M_res.

The kernel rounds the probabilities, the attention, the readout and their sum to bf16 (2^-8 of each,
the probabilities' against the values' magnitudes) and splits M_res into 16 mantissa bits.

And against attn_kernel, which M_res and outputs off their alignment take: the same bits."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("G,HD", [(1, 128), (2, 64), (3, 128), (4, 128), (4, 64), (8, 128)])
@pytest.mark.parametrize("t,old,a_len,slots,sinks,readout", [
    (128, 0, 128, True, 4, True), (1, 0, 0, False, 0, True), (33, 31, 0, False, 0, False), (256, 0, 256, True, 4, True),
    (31, 97, 129, True, 4, True), (64, 33, 128, False, 4, True), (5, 1, 3, True, 0, False), (100, 127, 200, True, 1, True)])
def test_chunk_step_matches_fp32(G, HD, t, old, a_len, slots, sinks, readout, gpu):
    from bolt3_amd import _abi as A
    print(f"[case] chunk step G={G} HD={HD} t={t} old={old} a={a_len}", flush=True)
    B, HKV, S, cap = 2, 2, 128, 512
    H = G * HKV
    g = torch.Generator(device=gpu).manual_seed(t + old)

    def r(*s, dt=BF):
        return torch.randn(*s, generator=g, device=gpu).to(dt)

    q, q_raw, eta = r(B, H, t, HD), r(B, H, t, HD), torch.tanh(r(B, H, t, dt=torch.float32))
    wk, wv = r(B, HKV, cap, HD), r(B, HKV, cap, HD)
    sk, sv, ck, cv = r(B * HKV, S, HD), r(B * HKV, S, HD), r(B, HKV, 4, HD), r(B, HKV, 4, HD)
    bias = torch.rand(B * HKV, S, generator=g, device=gpu) * 2
    bias[:, 5:9] = float("-inf")
    m = 0.3 * r(B, HKV, HD, HD, dt=torch.float32)
    gamma, res_w = torch.rand(HKV, generator=g, device=gpu) * 0.5 + 0.3, torch.rand(HD, generator=g, device=gpu) + 0.5
    y = torch.full((B, t + 1, H * HD), 7.0, dtype=BF, device=gpu)
    a0, b0 = 0, 256
    a = A.AttnArgs()
    a.dtype, a.B, a.H, a.HKV, a.HD, a.S, a.C, a.n_sinks, a.mode, a.n_q, a.score_round = 1, B, H, HKV, HD, S, 128, 4, 1, t, 0
    a.q_rope, a.q_raw, a.q_sb, a.q_sh = q.data_ptr(), q_raw.data_ptr(), q.stride(0), q.stride(1)
    a.eta, a.e_sb, a.e_sh = eta.data_ptr(), eta.stride(0), eta.stride(1)
    a.win_k, a.win_v, a.w_sb, a.w_sh = wk.data_ptr(), wv.data_ptr(), wk.stride(0), wk.stride(1)
    a.a_start, a.a_len, a.b_start, a.b_len = a0, a_len, b0, min(old, 256 - t) + t
    old = a.b_len - t
    a.sink_k, a.sink_v, a.s_sb, a.s_sh, a.n_sink_keys = ck.data_ptr(), cv.data_ptr(), ck.stride(0), ck.stride(1), sinks
    a.slot_k, a.slot_v, a.slot_bias, a.slot_step, a.has_slots = sk.data_ptr(), sv.data_ptr(), bias.data_ptr(), 0, int(slots)
    a.m_res, a.m_step = (m.data_ptr() if readout else None), 0
    a.gamma, a.res_w, a.eps = gamma.data_ptr(), res_w.data_ptr(), 1e-6
    a.y, a.y_sb, a.y_st = y.data_ptr(), y.stride(0), y.stride(1)
    A.call("bolt3_chunk_attn", a, gpu)
    assert bool((y[:, t] == 7).all())

    def heads(x):
        return x.float().repeat_interleave(G, dim=1)

    ks, vs, bs = [], [], []
    if sinks:
        ks.append(ck[:, :, :sinks]), vs.append(cv[:, :, :sinks]), bs.append(torch.zeros(B, HKV, sinks, device=gpu))
    if slots:
        ks.append(sk.view(B, HKV, S, HD)), vs.append(sv.view(B, HKV, S, HD)), bs.append(bias.view(B, HKV, S))
    n_pre = sum(k.shape[2] for k in ks) + a_len
    for s0, n in ((a0, a_len), (b0, a.b_len)):
        ks.append(wk[:, :, s0:s0 + n]), vs.append(wv[:, :, s0:s0 + n]), bs.append(torch.zeros(B, HKV, n, device=gpu))
    k, v, bb = heads(torch.cat(ks, 2)), heads(torch.cat(vs, 2)), torch.cat(bs, 2).repeat_interleave(G, dim=1)
    sc = q.float() @ k.transpose(-1, -2).contiguous() * HD ** -0.5 + bb.unsqueeze(2)
    pos = torch.arange(k.shape[2], device=gpu)
    sc = sc.masked_fill(pos[None, :] > n_pre + old + torch.arange(t, device=gpu)[:, None], float("-inf"))
    att = torch.softmax(sc, -1) @ v
    ref, rd = att, torch.zeros_like(att)
    if readout:
        u = F.normalize(q_raw.float(), dim=-1) @ heads(m)
        u = u * ((1 - gamma) / HD ** 0.5).repeat_interleave(G).view(1, H, 1, 1)
        rd = eta.unsqueeze(-1) * (u * torch.rsqrt(u.pow(2).mean(-1, keepdim=True) + 1e-6) * res_w)
        ref = att + rd
    got = y[:, :t].float().view(B, t, H, HD).transpose(1, 2)
    mass = torch.softmax(sc, -1) @ v.abs()          # every probability off by 2^-8 of itself
    bound = 1.1 * 2.0 ** -8 * (mass + att.abs() + rd.abs() + ref.abs()) + 1e-4 * (mass + rd.abs())
    worst = float(((got - ref).abs() / bound).max())
    assert worst <= 1.0, worst


def _step(gpu, G, HD, t, old, a_len, off):
    """One chunk step, its M_res off floats into a buffer and its output rows off elements apart from a
    multiple of four; every field in use, the first slots masked."""
    from bolt3_amd import _abi as A
    B, HKV, S, cap = 2, 2, 128, 512
    H = G * HKV
    g = torch.Generator(device=gpu).manual_seed(t + old + HD)

    def r(*s, dt=BF):
        return torch.randn(*s, generator=g, device=gpu).to(dt)

    q, q_raw, eta = r(B, H, t, HD), r(B, H, t, HD), torch.tanh(r(B, H, t, dt=torch.float32))
    wk, wv, sk, sv = r(B, HKV, cap, HD), r(B, HKV, cap, HD), r(B * HKV, S, HD), r(B * HKV, S, HD)
    ck, cv, m0 = r(B, HKV, 4, HD), r(B, HKV, 4, HD), 0.3 * r(B, HKV, HD, HD, dt=torch.float32)
    bias, gamma, res_w = (torch.rand(*s, generator=g, device=gpu) for s in ((B * HKV, S), (HKV,), (HD,)))
    bias[:, :40] = float("-inf")
    buf = torch.zeros(m0.numel() + 4, device=gpu)
    m = buf[off:off + m0.numel()].view(m0.shape).copy_(m0)
    st = H * HD + off
    y = torch.full((B * (t + 1) * st + 4,), 7.0, dtype=BF, device=gpu)[off:]
    a = A.AttnArgs()
    a.dtype, a.B, a.H, a.HKV, a.HD, a.S, a.C, a.n_sinks, a.mode, a.n_q, a.score_round = 1, B, H, HKV, HD, S, 128, 4, 1, t, 0
    a.q_rope, a.q_raw, a.q_sb, a.q_sh = q.data_ptr(), q_raw.data_ptr(), q.stride(0), q.stride(1)
    a.eta, a.e_sb, a.e_sh = eta.data_ptr(), eta.stride(0), eta.stride(1)
    a.win_k, a.win_v, a.w_sb, a.w_sh = wk.data_ptr(), wv.data_ptr(), wk.stride(0), wk.stride(1)
    a.a_start, a.a_len, a.b_start, a.b_len = 0, a_len, 256, old + t
    a.sink_k, a.sink_v, a.s_sb, a.s_sh, a.n_sink_keys = ck.data_ptr(), cv.data_ptr(), ck.stride(0), ck.stride(1), 4
    a.slot_k, a.slot_v, a.slot_bias, a.slot_step, a.has_slots = sk.data_ptr(), sv.data_ptr(), bias.data_ptr(), 0, 1
    a.m_res, a.m_step, a.gamma, a.res_w, a.eps = m.data_ptr(), 0, gamma.data_ptr(), res_w.data_ptr(), 1e-6
    a.y, a.y_sb, a.y_st = y.data_ptr(), (t + 1) * st, st
    A.call("bolt3_chunk_attn", a, gpu)
    out = y[:B * (t + 1) * st].view(B, t + 1, st)
    assert bool((out[:, t] == 7).all()) and bool((out[..., H * HD:] == 7).all())
    return out[:, :t, :H * HD]


@pytest.mark.parametrize("G,HD", [(1, 64), (1, 128), (2, 64), (2, 128), (4, 64), (4, 128), (8, 64), (8, 128)])
@pytest.mark.parametrize("t,old,a_len", [(128, 0, 128), (1, 5, 0), (33, 31, 129), (100, 127, 200)])
def test_chunk_step_gives_attn_kernels_bits(G, HD, t, old, a_len, gpu):
    """A state's later slot decisions follow every rounding of the layers below, so which kernel takes a
    chunk step must not show."""
    print(f"[case] chunk step bits G={G} HD={HD} t={t}", flush=True)
    staged = _step(gpu, G, HD, t, old, a_len, 0)
    for off in (1, 2):
        assert torch.equal(_step(gpu, G, HD, t, old, a_len, off), staged)
