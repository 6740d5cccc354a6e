"""bolt3_param_grads against fp64 torch sums of the same partial sums: row counts that are not a
multiple of a workgroup's pass, no consolidation step, no q/k norm, all biases or the gates' only,
fp32 and bf16 dz.  The bound is the fp32 sums' own: 2^-23 of the terms' magnitudes times the
longest run of additions in one thread and the tree above it."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,H,HKV,HD,steps,norm,all_bias,dt", [
    (1, 7, 2, 2, 64, 0, False, False, torch.float32),
    (2, 333, 6, 2, 64, 1, True, True, torch.bfloat16),
    (4, 700, 32, 8, 128, 4, True, False, torch.bfloat16),
    (1, 1100, 9, 3, 64, 7, False, True, torch.float32)])
def test_param_grads(B, T, H, HKV, HD, steps, norm, all_bias, dt, gpu):
    from bolt3_amd import _abi as A
    print(f"[case] param_grads B={B} T={T} H={H} HD={HD} steps={steps}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(T)
    n_chunks, nq, S, nb = -(-T // 128), 4, 128, -(-B * T // 2)
    bh, G = B * HKV, H // HKV

    def r(*s):
        return torch.randn(*s, generator=g, device=gpu)

    d_res, d_gam, d_bias = r(bh, n_chunks, HD), r(bh, n_chunks), r(max(steps, 1), B * H, nq, S)
    mass, d_gc = r(max(steps, 1), bh, S).abs() * 4, r(max(steps, 1), bh, HD // 32)
    d_qn, d_kn = r(nb, HD), r(nb, HD)
    cols = (H + 2 * HKV) * HD + HKV + H
    dz = r(B * T, cols + 8).to(dt)
    c0 = 0 if all_bias else (H + 2 * HKV) * HD
    lg = torch.linspace(-9.0, 9.0, HKV, device=gpu)      # both sides of the clamp's range
    out = {k: torch.full((n,), 9.0, device=gpu) for k, n in dict(g_res_w=HD, g_qn_w=HD, g_kn_w=HD, g_bias=cols - c0,
                                                                g_kappa=HKV, g_log_gamma=HKV).items()}
    a = A.ParamGradsArgs()
    a.dtype, a.B, a.T, a.H, a.HKV, a.HD, a.S = A.dtype_code(dt), B, T, H, HKV, HD, S
    a.n_chunks, a.n_qtiles, a.n_steps, a.n_blocks = n_chunks, nq, steps, nb
    a.d_res_w, a.d_gamma, a.log_gamma = d_res.data_ptr(), d_gam.data_ptr(), lg.data_ptr()
    a.d_bias, a.snap_mass, a.d_gamma_chain = d_bias.data_ptr(), mass.data_ptr(), d_gc.data_ptr()
    if norm:
        a.d_qn_w, a.d_kn_w = d_qn.data_ptr(), d_kn.data_ptr()
    a.dz, a.dz_row_stride, a.bias_col, a.n_bias = dz.data_ptr(), dz.stride(0), c0, cols - c0
    for k, t in out.items():
        setattr(a, k, t.data_ptr())
    A.call("bolt3_param_grads", a, gpu)

    def check(name, terms, dim, factor=1.0):
        ref, mag = (terms.sum(dim) * factor), (terms.abs().sum(dim) * abs(factor) if isinstance(factor, float)
                                               else terms.abs().sum(dim) * factor.abs())
        err = (out[name].double() - ref).abs()
        assert bool((err <= 2.0 ** -23 * 600 * mag + 1e-12).all()), (name, float((err / (mag + 1e-12)).max()))

    check("g_res_w", d_res.double().view(-1, HD), 0)
    check("g_bias", dz.double()[:, c0:cols], 0)
    if norm:
        check("g_qn_w", d_qn.double(), 0)
        check("g_kn_w", d_kn.double(), 0)
    else:
        assert bool((out["g_qn_w"] == 9).all())
    n = steps
    kt = d_bias[:n].double().view(n, B, HKV, G, nq, S) * mass[:n].double().clamp_min(1).log().view(n, B, HKV, 1, 1, S)
    check("g_kappa", kt.permute(2, 0, 1, 3, 4, 5).reshape(HKV, n * B * G * nq * S), 1)
    gt = torch.cat([d_gam.double().view(B, HKV, -1).permute(1, 0, 2).reshape(HKV, -1),
                    d_gc[:n].double().view(n, B, HKV, HD // 32).permute(2, 0, 1, 3).reshape(HKV, n * B * (HD // 32))], 1)
    sg = torch.sigmoid(lg.double())
    inside = ((0.999 * sg >= 1e-3) & (0.999 * sg <= 0.999)).double()
    check("g_log_gamma", gt, 1, 0.999 * sg * (1 - sg) * inside)
