"""The few-row linear layers (bolt3_rows_linear) against fp32 products of the same bf16 operands.

An element may differ from the rounded fp32 reference by the fp32 sums' order (about K * 2^-24 of
the terms' magnitude) and one rounding more: 2^-8 relative per rounding.  Row counts from 1 to the
largest, K whose steps do not divide among the wavefronts or are fewer than they are,
strided rows, all three epilogues; and mlp_rows against the module's own ops."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def _call(mode, x, w, gpu, w2=None, bias=None, res=None):
    from bolt3_amd import _abi as A
    M, K = x.shape
    N = w.shape[0]
    out = torch.full((M + 1, N + 4), 7.0, dtype=BF, device=gpu)
    a = A.RowsLinearArgs()
    a.mode, a.M, a.N, a.K = mode, M, N, K
    a.x, a.x_row_stride, a.w, a.w2, a.bias = x.data_ptr(), x.stride(0), w.data_ptr(), A.ptr(w2), A.ptr(bias)
    a.res, a.res_row_stride = A.ptr(res), 0 if res is None else res.stride(0)
    a.out, a.out_row_stride = out.data_ptr(), out.stride(0)
    A.call("bolt3_rows_linear", a, x.device)
    assert bool((out[M] == 7).all()) and bool((out[:M, N:] == 7).all())   # nothing outside [M][N]
    return out[:M, :N].float()


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("M,N,K", [(1, 16, 32), (1, 6192, 2560), (7, 48, 160), (16, 2560, 4096), (15, 32, 2592),
                                   (2, 64, 9728), (9, 16, 320), (16, 16, 288)])
def test_rows_linear(mode, M, N, K, gpu):
    print(f"[case] rows_linear mode={mode} M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(M * 7 + N + K)
    x = torch.randn(M, K + 8, generator=g, device=gpu).to(BF)[:, :K]
    w, w2 = ((torch.randn(N, K, generator=g, device=gpu) * K ** -0.5).to(BF) for _ in range(2))
    bias = torch.randn(N, generator=g, device=gpu).to(BF) if mode == 0 else None
    res = torch.randn(M, N + 4, generator=g, device=gpu).to(BF)[:, :N] if mode == 2 else None
    got = _call(mode, x, w, gpu, w2 if mode == 1 else None, bias, res)
    y = x.float() @ w.float().t()
    if mode == 0:
        ref = y + bias.float()
        bound = 2.0 ** -8 * ref.abs()
    elif mode == 1:
        u = x.float() @ w2.float().t()
        ref = F.silu(y) * u
        # silu's slope is at most 1.1; y, silu, u and the product are rounded
        bound = 2.0 ** -8 * (1.1 * y.abs() * u.abs() + 3 * ref.abs())
    else:
        ref = y + res.float()
        bound = 2.0 ** -8 * (y.abs() + ref.abs())
    bound = 1.01 * bound + 1e-3 * (1.0 if mode != 1 else u.abs() + 1.0)
    assert bool(((got - ref).abs() <= bound).all()), float(((got - ref).abs() / bound).max())


@pytest.mark.parametrize("M", [1, 5, 16])
def test_mlp_rows_matches_module(M, gpu):
    from bolt3_amd.layers import MLP, mlp_rows
    g = torch.Generator(device=gpu).manual_seed(M)
    mlp = MLP(dict(dim=512, intermediate=1536)).to(gpu).to(BF)
    with torch.no_grad():
        for p in mlp.parameters():
            p.normal_(0.0, 0.05, generator=g)
        h, res = (torch.randn(M, 1, 512, generator=g, device=gpu).to(BF) for _ in range(2))
        ref = res + mlp(h)
        got = mlp_rows(mlp, h, res)
        assert got.shape == ref.shape
        # the same roundings: sums in another order flip single roundings of the 1536 products
        assert float((got.float() - ref.float()).norm() / ref.float().norm()) < 4e-3
        seen = []
        hook = mlp.up_proj.register_forward_hook(lambda *_: seen.append(1))
        assert mlp_rows(mlp, h, res) is None         # hooks, other dtypes and more rows: the module's ops
        hook.remove()
        assert mlp_rows(mlp, h.float(), res.float()) is None
        many = torch.zeros(17, 1, 512, dtype=BF, device=gpu)
        assert mlp_rows(mlp, many, many) is None
    assert mlp_rows(mlp, h, res) is None             # gradients enabled


@pytest.mark.parametrize("shape", [(1, 1, 8), (3, 7, 1544), (2, 700, 1536)])
def test_mlp_swiglu_equals_module(shape, gpu):
    """One pass for silu(gate) * up, bit for bit the module's two (each of their roundings kept)."""
    from bolt3_amd.layers import MLP, mlp_swiglu
    g = torch.Generator(device=gpu).manual_seed(shape[1])
    mlp = MLP(dict(dim=64, intermediate=shape[2])).to(gpu).to(BF)
    h = (4 * torch.randn(*shape[:2], 64, generator=g, device=gpu)).to(BF)
    h[0, 0, 0] = float("inf")
    with torch.no_grad():
        for p in mlp.parameters():
            p.normal_(0.0, 0.5, generator=g)
        got, ref = mlp_swiglu(mlp, h), mlp(h)
        assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.nan_to_num(), ref.nan_to_num())
        assert mlp_swiglu(mlp, h.float()) is None
    assert mlp_swiglu(mlp, h) is None


def test_mlp_hooks_and_overrides_see_their_calls(gpu):
    """Both short cuts leave the MLP to its own call where a hook or another forward would see it, and one
    of its linears where only that one has them."""
    from types import SimpleNamespace
    from bolt3_amd import Bolt3Decoder, HybridLM
    from bolt3_amd.layers import MLP, mlp_rows, mlp_swiglu
    mlp = MLP(dict(dim=64, intermediate=128)).to(gpu).to(BF)
    blk = SimpleNamespace(norm2=torch.nn.Identity(), mlp=mlp)
    dec = Bolt3Decoder(HybridLM(vocab_size=8, dim=64, num_layers=0, num_heads=1, num_kv_heads=1, intermediate=8,
                                layer_types=[]).to(gpu))
    few, many = (torch.randn(*s, 64, device=gpu).to(BF) for s in ((3, 1), (2, 40)))
    seen = []

    def calls(m):
        """The calls of m that a step and a prompt make, with and without the few-row form."""
        n = []
        for dec.fuse_mlp in (False, True):
            for x in (few, many):
                seen.clear()
                dec._mlp(blk, x)
                n.append(sum(s is m for s in seen))
        return n

    def note(m, *_):
        seen.append(m)

    with torch.no_grad():
        assert mlp_swiglu(mlp, many) is not None and mlp_rows(mlp, few, few) is not None
        hook = torch.nn.modules.module.register_module_forward_hook(note)
        try:
            assert calls(mlp) == [1, 1, 1, 1] and calls(mlp.up_proj) == [1, 1, 1, 1]
        finally:
            hook.remove()
        for m in (mlp, mlp.down_proj):
            hook = m.register_forward_pre_hook(note)
            assert calls(m) == [1, 1, 1, 1]
            hook.remove()
            own = type(m).forward.__get__(m)
            m.forward = lambda x, m=m, own=own: (note(m), own(x))[1]
            assert calls(m) == [1, 1, 1, 1]
            del m.forward
        assert calls(mlp) == [0, 0, 0, 0]
