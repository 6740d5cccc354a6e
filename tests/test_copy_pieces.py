"""Several strided copies in one launch: the rule that makes a piece of a pair of tensors (bytes moved
on the CPU as the kernel moves them, against Tensor.copy_), and the kernel."""
import ctypes

import pytest
import torch

from bolt3_amd import decoder as D

F32, BF, U8 = torch.float32, torch.bfloat16, torch.uint8


def _pairs(device, dtype):
    """(dst, src) over the forms: whole tensors, slices of a dimension in the middle, odd lengths and
    offsets, one element, expanded, transposed and stepped sources, permuted targets."""
    g = torch.Generator().manual_seed(3)

    def new(*shape):
        return torch.randint(0, 255, shape, generator=g).to(dtype).to(device)

    yield new(2, 3, 8, 16), new(2, 3, 8, 16)
    yield new(2, 3, 40, 16)[:, :, 8:29], new(2, 3, 33, 16)[:, :, 5:26]
    yield new(2, 3, 40)[:, :, 3:24], new(2, 3, 33)[:, :, 1:22]
    yield new(2, 3, 40)[:, :, 3:24], new(2, 3, 21)
    yield new(2, 3, 21), new(2, 3, 33)[:, :, 12:]
    yield new(50)[7:8], new(1)
    yield new(4, 1, 5, 1), new(4, 2, 5, 3)[:, 1:, :, :1]
    yield new(4, 6), new(1, 6).expand(4, 6)
    yield new(4, 6), new(6, 4).t()
    yield new(4, 6), new(4, 12)[:, ::2]
    yield new(3, 4, 6).permute(1, 0, 2), new(4, 3, 6)
    yield new(2, 3, 9, 6)[:, :2, 1:4], new(2, 2, 3, 6)
    yield new(2, 700, 130)[:, 1:, :129], new(2, 699, 129)


@pytest.mark.parametrize("dtype", [F32, BF, U8])
def test_piece_moves_what_copy_moves(dtype):
    made = 0
    for dst, src in _pairs("cpu", dtype):
        f = D._copy_piece(dst, src)
        if f is None:
            continue
        made += 1
        rows, nbytes, ss, ds = f
        ref = torch.empty_like(src).copy_(src)
        for r in range(rows):
            ctypes.memmove(dst.data_ptr() + r * ds, src.data_ptr() + r * ss, nbytes)
        assert torch.equal(dst, ref), (dst.shape, dst.stride(), src.stride())
    assert made >= 8
    a = torch.zeros(4, 6)
    assert D._copy_piece(a, a.double()) is None and D._copy_piece(a, torch.zeros(1, 6)) is None


def test_copy_all_keeps_the_order_of_overlapping_pairs():
    x, y = torch.arange(12.0), torch.arange(12.0)
    D._copy_all([(x[6:], x[:6]), (x[:6], x[6:])])
    y[6:].copy_(y[:6].clone())
    y[:6].copy_(y[6:].clone())
    assert torch.equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, BF, U8])
def test_copy_all_on_the_gpu(dtype, gpu):
    pairs = list(_pairs(gpu, dtype))
    whole = [d._base if d._base is not None else d for d, _ in pairs]
    ref = [w.clone() for w in whole]
    for (d, s), r in zip(pairs, ref):
        r.as_strided(d.shape, d.stride(), d.storage_offset()).copy_(s)
    D._copy_all(pairs)
    for i, (w, r) in enumerate(zip(whole, ref)):
        assert torch.equal(w, r), i          # and nothing beside the target has changed
