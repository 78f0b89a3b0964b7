"""mi355x_copy over dimension orders, strides and row lengths, exact."""

import itertools

import pytest
import torch

from abi import CODE, call, i64

pytestmark = pytest.mark.gpu


def _copy(dst, src):
    call("mi355x_copy", dst.data_ptr(), CODE[dst.dtype], i64(*dst.stride()), src.data_ptr(), CODE[src.dtype],
         i64(*src.stride()), i64(*src.shape), src.dim(), None)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.uint8, torch.int64])
@pytest.mark.parametrize("shape", [(3, 5, 7, 64), (2, 1, 9, 16), (4, 3, 2, 520), (2, 3, 4, 5), (1, 6, 1, 8),
                                   (2, 70, 3, 131), (65, 8, 64, 9), (130, 7, 2, 66)])
def test_copy_every_order(kernels, dtype, shape):
    """Source and destination each in every dimension order, dense or as a
    slice of a wider buffer, on bases that are 16-byte aligned and not."""
    n = 4 * torch.Size(shape).numel()
    values = torch.randint(0, 100, (n + 64,), device="cuda").to(dtype)
    cases = list(itertools.permutations(range(4)))
    for k, (ps, pd) in enumerate(itertools.product(cases[::5], cases[::3])):
        sshape, dshape = [shape[i] for i in ps], [shape[i] for i in pd]
        off = (0, 16, 1, 3)[k % 4]
        wide = 2 if k % 3 else 1  # every second block of the second dimension
        src = values[off:off + wide * torch.Size(shape).numel()]
        src = src.view(sshape[0], wide * sshape[1], sshape[2], sshape[3])[:, :sshape[1]]
        src = src.permute([ps.index(i) for i in range(4)])
        store = torch.full((n + 64,), 7, device="cuda").to(dtype)
        dst = store[off:off + wide * torch.Size(shape).numel()]
        dst = dst.view(dshape[0], wide * dshape[1], dshape[2], dshape[3])[:, :dshape[1]]
        dst = dst.permute([pd.index(i) for i in range(4)])
        want = store.clone()
        torch.as_strided(want, dst.shape, dst.stride(), dst.storage_offset()).copy_(src)
        _copy(dst, src)
        assert torch.equal(store, want), (ps, pd, off, wide)


@pytest.mark.parametrize("src_dtype,dst_dtype", [(torch.float32, torch.bfloat16), (torch.float32, torch.float16),
                                                 (torch.bfloat16, torch.float32), (torch.float16, torch.float32),
                                                 (torch.int64, torch.float32), (torch.bfloat16, torch.float16)])
@pytest.mark.parametrize("shape", [(3, 70, 131), (129, 8, 64), (5, 7, 300)])
def test_cast_every_order(kernels, src_dtype, dst_dtype, shape):
    """Casts between every pair of dimension orders: the rounding of torch's."""
    values = torch.randn(torch.Size(shape).numel(), device="cuda") * 100
    for ps, pd in itertools.product(itertools.permutations(range(3)), repeat=2):
        src = values.to(src_dtype).view([shape[i] for i in ps]).permute([ps.index(i) for i in range(3)])
        dst = torch.zeros([shape[i] for i in pd], dtype=dst_dtype, device="cuda").permute([pd.index(i) for i in range(3)])
        _copy(dst, src)
        assert torch.equal(dst, src.to(dst_dtype)), (ps, pd)


@pytest.mark.parametrize("rows,row_bytes", [(1, 16384), (3, 16384 * 3), (5, 16384 * 2 + 16), (16, 16368), (2047, 32784),
                                            (2048, 32784)])
def test_copy_few_long_rows(kernels, rows, row_bytes):
    """Rows cut into pieces of 16 KB (below 2048 of them) and rows that a wave takes
    whole, from a strided source and from one row broadcast; nothing else is written."""
    n, wide = row_bytes // 4, row_bytes // 4 + 8
    src = torch.randn(rows, wide, device="cuda")
    for view in (src[:, 4:4 + n], src[:1, :n].expand(rows, n)):
        store = torch.full((rows, wide), 7.0, device="cuda")
        _copy(store[:, :n], view)
        assert torch.equal(store[:, :n], view) and bool((store[:, n:] == 7.0).all())
