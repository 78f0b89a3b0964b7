"""The native host module: metadata views against torch's on the CPU, and
kernel calls with every kind of argument against the ctypes binding."""

import ctypes

import pytest
import torch

from torch_mojo_backend import eager_kernels as ek
from torch_mojo_backend.mojo_device.torch_mojo_tensor import TorchMojoTensor, host


@pytest.mark.parametrize("shape", [(), (1,), (0, 3), (4, 6), (2, 1, 5), (3, 4, 1, 2), (1,) * 8])
def test_views_match_torch(mojo, shape):
    x = torch.arange(torch.Size(shape).numel(), dtype=torch.float32).reshape(shape)
    m = x.to("mojo")
    pairs = [(m.detach(), x.detach()), (m.view(-1), x.view(-1)), (m.unsqueeze(0), x.unsqueeze(0))]
    for a in range(-len(shape), len(shape)):
        for b in range(len(shape)):
            pairs.append((m.transpose(a, b), x.transpose(a, b)))
            pairs.append((m.transpose(a, b).detach(), x.transpose(a, b)))
    for d in range(len(shape)):
        pairs += list(zip(m.split(2, d), x.split(2, d)))
        pairs += list(zip(m.transpose(0, d).split([1] * shape[d], d), x.transpose(0, d).split([1] * shape[d], d))) \
            if shape[0] == shape[d] else []
    for got, ref in pairs:
        assert got.shape == ref.shape and got.dtype == ref.dtype
        assert all(s == r for n, s, r in zip(ref.shape, got._strides, ref.stride()) if n > 1) or ref.numel() == 0
        assert got._is_contiguous == ref.is_contiguous() or ref.numel() == 0
        assert got._numel == ref.numel() and got.storage_offset() == got._offset
        assert torch.equal(got.cpu(), ref)


def test_errors_stay_errors(mojo):
    m = torch.zeros(4, 6).to("mojo")
    with pytest.raises(IndexError):
        m.transpose(0, 2)
    for call in (lambda: m.view(5, 5), lambda: m.view(-1, -1), lambda: m.view(-1, 0), lambda: m.t().view(24)):
        with pytest.raises(RuntimeError):
            call()
    with pytest.raises(NotImplementedError):
        TorchMojoTensor._alloc((1,) * 9, torch.float32, 0)
    with pytest.raises(RuntimeError):
        host().alias(torch.zeros(2))
    assert m.view(4, 6, 1, 1, 1, 1, 1, 1).unsqueeze(0).dim() == 9  # a view has no allocation's limit


@pytest.fixture(scope="module")
def both():
    return ek._load(), ek._NativeLibrary(ek._load())


def test_calls_match_ctypes(both):
    """Integers, pointers (None, addresses, buffers), arrays (tuples, lists,
    ctypes arrays) and floats, through calls that the library answers on the
    host."""
    c, n = both
    for args in ((None, 768, 1, 0, None, 1, 768, 0, 1, 1, 77, 768, 3072), (4096, 1, 300, 0, 8192, 200, 1, 0, 1, 1, 300, 200, 5000)):
        assert n.mi355x_gemm_workspace_bytes(*args) == c.mi355x_gemm_workspace_bytes(*args) > 0
    sizes = [3, 1 << 20, 7]
    arr = (ctypes.c_int64 * 3)(*sizes)
    want = c.mi355x_foreach_norm_workspace_bytes(arr, 3)
    for given in (arr, tuple(sizes), sizes, ctypes.addressof(arr)):
        assert n.mi355x_foreach_norm_workspace_bytes(given, 3) == want > 0
    assert c.mi355x_foreach_norm_workspace_bytes(tuple(sizes), 3) == want
    bad = (None, (0, 0, 0), None, None, [0, 0, 0], None, (ctypes.c_int64 * 3)(), None, (0, 0, 0), 1, 1, 8, 8, 48, 0.1,
           1, 1, None)
    assert n.mi355x_attn_fwd(*bad) == 3 and b"head_dim" in n.mi355x_last_error()
    for wrong in (bad[:-1], bad[:1] + ("x",) + bad[2:], bad[:1] + (tuple(range(65)),) + bad[2:], bad[:9] + (1.5,) + bad[10:]):
        with pytest.raises((TypeError, ValueError)):
            n.mi355x_attn_fwd(*wrong)


def test_every_entry_point_is_native(both):
    slow = {name for name in ek.SIGNATURES if getattr(both[1], name).__class__ is not len.__class__}
    assert slow == {"mi355x_abi_version", "mi355x_last_error", "mi355x_target", "mi355x_source_hash"}
