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
    for call, text in ((lambda: torch.as_strided(m, (2, 2), (1,)), "dimensionality of sizes"),
                       (lambda: m.split([-1, 5]), "non-negative")):
        with pytest.raises(RuntimeError, match=text):
            call()
    with pytest.raises(NotImplementedError):
        TorchMojoTensor._alloc((1,) * 9, torch.float32, 0)
    with pytest.raises(RuntimeError):
        host().alias(torch.zeros(2))
    assert m.view(4, 6, 1, 1, 1, 1, 1, 1).unsqueeze(0).dim() == 9  # a view has no allocation's limit


@pytest.mark.parametrize("shape,dtype", [
    ((2 ** 61,), torch.float32),  # 2^63 bytes: negative
    ((2 ** 30, 2 ** 31), torch.float32),
    ((2 ** 62,), torch.float32),  # 2^64 bytes: zero
    ((2 ** 62 + 4,), torch.float32),  # a small positive number
    ((2 ** 62,), torch.bfloat16), ((2 ** 63 - 1,), torch.bfloat16), ((2 ** 63 - 1,), torch.int64),
    ((2 ** 32, 2 ** 32), torch.uint8), ((2 ** 32, 2 ** 32, 3), torch.float32), ((2 ** 21,) * 8, torch.uint8),
])
def test_sizes_past_64_bits_are_refused(mojo, shape, dtype):
    """Counts of elements or bytes that do not fit in 64 bits, whatever they
    wrap to, raise (as torch.empty does for the CPU) and allocate nothing."""
    for make in (lambda: torch.empty(shape, dtype=dtype, device="mojo"), lambda: torch.zeros(shape, dtype=dtype, device="mojo"),
                 lambda: TorchMojoTensor._alloc(shape, dtype, 0), lambda: host().alloc(shape, dtype, 0)):
        with pytest.raises(Exception):  # noqa: B017 torch's own checks and this module's
            make()
    one = torch.zeros((1,) * len(shape), dtype=dtype).to("mojo")
    with pytest.raises(Exception):  # noqa: B017
        one.expand(shape).contiguous()


def test_views_past_64_bits_are_refused(mojo):
    empty, m = torch.zeros(0, 4).to("mojo"), torch.zeros(4, 6).to("mojo")
    for call in (lambda: empty.view(2 ** 32, 2 ** 32), lambda: m.view(2 ** 32, 2 ** 32, 24), lambda: empty.view(2 ** 33, 2 ** 33, 0),
                 lambda: m.expand(2 ** 40, 2 ** 40, 4, 6), lambda: torch.as_strided(m, (1,), (1,), 2 ** 62),
                 lambda: host().view_of(m, (2 ** 32, 2 ** 32), (0, 0), 0, None), lambda: host().narrow(m, 0, 2 ** 62, 2 ** 62),
                 lambda: host().view_of(m[1:], (1,), (1,), -2 ** 63, None),
                 lambda: host().make(m._holder, m._ptr, (2 ** 32, 2 ** 32), (0, 0), 0, m.dtype, 0, None)):
        with pytest.raises((RuntimeError, IndexError)):
            call()
    assert empty.view(2 ** 40, 0).shape == (2 ** 40, 0) and m.expand(2 ** 40, 4, 6).shape[0] == 2 ** 40


def test_operands_of_other_sizes_are_refused(mojo):
    """A bias that does not broadcast to the product raises, as on the CPU: its
    elements past the end are not read."""
    x, w = torch.ones(3, 6).to("mojo"), torch.ones(6, 6).to("mojo")
    for shape in ((4,), (4, 1), (3, 5), (2, 3, 6)):
        b = torch.ones(shape)
        cpu, dev = (lambda: torch.addmm(b, x.cpu(), w.cpu())), (lambda: torch.addmm(b.to("mojo"), x, w))
        for call in (cpu, dev, lambda: torch.nn.functional.linear(x, w, b.to("mojo")),
                     lambda: torch.addmm(b.to("mojo"), x, w, beta=2.0)):
            with pytest.raises(RuntimeError):
                call()


def test_views_stay_in_their_storage(mojo):
    """as_strided past the storage, with a negative stride or offset, and permute
    with a dimension twice or left out raise, as on the CPU."""
    m = torch.arange(24.0).reshape(4, 6).to("mojo")
    for args in (((4, 6), (6, 1), 1), ((2, 2), (1, 23), 0), ((2,), (-1,), 3), ((2,), (1,), -1), ((25,), (1,)), ((1,), (1,), 24),
                 ((-1,), (1,))):
        for t in (m, m.cpu()):
            with pytest.raises(RuntimeError):
                torch.as_strided(t, *args)
    for dims in ((0, 0), (0,), (1, 0, 1)):
        for t in (m, m.cpu()):
            with pytest.raises(RuntimeError):
                t.permute(dims)
    for t, args in ((m, ((3, 4), (2, 3), 5)), (m[2:], ((2, 2), (1, 2))), (m[2:], ((4, 6), (6, 1), 0)), (m, ((0, 9), (1, 1), 99)),
                    (m.t(), ((24,), (1,)))):
        assert torch.equal(torch.as_strided(t, *args).cpu(), torch.as_strided(m.cpu(), *args[:2], args[2] if len(args) > 2
                                                                              else t.storage_offset()))


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


@pytest.mark.parametrize("m,n,k,tile,splits", [(768, 768, 4096, 64, 3), (768, 768, 8192, 128, 13), (384, 1536, 8192, 128, 13),
                                               (512, 2048, 4096, 128, 8), (2304, 768, 2048, 64, 1), (256, 1152, 16384, 128, 26)])
def test_weight_gradient_plans(both, m, n, k, tile, splits):
    """The K splits (and, by the row sums' slots, the tiles) that weight gradients
    dY^T X take, from the workspace they ask for: 64x64 tiles up to 3.8e9
    multiply-adds, 128x128 above."""
    up = lambda v: (v + 255) // 256 * 256  # noqa: E731
    got = both[1].mi355x_gemm_workspace_bytes(4096, 1, m, 0, 8192, n, 1, 0, 1, 1, m, n, k)
    slots = -(-n // tile) * 2
    assert got == (up(splits * m * n * 4) + up(splits * slots * m * 4) if splits > 1 else 0)


def _plan(native, layout, m, n, k):
    """(tile columns, K splits) of a product, from its workspace: the partial sums
    and the row sums' slots; splits 1 and no tile without a workspace."""
    up = lambda v: (v + 255) // 256 * 256  # noqa: E731
    a = (4096, k, 1, 0) if layout[0] == "N" else (4096, 1, m, 0)
    b = (8192, n, 1, 0) if layout[1] == "N" else (8192, 1, k, 0)
    got = native.mi355x_gemm_workspace_bytes(*a, *b, 1, 1, m, n, k)
    return [(t, s) for t, w in ((64, 2), (128, 2), (192, 2), (256, 4)) for s in range(2, 65)
            if got == up(s * m * n * 4) + up(s * -(-n // t) * w * m * 4)] if got else [(None, 1)]


@pytest.mark.parametrize("layout,m,n,k,tile,splits", [("NT", 80, 768, 3072, 64, 6), ("NT", 568, 1840, 4096, 128, 6),
                                                      ("NT", 2808, 328, 5144, 128, 7), ("NT", 392, 656, 9192, 64, 6)])
def test_small_output_plans(both, layout, m, n, k, tile, splits):
    """From K = 2048 on 64x64 tiles take up to 2.9e9 multiply-adds, counting whole
    tiles; past that K is split over larger ones."""
    assert (tile, splits) in _plan(both[1], layout, m, n, k)


@pytest.mark.parametrize("m,n,k,tile,splits", [(2000, 2248, 2304, None, 1), (3072, 1816, 2304, None, 1),
                                               (2216, 2280, 4392, 192, 2)])
def test_splits_of_three_quarters_of_a_round(both, m, n, k, tile, splits):
    """128x192 tiles on three quarters of the CUs are split where the second block
    per CU saves more than the partial sums cost."""
    assert (tile, splits) in _plan(both[1], "NT", m, n, k)


@pytest.mark.parametrize("m,n,k,tile,splits", [(816, 1384, 8192, 128, 6), (4424, 320, 14520, 128, 4), (1500, 1400, 20008, 256, 6)])
def test_long_k_plans(both, m, n, k, tile, splits):
    """Splits over a long K go to the 256x256 tiles of four waves where each is long
    enough and they save enough."""
    assert (tile, splits) in _plan(both[1], "NT", m, n, k)


def test_every_entry_point_is_native(both):
    slow = {name for name in ek.SIGNATURES if getattr(both[1], name).__class__ is not len.__class__}
    assert slow == {"mi355x_abi_version", "mi355x_last_error", "mi355x_target", "mi355x_source_hash"}
