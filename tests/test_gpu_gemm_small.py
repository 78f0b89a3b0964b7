"""The 16-bit GEMM's tiles, plans and stores through the C ABI, against 64-bit
results."""

import pytest
import torch

from abi import CODE, call, dev, host, lib, p, workspace

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("layout", ["NT", "NN", "TN", "TT"])
@pytest.mark.parametrize("m,n,k,batch", [(1, 8, 8, 1), (63, 72, 64, 2), (64, 64, 72, 1), (65, 128, 192, 1),
                                         (77, 200, 256, 1), (129, 64, 328, 3), (8, 768, 3072, 1), (200, 136, 2200, 2)])
def test_gemm_64_tiles(kernels, dtype, layout, m, n, k, batch):
    """Fewer k-steps than stages, exactly as many, more, a ragged last one and
    K splits; edges of the tile; operands read in place where their extents
    allow and packed otherwise; C in f32 with the row sums of A.  Products of
    16-bit operands are exact in f32, so a chain of k sums (each rounded or
    cut) is within (k + 3) * 2^-23 of sum |a||b|."""
    gen = torch.Generator().manual_seed(m * 7919 + n * 31 + k)
    A, B = (torch.randn(batch, *s, generator=gen).to(dtype) for s in ((m, k), (k, n)))
    ta = dev((A.transpose(1, 2) if layout[0] == "T" else A).contiguous())
    tb = dev((B.transpose(1, 2) if layout[1] == "T" else B).contiguous())
    a_rs, a_cs = (k, 1) if layout[0] == "N" else (1, m)
    b_rs, b_cs = (n, 1) if layout[1] == "N" else (1, k)
    a_args, b_args = (p(ta), a_rs, a_cs, m * k), (p(tb), b_rs, b_cs, k * n)
    ws_n = lib().mi355x_gemm_workspace_bytes(*a_args, *b_args, CODE[dtype], batch, m, n, k)
    ws = workspace(ws_n) if ws_n else None
    c = torch.full((batch, m, n), float("nan"), device="cuda")
    rows = torch.full((batch, m), float("nan"), device="cuda")
    call("mi355x_gemm_ex", p(c), 0, n, m * n, *a_args, *b_args, CODE[dtype], None, 0, 0, p(rows), 0, batch, m, n, k,
         p(ws), ws_n, None)
    a, b, u = A.double(), B.double(), (k + 3) * 2.0 ** -23
    assert bool(((host(c).double() - a @ b).abs() <= u * (a.abs() @ b.abs())).all())
    assert bool(((host(rows).double() - a.sum(2)).abs() <= u * a.abs().sum(2)).all())


@pytest.mark.parametrize("m,n,layout", [(65, 67, "NT"), (1030, 2051, "NN"), (4100, 2301, "NT"), (8200, 5003, "NN")])
@pytest.mark.parametrize("c_dtype,flags", [(torch.bfloat16, 0), (torch.float16, 0), (torch.float32, 0), (torch.float32, 2),
                                           (torch.bfloat16, 1)])
def test_gemm_stores_at_any_alignment(kernels, m, n, layout, c_dtype, flags):
    """Partial tiles (64x64, 128x128 and twice 128x192) into rows of C at every
    alignment."""
    _stores_at_any_alignment(m, n, 64, layout, c_dtype, flags)


@pytest.mark.parametrize("k", [64, 2056])
@pytest.mark.parametrize("c_dtype,flags", [(torch.bfloat16, 0), (torch.float32, 0), (torch.float32, 2), (torch.bfloat16, 1)])
def test_gemm_wide_tiles_store_at_any_alignment(kernels, k, c_dtype, flags):
    """The same from 256x256 tiles: of eight waves, and (K = 2056) of four."""
    _stores_at_any_alignment(4090, 4093, k, "NT", c_dtype, flags)


def _stores_at_any_alignment(m, n, k, layout, c_dtype, flags):
    """C into an odd row stride and a base shifted by one element: every element
    of C right, nothing else written.  Sums of k exact products, rounded once to
    the output type (and through bf16 with ROUND)."""
    ld, shift = n + 3 + n % 2, 1
    gen = torch.Generator().manual_seed(m + n)
    A, B, bias = (torch.randn(*s, generator=gen).bfloat16() for s in ((m, k), (k, n), (n,)))
    ta, tb, tbias = dev(A), dev((B.t() if layout[1] == "T" else B).contiguous()), dev(bias)
    b_rs, b_cs = (n, 1) if layout[1] == "N" else (1, k)
    store = torch.full((shift + m * ld,), 3.0, dtype=c_dtype, device="cuda")
    args = (p(ta), k, 1, 0, p(tb), b_rs, b_cs, 0, 1)
    ws_n = lib().mi355x_gemm_workspace_bytes(*args, 1, m, n, k)
    ws = workspace(ws_n) if ws_n else None
    call("mi355x_gemm_ex", p(store) + shift * store.element_size(), CODE[c_dtype], ld, 0, *args, p(tbias), 1, flags, None,
         0, 1, m, n, k, p(ws), ws_n, None)
    got = store[shift:].view(m, ld)
    assert bool((got[:, n:] == 3.0).all()) and float(store[0]) == 3.0
    exact = ta.double() @ dev(B).double() + tbias.double() + (3.0 if flags == 1 else 0.0)
    ulp = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}[c_dtype]
    if flags == 2:
        ulp = 2.0 ** -8
        assert torch.equal(got[:, :n], got[:, :n].bfloat16().float())
    bound = ulp * exact.abs() + (k + 3) * 2.0 ** -23 * (ta.double().abs() @ dev(B).double().abs() + 4)
    assert bool(((got[:, :n].double() - exact).abs() <= bound).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("layout", ["NT", "NN", "TN", "TT"])
@pytest.mark.parametrize("m,n,k,batch", [(700, 6000, 768, 1), (2500, 10007, 520, 2), (130, 33000, 136, 1), (400, 4104, 640, 2),
                                         (9000, 15003, 288, 1)])
def test_gemm_groups_of_tile_rows(kernels, dtype, layout, m, n, k, batch):
    """B beyond 8 MB: the tiles are walked in groups of rows, the last group a
    partial one; beyond 4 MB in one group where A is small; and row by row where
    K is short and C, in rows that are not aligned, past 256 MB.  Each element of
    C against products exact in f64."""
    gen = torch.Generator().manual_seed(m + n + k)
    A, B = (torch.randn(batch, *s, generator=gen).to(dtype) for s in ((m, k), (k, n)))
    ta = dev((A.transpose(1, 2) if layout[0] == "T" else A).contiguous())
    tb = dev((B.transpose(1, 2) if layout[1] == "T" else B).contiguous())
    a_rs, a_cs = (k, 1) if layout[0] == "N" else (1, m)
    b_rs, b_cs = (n, 1) if layout[1] == "N" else (1, k)
    args = (p(ta), a_rs, a_cs, m * k, p(tb), b_rs, b_cs, k * n)
    ws_n = lib().mi355x_gemm_workspace_bytes(*args, CODE[dtype], batch, m, n, k)
    ws = workspace(ws_n) if ws_n else None
    c = torch.full((batch, m, n), float("nan"), device="cuda")
    call("mi355x_gemm_ex", p(c), 0, n, m * n, *args, CODE[dtype], None, 0, 0, None, 0, batch, m, n, k, p(ws), ws_n, None)
    for i in range(batch):
        a, b = dev(A[i]).double(), dev(B[i]).double()
        assert bool(((c[i].double() - a @ b).abs() <= (k + 3) * 2.0 ** -23 * (a.abs() @ b.abs())).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("layout", ["NT", "NN", "TN", "TT"])
@pytest.mark.parametrize("m,n,k,rows", [(520, 300, 8200, False), (2100, 776, 8192, False), (3600, 3850, 2048, False),
                                        (1540, 3090, 4104, True), (1540, 3090, 4160, False)])
def test_gemm_long_k(kernels, dtype, layout, m, n, k, rows):
    """Long K in each plan around the 256x256 tiles of four waves (which take the
    whole K of 3600 x 3850): 64x64 tiles and 128x128 tiles in splits, 128x192 tiles
    whole and in two splits, ragged last stages, and row sums."""
    gen = torch.Generator().manual_seed(m + 3 * n + k)
    n8, m8 = (n + 7) // 8 * 8, (m + 7) // 8 * 8  # rows in place: strides of whole 16 bytes
    A, B = (torch.randn(*s, generator=gen).to(dtype) for s in ((m8, k), (k, n8)))
    ta = dev((A.t() if layout[0] == "T" else A).contiguous())
    tb = dev((B.t() if layout[1] == "T" else B).contiguous())
    a_rs, a_cs = (k, 1) if layout[0] == "N" else (1, m8)
    b_rs, b_cs = (n8, 1) if layout[1] == "N" else (1, k)
    args = (p(ta), a_rs, a_cs, 0, p(tb), b_rs, b_cs, 0)
    ws_n = lib().mi355x_gemm_workspace_bytes(*args, CODE[dtype], 1, m, n, k)
    ws = workspace(ws_n) if ws_n else None
    c = torch.full((m, n), float("nan"), device="cuda")
    sums = torch.full((m,), float("nan"), device="cuda") if rows else None
    call("mi355x_gemm_ex", p(c), 0, n, 0, *args, CODE[dtype], None, 0, 0, p(sums) if rows else None, 0, 1, m, n, k, p(ws),
         ws_n, None)
    a, b, u = dev(A[:m]).double(), dev(B[:, :n]).double(), (k + 3) * 2.0 ** -23
    assert bool(((c.double() - a @ b).abs() <= u * (a.abs() @ b.abs())).all())
    if rows:
        assert bool(((sums.double() - a.sum(1)).abs() <= u * a.abs().sum(1)).all())


@pytest.mark.parametrize("layout", ["NT", "NN", "TN", "TT"])
@pytest.mark.parametrize("k", [2048, 2056, 2112, 2176, 2240])
def test_gemm_long_k_ends(kernels, layout, k):
    """Every place in the ring for the last stage, whole and ragged, against
    the same product in f64 (K from 2048: the four-wave tiles)."""
    m, n = 3608, 3848
    gen = torch.Generator().manual_seed(k)
    A, B = (torch.randn(*s, generator=gen).bfloat16() for s in ((m, k), (k, n)))
    ta = dev((A.t() if layout[0] == "T" else A).contiguous())
    tb = dev((B.t() if layout[1] == "T" else B).contiguous())
    a_rs, a_cs = (k, 1) if layout[0] == "N" else (1, m)
    b_rs, b_cs = (n, 1) if layout[1] == "N" else (1, k)
    args = (p(ta), a_rs, a_cs, 0, p(tb), b_rs, b_cs, 0)
    ws_n = lib().mi355x_gemm_workspace_bytes(*args, 1, 1, m, n, k)
    ws = workspace(ws_n) if ws_n else None
    c = torch.full((m, n), float("nan"), device="cuda")
    call("mi355x_gemm_ex", p(c), 0, n, 0, *args, 1, None, 0, 0, None, 0, 1, m, n, k, p(ws), ws_n, None)
    a, b = dev(A).double(), dev(B).double()
    assert bool(((c.double() - a @ b).abs() <= (k + 3) * 2.0 ** -23 * (a.abs() @ b.abs())).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("layout,m,n,k,splits,batch", [("NT", 1500, 1400, 20008, 6, 1), ("NN", 1500, 1400, 20000, 6, 1),
                                                       ("NN", 1000, 1100, 20008, 6, 2), ("TN", 1500, 2900, 8200, 3, 1),
                                                       ("TT", 1500, 2900, 8200, 3, 1), ("TN", 1500, 2900, 6144, 3, 1),
                                                       ("TT", 1500, 2900, 6152, 3, 1)])
@pytest.mark.parametrize("rows", [False, True])
def test_gemm_wide_tiles_in_splits(kernels, dtype, layout, m, n, k, splits, batch, rows):
    """K splits of the 256x256 tiles (an odd count of 128-wide columns tells their
    row-sum slots from the smaller tiles', so that the workspace's size names the
    plan), the last split shorter and ragged or whole: of four waves, and with row
    sums of eight."""
    n8, m8, up = (n + 7) // 8 * 8, (m + 7) // 8 * 8, lambda v: (v + 255) // 256 * 256
    gen = torch.Generator().manual_seed(m + 3 * n + k)
    A, B = (torch.randn(batch, *s, generator=gen).to(dtype) for s in ((m8, k), (k, n8)))
    ta = dev((A.transpose(1, 2) if layout[0] == "T" else A).contiguous())
    tb = dev((B.transpose(1, 2) if layout[1] == "T" else B).contiguous())
    a_rs, a_cs = (k, 1) if layout[0] == "N" else (1, m8)
    b_rs, b_cs = (n8, 1) if layout[1] == "N" else (1, k)
    args = (p(ta), a_rs, a_cs, m8 * k, p(tb), b_rs, b_cs, k * n8)
    ws_n = lib().mi355x_gemm_workspace_bytes(*args, CODE[dtype], batch, m, n, k)
    assert ws_n == up(splits * batch * m * n * 4) + up(splits * batch * -(-n // 256) * 4 * m * 4)
    ws, c = workspace(ws_n), torch.full((batch, m, n), float("nan"), device="cuda")
    sums = torch.full((batch, m), float("nan"), device="cuda") if rows else None
    call("mi355x_gemm_ex", p(c), 0, n, m * n, *args, CODE[dtype], None, 0, 0, p(sums), 0, batch, m, n, k, p(ws), ws_n, None)
    for i in range(batch):
        a, b, u = dev(A[i, :m]).double(), dev(B[i, :, :n]).double(), (k + 3) * 2.0 ** -23
        assert bool(((c[i].double() - a @ b).abs() <= u * (a.abs() @ b.abs())).all())
        if rows:
            assert bool(((sums[i].double() - a.sum(1)).abs() <= u * a.abs().sum(1)).all())


@pytest.mark.parametrize("layout", ["TN", "TT"])
@pytest.mark.parametrize("k", [72, 520, 1984])
def test_gemm_row_sums_of_whole_wide_tiles(kernels, layout, k):
    """Row sums beside the whole K of 256x256 tiles with an m-contiguous A: its
    fragments are read one at a time there."""
    m, n = 4090, 4104
    gen = torch.Generator().manual_seed(k)
    A, B = (torch.randn(*s, generator=gen).bfloat16() for s in ((4096, k), (k, n)))
    ta, tb = dev(A.t().contiguous()), dev((B.t() if layout[1] == "T" else B).contiguous())
    b_rs, b_cs = (n, 1) if layout[1] == "N" else (1, k)
    args = (p(ta), 1, 4096, 0, p(tb), b_rs, b_cs, 0)
    ws_n = lib().mi355x_gemm_workspace_bytes(*args, 1, 1, m, n, k)
    ws = workspace(ws_n)
    c, sums = torch.full((m, n), float("nan"), device="cuda"), torch.full((m,), float("nan"), device="cuda")
    call("mi355x_gemm_ex", p(c), 0, n, 0, *args, 1, None, 0, 0, p(sums), 0, 1, m, n, k, p(ws), ws_n, None)
    a, b, u = dev(A[:m]).double(), dev(B).double(), (k + 3) * 2.0 ** -23
    assert bool(((c.double() - a @ b).abs() <= u * (a.abs() @ b.abs())).all())
    assert bool(((sums.double() - a.sum(1)).abs() <= u * a.abs().sum(1)).all())
