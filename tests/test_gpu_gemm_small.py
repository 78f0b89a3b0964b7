"""The 64x64 GEMM tiles (outputs too small to fill the CUs with larger ones),
through the C ABI, against 64-bit results."""

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
