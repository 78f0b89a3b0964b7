"""The f32 kernels on matrix cores, through the C ABI, against 64-bit results."""

import pytest
import torch

from abi import call, dev, host, lib, p, workspace

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["NT", "NN", "TN", "TT"])
@pytest.mark.parametrize("m,n,k,batch,shift", [(1, 1, 1, 1, 0), (5, 3, 31, 2, 0), (64, 64, 32, 1, 0), (65, 129, 33, 1, 0),
                                               (128, 128, 64, 1, 1), (130, 68, 100, 3, 0), (96, 100, 4100, 1, 0),
                                               (260, 2052, 36, 1, 0), (3000, 2900, 8, 1, 0)])
def test_gemm_f32_tiles_and_splits(kernels, layout, m, n, k, batch, shift):
    """f32 GEMM at the edges of its 64 and 128 tiles, its 32-k stages and its K
    splits, 4- and 16-byte loads (odd strides, a base shifted by one element),
    with bias and beta, and without the workspace that its splits use.  A
    chain of k FMAs and the partial sums are within (k + 3) * 2^-24 of
    sum |a||b| + |bias| + |C|."""
    gen = torch.Generator().manual_seed(m * 7919 + n * 31 + k)
    A, B, C0 = (torch.randn(batch, *s, generator=gen) for s in ((m, k), (k, n), (m, n)))
    bias = torch.randn(n, generator=gen)

    def store(x, transposed):
        x = (x.transpose(1, 2) if transposed else x).contiguous()
        t = dev(torch.cat([torch.zeros(shift), x.reshape(-1)]))
        return t[shift:]

    ta, tb, tbias = store(A, layout[0] == "T"), store(B, layout[1] == "T"), dev(bias)
    a_rs, a_cs = (k, 1) if layout[0] == "N" else (1, m)
    b_rs, b_cs = (n, 1) if layout[1] == "N" else (1, k)
    need = lib().mi355x_gemm_workspace_bytes(p(ta), a_rs, a_cs, m * k, p(tb), b_rs, b_cs, k * n, 0, batch, m, n, k)
    exp = A.double() @ B.double() + bias.double() + C0.double()
    bound = (k + 3) * 2.0 ** -24 * (A.double().abs() @ B.double().abs() + bias.double().abs() + C0.double().abs())
    for ws_n in {need, 0}:
        tc, ws = dev(C0), workspace(ws_n) if ws_n else None
        call("mi355x_gemm", p(tc), 0, n, m * n, p(ta), a_rs, a_cs, m * k, p(tb), b_rs, b_cs, k * n, 0, p(tbias), 0,
             1, batch, m, n, k, p(ws), ws_n, None)
        err = (host(tc).double() - exp).abs()
        assert bool((err <= bound).all()), (ws_n, float((err / bound).max()))
