"""LayerNorm of 16-bit rows with its statistics in the row type, through the
C ABI and through torch on the mojo device."""

import pytest
import torch
import torch.nn.functional as F

from abi import CODE, call, dev, host, p

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,cols", [(1, 768), (77, 768), (5, 3), (3, 2048), (2, 2052)])
def test_layer_norm_low_statistics(kernels, mojo, dtype, rows, cols):
    """The bits of mi355x_layer_norm_fwd with its f32 statistics rounded."""
    gen = torch.Generator().manual_seed(rows * 31 + cols)
    x, g, b = (torch.randn(*s, generator=gen).to(dtype) for s in ((rows, cols), (cols,), (cols,)))
    tx, tg, tb = dev(x), dev(g), dev(b)
    y, y2 = (torch.empty(rows, cols, dtype=dtype, device="cuda") for _ in range(2))
    mean, rstd = (torch.empty(rows, device="cuda") for _ in range(2))
    mean2, rstd2 = (torch.empty(rows, dtype=dtype, device="cuda") for _ in range(2))
    call("mi355x_layer_norm_fwd", p(y), p(mean), p(rstd), p(tx), p(tg), p(tb), rows, cols, 1e-5, CODE[dtype], None)
    call("mi355x_layer_norm_fwd_low", p(y2), p(mean2), p(rstd2), p(tx), p(tg), p(tb), rows, cols, 1e-5, CODE[dtype],
         None)
    assert torch.equal(host(y), host(y2))
    assert torch.equal(host(mean).to(dtype), host(mean2)) and torch.equal(host(rstd).to(dtype), host(rstd2))
    out, m, r = torch.native_layer_norm(x.to("mojo"), (cols,), g.to("mojo"), b.to("mojo"), 1e-5)
    assert m.dtype == r.dtype == dtype and m.shape == (rows, 1)
    assert torch.equal(out.cpu(), host(y)) and torch.equal(r.cpu().flatten(), host(rstd2))
    assert torch.equal(F.layer_norm(x.to("mojo"), (cols,)).cpu().isfinite(), torch.ones(rows, cols).bool())
