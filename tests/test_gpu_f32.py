"""The f32 kernels on matrix cores, through the C ABI, against 64-bit results."""

import pytest
import torch

from abi import bhs, call, dev, host, lib, p, workspace

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


@pytest.mark.parametrize("layout", ["NT", "NN", "TN", "TT"])
@pytest.mark.parametrize("m,n,k,batch", [(130, 3000, 8, 1), (1000, 1090, 16, 7), (1000, 1090, 16, 8), (1000, 1090, 17, 1),
                                         (161, 9000, 9, 6), (160, 9000, 9, 6), (3, 24577, 48, 2), (3, 24577, 49, 2),
                                         (16, 24577, 80, 2), (49160, 17, 48, 1), (1000, 1090, 64, 1), (3000, 1500, 40, 1)])
def test_gemm_f32_short_k(kernels, layout, m, n, k, batch):
    """The FMA kernel and the matrix cores on both sides of each line between them,
    into rows of C at every alignment (an odd stride, a base shifted by one
    element) with bias: nothing else is written.  A chain of k products is within
    (k + 2) * 2^-24 of sum |a||b| + |bias|."""
    gen = torch.Generator().manual_seed(m + n + k)
    A, B, bias = (torch.randn(*x, generator=gen) for x in ((batch, m, k), (batch, k, n), (n,)))
    ta = dev((A.transpose(1, 2) if layout[0] == "T" else A).contiguous())
    tb = dev((B.transpose(1, 2) if layout[1] == "T" else B).contiguous())
    a_rs, a_cs = (k, 1) if layout[0] == "N" else (1, m)
    b_rs, b_cs = (n, 1) if layout[1] == "N" else (1, k)
    args, tbias, ld = (p(ta), a_rs, a_cs, m * k, p(tb), b_rs, b_cs, k * n, 0), dev(bias), n + 3 + n % 2
    ws_n = lib().mi355x_gemm_workspace_bytes(*args, batch, m, n, k)
    ws, store = workspace(ws_n) if ws_n else None, torch.full((1 + batch * m * ld,), 3.0, device="cuda")
    call("mi355x_gemm", p(store) + 4, 0, ld, m * ld, *args, p(tbias), 0, 0, batch, m, n, k, p(ws), ws_n, None)
    got = store[1:].view(batch, m, ld)
    assert float(store[0]) == 3.0 and bool((got[..., n:] == 3.0).all())
    for i in range(batch):
        a, b = dev(A[i]).double(), dev(B[i]).double()
        bound = (k + 2) * 2.0 ** -24 * (a.abs() @ b.abs() + tbias.double().abs())
        assert bool(((got[i, :, :n].double() - (a @ b + tbias.double())).abs() <= bound).all())


def _attention_bounds(q, k, v, do, causal, scale):
    """(O, LSE, dQ, dK, dV) in 64 bits, and what f32 sums and products may be
    off by: u = 2^-24; a score D + 4 roundings of sum |q||k|, a probability
    twice the row's largest such error and 8 u for exp2 and the
    normalisation, sums of n terms n + 3 roundings of their absolute sum."""
    u, d, n, m = 2.0 ** -24, q.shape[-1], k.shape[-2], q.shape[-2]
    s, sa = q @ k.transpose(-2, -1) * scale, q.abs() @ k.abs().transpose(-2, -1) * scale
    if causal:
        keep = torch.arange(n)[None, :] <= torch.arange(m)[:, None]
        s, sa = s.masked_fill(~keep, float("-inf")), sa.masked_fill(~keep, 0.0)
    es = (d + 4) * u * sa.amax(-1, keepdim=True)
    pr = torch.softmax(s, -1)
    rel = 2 * es + 8 * u
    o, oa = pr @ v, pr @ v.abs()
    eo = (rel + (n + 8) * u) * oa
    lse = torch.logsumexp(s, -1)
    el = es[..., 0] + (n + 8) * u + 8 * u * lse.abs()
    dp, dpa = do @ v.transpose(-2, -1), do.abs() @ v.abs().transpose(-2, -1)
    di, dia = (do * o).sum(-1, keepdim=True), (do * o).abs().sum(-1, keepdim=True)
    ds = pr * (dp - di)
    edi = (d + 4) * u * dia + (do.abs() * eo).sum(-1, keepdim=True)
    relp = rel + el[..., None]
    eds = pr * ((relp + 8 * u) * (dp - di).abs() + (d + 8) * u * dpa + edi + 8 * u * (dp.abs() + di.abs()))
    t = lambda x: x.transpose(-2, -1)  # noqa: E731
    out = {"o": (o, eo), "lse": (lse, el),
           "dq": (scale * (ds @ k), scale * ((eds + (n + 8) * u * ds.abs()) @ k.abs())),
           "dk": (scale * (t(ds) @ q), scale * (t(eds + (m + 8) * u * ds.abs()) @ q.abs())),
           "dv": (t(pr) @ do, t((relp + (m + 8) * u) * pr) @ do.abs())}
    return out


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("sq,skv,layout", [(1, 1, "bhsd"), (16, 17, "bshd"), (33, 33, "bshd"), (63, 65, "bhsd"),
                                           (100, 40, "bshd"), (40, 130, "bshd"), (255, 255, "split"),
                                           (256, 256, "split"), (70, 70, "odd")])
def test_attention_f32_matrix_cores(kernels, d, causal, sq, skv, layout):
    """f32 attention at the edges of its 16-row waves, 32-row tiles and 64-row
    blocks, more keys than queries and fewer, rows inside a fused projection,
    and ("odd") rows that are not 16-byte aligned, which the general kernels
    take."""
    B, H, scale = 2, 3, 0.3 / d ** 0.5 * 3
    gen = torch.Generator().manual_seed(d * 1000 + sq * 7 + skv)
    q, do = (torch.randn(B, H, sq, d, generator=gen) for _ in range(2))
    k, v = (torch.randn(B, H, skv, d, generator=gen) for _ in range(2))

    def store(x, pad):
        if layout == "bhsd":
            return dev(x)
        t = torch.zeros(x.shape[0], x.shape[2], x.shape[1] * d + pad, device="cuda")
        w = t[..., : x.shape[1] * d].unflatten(-1, (x.shape[1], d)).transpose(1, 2)
        w.copy_(x)
        return w

    pad = {"split": 2 * H * d, "odd": 1}.get(layout, 0)
    tq, tk, tv, tdo = (store(x, pad) for x in (q, k, v, do))
    o, dq = (store(torch.zeros_like(q), pad) for _ in range(2))
    dk, dv = (store(torch.zeros_like(k), pad) for _ in range(2))
    lse = torch.empty(B, H, sq, device="cuda")
    call("mi355x_attn_fwd_gen", p(o), bhs(o), p(lse), p(tq), bhs(tq), p(tk), bhs(tk), p(tv), bhs(tv), B, H, H, sq, skv,
         d, scale, int(causal), 0, 0, None)
    ws_n = lib().mi355x_attn_bwd_gen_workspace_bytes(B, H, H, sq, skv, d)
    ws = workspace(ws_n)
    call("mi355x_attn_bwd_gen", p(dq), bhs(dq), p(dk), bhs(dk), p(dv), bhs(dv), p(tdo), bhs(tdo), p(tq), bhs(tq),
         p(tk), bhs(tk), p(tv), bhs(tv), p(o), bhs(o), p(lse), B, H, H, sq, skv, d, scale, int(causal), 0, 0, p(ws),
         ws_n, None)
    want = _attention_bounds(*(x.double() for x in (q, k, v, do)), causal, scale)
    for name, got in (("o", o), ("lse", lse), ("dq", dq), ("dk", dk), ("dv", dv)):
        ref, bound = want[name]
        err = (host(got).double() - ref).abs()
        assert bool((err <= bound).all()), (name, float((err / bound.clamp_min(1e-300)).max()))


@pytest.mark.parametrize("d", [32, 64, 128])
def test_attention_f32_scores_are_partial_sums(kernels, d):
    """A score's rounding error is that of eight partial sums (four at head_dim
    32) added in a tree, not of one chain.  With one key LSE is the score; its
    terms are positive, so a rounding of a partial sum that holds a share x of
    the score is off by at most u x (u = 2^-24; by u x / sqrt(3) in the root
    mean square).  Partial sums of d / 8 terms and the tree have shares whose
    squares sum to 2.4 (the factor to natural logarithms adds 1, the operand's
    scaling next to nothing): 1.1 u.  One chain of d terms has d / 3 more, 1.9 u
    (d = 32) to 3.8 u."""
    n = 8192
    gen = torch.Generator().manual_seed(d)
    q, k = 1 + torch.rand(1, 1, n, d, generator=gen), 1 + torch.rand(1, 1, 1, d, generator=gen)
    tq, tk, o, lse = dev(q), dev(k), torch.empty(1, 1, n, d, device="cuda"), torch.empty(1, 1, n, device="cuda")
    call("mi355x_attn_fwd_gen", p(o), bhs(o), p(lse), p(tq), bhs(tq), p(tk), bhs(tk), p(tk), bhs(tk), 1, 1, 1, n, 1, d, 1.0,
         0, 0, 0, None)
    log2e, ln2 = (torch.tensor(x, dtype=torch.float64).float().double() for x in (1.4426950408889634, 0.6931471805599453))
    exact = (q.double() * k.double()).sum(-1) * (log2e * ln2)
    rms = float(((host(lse).double() - exact) / exact).square().mean().sqrt()) * 2.0 ** 24
    assert rms <= 1.1, rms


@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("sq,skv,causal", [(1, 1, 1), (3, 1, 0), (40, 200, 1), (70, 70, 1)])
def test_attention_f32_one_key_has_no_gradient(kernels, d, sq, skv, causal):
    """A query that sees one key gives it all its weight, whatever Q and K are: its
    output is that key's V and its dQ exactly zero (D is summed as dP is), and so is
    dK where no query sees two keys."""
    B, H = 2, 3
    gen = torch.Generator().manual_seed(d + sq)
    q, do, k, v = (dev(torch.randn(B, H, n, d, generator=gen)) for n in (sq, sq, skv, skv))
    o, dq, dk, dv, lse = (torch.full_like(x, float("nan")) for x in (q, q, k, v, q[..., 0]))
    call("mi355x_attn_fwd_gen", p(o), bhs(o), p(lse), p(q), bhs(q), p(k), bhs(k), p(v), bhs(v), B, H, H, sq, skv, d, d ** -0.5,
         causal, 0, 0, None)
    ws_n = lib().mi355x_attn_bwd_gen_workspace_bytes(B, H, H, sq, skv, d)
    ws = workspace(ws_n)
    call("mi355x_attn_bwd_gen", p(dq), bhs(dq), p(dk), bhs(dk), p(dv), bhs(dv), p(do), bhs(do), p(q), bhs(q), p(k), bhs(k),
         p(v), bhs(v), p(o), bhs(o), p(lse), B, H, H, sq, skv, d, d ** -0.5, causal, 0, 0, p(ws), ws_n, None)
    rows = slice(None) if skv == 1 else slice(1)
    assert torch.equal(o[:, :, rows], v[:, :, :1].expand_as(o[:, :, rows])) and not dq[:, :, rows].any()
    assert skv > 1 or not dk.any()


def test_attention_f32_heads_past_one_grid_dimension(kernels):
    """2^24 blocks of the matrix-core kernels are more threads than one dimension of
    a launch takes: such calls stay on the general kernels.  With one key O is V, and
    dV is dO but for the probability, exp2 of a score (8.2 at most) less itself through
    LSE and back: 4 roundings, u = 2^-24 of 8.2 ln 2 each, and exp2's."""
    B, H, d = 65535, 257, 32
    q, k, v, do, o, dq, dk, dv = (torch.empty(B, H, 1, d, device="cuda") for _ in range(8))
    for x in (q, k, v, do):
        x.uniform_(-1, 1)
    lse = torch.empty(B, H, 1, device="cuda")
    call("mi355x_attn_fwd_gen", p(o), bhs(o), p(lse), p(q), bhs(q), p(k), bhs(k), p(v), bhs(v), B, H, H, 1, 1, d, d ** -0.5,
         0, 0, 0, None)
    assert torch.equal(o, v)
    ws_n = lib().mi355x_attn_bwd_gen_workspace_bytes(B, H, H, 1, 1, d)
    ws = workspace(ws_n)
    call("mi355x_attn_bwd_gen", p(dq), bhs(dq), p(dk), bhs(dk), p(dv), bhs(dv), p(do), bhs(do), p(q), bhs(q), p(k), bhs(k),
         p(v), bhs(v), p(o), bhs(o), p(lse), B, H, H, 1, 1, d, d ** -0.5, 0, 0, 0, p(ws), ws_n, None)
    assert bool(((dv - do).abs() <= 26 * 2.0 ** -24 * do.abs()).all()) and not dq.any() and not dk.any()


def test_attention_f32_infinities_and_nan(kernels, mojo):
    """A NaN or infinite element of Q shows in its own query's row alone; one of V
    in every query's that sees its key, and, the probabilities of keys out of sight
    being zeros in the same product, in earlier queries' that share its 32-key tile
    (from row 32 here, whose V element lies at 40): in no others, and in no other
    column."""
    gen = torch.Generator().manual_seed(5)
    for bad in (float("nan"), float("inf")):
        q, k, v = (torch.randn(1, 2, 70, 64, generator=gen) for _ in range(3))
        q[0, 0, 7, 3] = bad
        v[0, 1, 40, 5] = bad
        got = torch.nn.functional.scaled_dot_product_attention(q.to("mojo"), k.to("mojo"), v.to("mojo"), is_causal=True)
        got = got.cpu()
        assert got[0, 0, 7].isnan().all() and got[0, 0, 8:].isfinite().all() and got[0, 0, :7].isfinite().all()
        assert not got[0, 1, 40:, 5].isfinite().any() and got[0, 1, :32].isfinite().all()
        others = torch.arange(64) != 5
        assert got[0, 1][:, others].isfinite().all()
