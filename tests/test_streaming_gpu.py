"""Edges of the streaming kernels: sizes around one workgroup's share, odd row lengths and strides."""
import pytest
import torch

from distributed_llm_alignment_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("n", [8, 1016, 1024, 1032, 256 * 1024 + 8])
@pytest.mark.parametrize("grad_dtype", [torch.bfloat16, torch.float32])
def test_adamw_sizes(n, grad_dtype):
    """Every parameter of a flat buffer is updated once, none past its end (float64 reference; the bound is
    a few roundings of the fp32 state)."""
    from distributed_llm_alignment_amd.optim.adamw import adamw_update

    g0 = torch.Generator().manual_seed(n)
    guard = 64
    state = {k: torch.randn(n + guard, generator=g0).to(DEV) for k in ("w", "m", "v")}
    state["v"] = state["v"].abs()
    grad = torch.randn(n, generator=g0).to(DEV, grad_dtype)
    p = torch.zeros(n + guard, device=DEV, dtype=torch.bfloat16)
    want = {k: t.double().clone() for k, t in state.items()}
    adamw_update(p[:n], state["w"][:n], grad, state["m"][:n], state["v"][:n], 1e-2, 0.9, 0.95, 1e-8, 0.01, 3)
    w, m, v = (want[k][:n] for k in ("w", "m", "v"))
    g = grad.double()
    w.mul_(1 - 1e-2 * 0.01)
    m.mul_(0.9).add_(0.1 * g)
    v.mul_(0.95).add_(0.05 * g * g)
    w.sub_(1e-2 / (1 - 0.9 ** 3) * m / (v.sqrt() / (1 - 0.95 ** 3) ** 0.5 + 1e-8))
    for k in want:
        torch.testing.assert_close(state[k].double(), want[k], rtol=2e-6, atol=2e-6)
    assert torch.equal(p[:n], state["w"][:n].bfloat16()) and not p[n:].any()


@pytest.mark.parametrize("V,ld", [(8, 8), (1, 8), (777, 784), (2051, 2112), (2048, 2048), (50257, 50304), (777, 777), (1000, 1001)])
def test_logprob_row_ends(V, ld):
    """Rows with a padded stride, a vocabulary that is not a multiple of a piece, and unaligned rows: log-probabilities and
    in-place gradients against float64 (fp32 sums; the bf16 gradient rounds by 2^-8), the padding left alone."""
    from distributed_llm_alignment_amd.ops import _ext

    g0 = torch.Generator(device=DEV).manual_seed(V)
    N = 33
    buf = (torch.randn(N, ld, generator=g0, device=DEV) * 3).bfloat16()
    x, pad = buf[:, :V], buf[:, V:].clone()
    z = x.double()
    tgt = torch.randint(0, V, (N,), generator=g0, device=DEV)
    tgt[3], tgt[4], tgt[5] = -100, V - 1, 0
    gr = torch.randn(N, generator=g0, device=DEV)
    lp, lse = _ext.require().logprob_fwd(x, tgt)
    want = torch.where(tgt >= 0, torch.log_softmax(z, -1).gather(1, tgt.clamp(min=0)[:, None])[:, 0], 0)
    torch.testing.assert_close(lse.double(), torch.logsumexp(z, -1), rtol=1e-5, atol=1e-5)
    torch.testing.assert_close(lp.double(), want, rtol=1e-5, atol=2e-5)
    _ext.require().logprob_bwd(x, tgt, lse, gr)
    hot = torch.nn.functional.one_hot(tgt.clamp(min=0), V).double()
    dz = (gr * (tgt >= 0)).double()[:, None] * (hot - z.softmax(-1))
    assert float((x.double() - dz).norm()) <= 4e-3 * float(dz.norm()) + 1e-12
    assert torch.equal(buf[:, V:], pad)


@pytest.mark.parametrize("V", [97, 8191, 8193, 8200])
def test_linear_logprob_padded_rows(V):
    """The LM head over vocabularies that need padded rows and ones that do not, gradients included (float64; bf16 products)."""
    g0 = torch.Generator(device=DEV).manual_seed(V)
    h = torch.randn(40, 64, generator=g0, device=DEV).bfloat16().requires_grad_()
    w = (torch.randn(V, 64, generator=g0, device=DEV) * 0.2).bfloat16().requires_grad_()
    tgt, gr = torch.randint(0, V, (40,), generator=g0, device=DEV), torch.randn(40, generator=g0, device=DEV)
    (ops.linear_logprob(h, w, tgt) * gr).sum().backward()
    hd, wd = h.detach().double().requires_grad_(), w.detach().double().requires_grad_()
    lp = torch.log_softmax(hd @ wd.T, -1).gather(1, tgt[:, None])[:, 0]
    (lp * gr).sum().backward()
    with torch.no_grad():
        got = ops.linear_logprob(h, w, tgt)
    assert float((got.double() - lp).norm()) <= 8e-3 * float(lp.norm())
    for a, b in ((h, hd), (w, wd)):
        assert float((a.grad.double() - b.grad).norm()) <= 2e-2 * float(b.grad.norm())


@pytest.mark.parametrize("N,H", [(1, 8), (16, 8), (17, 520), (33, 512), (4100, 768)])
@pytest.mark.parametrize("gdtype", [torch.bfloat16, torch.float32])
def test_embedding_runs(N, H, gdtype):
    """Runs of every length and place (one id, no repeats, the pad id over most positions, invalid ids at both ends) into a
    gradient that holds something already: float64 sums; fp32 over a run (n * 2^-24 relative), bf16 rounds once (2^-8)."""
    from distributed_llm_alignment_amd.ops import _ext

    V = 97
    g0 = torch.Generator(device=DEV).manual_seed(N + H)
    for case in range(4):
        ids = torch.randint(0, V, (N,), generator=g0, device=DEV)
        if case == 0:
            ids.fill_(V - 1)
        elif case == 1:
            ids = torch.arange(N, device=DEV) * V // max(N, V)
        elif case == 2:
            ids[torch.rand(N, generator=g0, device=DEV) < 0.8] = 3
        else:
            ids[: N // 3] = -1
            ids[N - N // 4:] = V
        dy = torch.randn(N, H, generator=g0, device=DEV).bfloat16()
        grad = torch.randn(V, H, generator=g0, device=DEV).to(gdtype)
        ok = (ids >= 0) & (ids < V)
        want = grad.double().index_add(0, ids[ok], dy[ok].double())
        sid, perm = torch.sort(ids, stable=True)
        _ext.require().embed_bwd(sid, perm, dy, grad)
        size = grad.double().abs().index_add(0, ids[ok], dy[ok].double().abs())
        tol = (2 ** -8 if gdtype == torch.bfloat16 else 0) * want.abs() + N * 2 ** -24 * size
        assert bool(((grad.double() - want).abs() <= tol).all()), case


@pytest.mark.parametrize("M,N,pad", [(1, 8, 0), (7, 256, 0), (33, 264, 8), (1000, 768, 0), (8000, 2304, 0), (4097, 3072, 16)])
def test_column_sum(M, N, pad):
    """Bias gradients over row and column remainders and a padded stride, against float64: fp32 sums (M * 2^-24 of the sum of
    sizes at most) and one bf16 rounding; a stride the kernel does not take gives the same."""
    from distributed_llm_alignment_amd.ops.linear import bias_grad

    g0 = torch.Generator(device=DEV).manual_seed(M + N)
    x = torch.randn(M, N + pad, generator=g0, device=DEV).bfloat16()[:, :N]
    want, size = x.double().sum(0), x.double().abs().sum(0)
    odd = torch.empty(M, N + pad + 1, dtype=x.dtype, device=DEV)[:, :N].copy_(x)
    for y in (x, odd):
        assert bool(((bias_grad(y).double() - want).abs() <= 2 ** -8 * want.abs() + M * 2 ** -24 * size).all())


@pytest.mark.parametrize("rows,H", [(1, 8), (3, 512), (5, 520), (2049, 768), (4100, 1024), (770, 1032)])
@pytest.mark.parametrize("rms,dres", [(True, True), (True, False), (False, True), (False, False)])
def test_norm_backward_narrow_rows(rows, H, rms, dres):
    """A wave per row up to 1024 columns, a block per row above: against float64, ds rounds once (2^-8), dw / db add fp32
    terms of every row (rows * 2^-24 of their sizes) and round once."""
    from distributed_llm_alignment_amd.ops import _ext

    g0 = torch.Generator(device=DEV).manual_seed(rows + H)

    def r(*s):
        return torch.randn(*s, generator=g0, device=DEV).bfloat16()

    s, dy, w, add = r(rows, H), r(rows, H), r(H), (r(rows, H) if dres else None)
    sd, dyd, wd = s.double(), dy.double(), w.double()
    mean = torch.zeros(rows, 1, device=DEV, dtype=torch.float64) if rms else sd.mean(1, keepdim=True)
    rstd = ((sd - mean).pow(2).mean(1, keepdim=True) + 1e-5).rsqrt()
    ds, dw, db = _ext.require().norm_bwd(dy, s, w, rstd.float().view(-1), None if rms else mean.float().view(-1), add, not rms, rms)
    xh, g = (sd - mean) * rstd, dyd * wd
    want = (g - xh * (g * xh).mean(1, keepdim=True) - (0 if rms else g.mean(1, keepdim=True))) * rstd
    size = want.abs().amax() if want.numel() else 0
    if dres:
        want = want + add.double()
    assert bool(((ds.double() - want).abs() <= 2 ** -8 * want.abs() + 1e-5 * size + 1e-6).all())
    for have, term in ((dw, dyd * xh), (db, dyd)):
        if have.numel():
            t = term.sum(0)
            assert bool(((have.double() - t).abs() <= 2 ** -8 * t.abs() + (rows + 16) * 2 ** -23 * term.abs().sum(0)).all())
