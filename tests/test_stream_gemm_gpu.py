"""Decode projections on the fp32 stream: every tile of the dispatch, its edges, every epilogue, against float64."""
import pytest
import torch

from distributed_llm_alignment_amd.ops import _ext
from distributed_llm_alignment_amd.ops import stream as st

pytestmark = pytest.mark.gpu
DEV, EPS = "cuda", 1e-3


def close(got, want, what):
    """A bf16 result has 8 bits: it is off by at most 2^-8 = 3.9e-3 of itself, so is a vector of them; the fp32 sum
    before it by a few 1e-6; fp32 results by the latter."""
    got, want = got.double().reshape(want.shape), want.double()
    off, size = float((got - want).norm()), float(want.norm())
    assert off <= (4e-3 if what != "fp32" else 2e-5) * size, (what, off, size)


def silu_like(z):
    return torch.nn.functional.gelu(z, approximate="tanh")


# (N, K): 8 columns (one stage and less, ragged K), 16, 16 deep, 32 and 64 columns per workgroup, weights under and over 8 MB
@pytest.mark.parametrize("N,K", [(8, 8), (40, 72), (200, 2056), (2044, 2304), (72, 8200), (2100, 200), (5124, 264), (16388, 136)])
@pytest.mark.parametrize("M", [1, 8, 9, 16, 17, 32, 33, 48, 49, 64])
def test_projection_tiles(M, N, K):
    g = torch.Generator(device=DEV).manual_seed(1000 * M + N)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)  # noqa: E731
    a, w = rnd(M, K).bfloat16(), (rnd(N, K) * K ** -0.5).bfloat16()
    gated = (rnd(2 * N, K) * K ** -0.5).bfloat16()
    nw, b, rw = (rnd(N).bfloat16() for _ in range(3))
    ids = torch.randint(0, 50, (M, 1), generator=g, device=DEV)
    if M > 1:
        ids[M // 2] = 77  # outside the table: its row is zero
    table = rnd(50, N + 24).bfloat16()
    ssq = rnd(M, 300).square()  # partial sums of squares, more than one load of them per lane
    scale = torch.rsqrt(ssq.double().sum(1, keepdim=True) / K + EPS)
    z, zg = a.double() @ w.double().T, a.double() @ gated.double().T
    close(st.fused_linear(a, w), z, "store")
    close(st.fused_linear(a, w, ssq, EPS, relu2=True), torch.relu(z * scale) ** 2, "relu2")
    close(st.fused_geglu(a, gated, ssq, EPS), silu_like(zg[:, :N] * scale) * (zg[:, N:] * scale), "geglu")
    rows = table.double()[ids[:, 0].clamp(max=49), 16:16 + N] * (ids < 50)
    close(st.fused_gate(a, w, ids, table, 16), silu_like(z) * rows, "gate")
    close(_ext.require("mix").stream_gemm_cap(a, w, 5.0), 5 * torch.tanh(z / 5), "fp32")
    x = rnd(M, N)
    want = x.double() + z
    y, sq = st.fused_add(a, w, x, nw, 1.0)
    close(x, want, "fp32")
    close(y, want * (1 + nw.double()), "stream rows")
    close(sq.sum(1), want.square().sum(1), "fp32")
    x, rs = rnd(M, N), rnd(M, 5).square()
    want = 1.5 * x.double() * torch.rsqrt(rs.double().sum(1, keepdim=True) / N + EPS) * rw.double() + z + b.double()
    y, sq = st.fused_post(a, w, x, 1.5, b, rs, rw, nw, EPS)
    close(x, want, "fp32")
    close(y, want * nw.double(), "post rows")
    close(sq.sum(1), want.square().sum(1), "fp32")


def test_rows_do_not_mix():
    """A row of NaN reaches its own outputs only, also where a row tile is not full."""
    for M in (3, 11, 20, 40, 60):
        a, w = torch.ones(M, 256, device=DEV).bfloat16(), torch.ones(48, 256, device=DEV).bfloat16()
        a[M - 1] = float("nan")
        y = st.fused_linear(a, w)
        assert torch.equal(y[: M - 1], torch.full_like(y[: M - 1], 256.0)) and bool(y[M - 1].isnan().all())
