"""Edges of the streaming kernels: sizes around one workgroup's share, odd row lengths and strides."""
import pytest
import torch

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
