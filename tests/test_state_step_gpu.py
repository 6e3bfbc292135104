"""One decoded token of retention, gated linear attention and latent attention: sizes at the edges of the kernels' lanes,
rows and tiles, states split over workgroups, both element types, against the CPU forms."""
import pytest
import torch

from distributed_llm_alignment_amd import ops

pytestmark = pytest.mark.gpu
EPS = 1e-5
# (B, H, dim, vdim): 16 / 32 / 64 lanes a row, a last lane group that is not full, value rows that are not a multiple of
# eight or of a pass, 128 KB states whose rows are shared, sizes below and beyond the kernel's
SIZES = [(2, 3, 32, 8), (1, 2, 36, 20), (3, 2, 64, 130), (2, 2, 100, 96), (5, 4, 128, 128), (2, 1, 132, 300), (1, 2, 252, 264),
         (2, 3, 256, 256), (1, 1, 256, 512), (2, 2, 24, 40), (1, 2, 260, 64)]


def close(got, want, dtype):
    """fp32 sums of some hundred terms in another order: a few 1e-6 of the result's norm; a bf16 result rounds by 2^-8."""
    off, size = float((got.cpu().double() - want.double()).norm()), float(want.double().norm())
    assert off <= (4e-3 if dtype == torch.bfloat16 else 2e-5) * size


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,H,dim,vdim", SIZES)
def test_retention_step(B, H, dim, vdim, dtype):
    g = torch.Generator().manual_seed(dim + vdim)
    rot = dim // 8 * 8 if dim != 100 else 40
    qkvg = torch.randn(B, 1, 2 * H * (dim + vdim), generator=g).to(dtype)
    state = torch.randn(B, H, vdim, dim, generator=g)
    d = torch.rand(H, generator=g) * 0.5 + 0.5
    decay = torch.stack([d, d.log2()])
    ang = torch.rand(64, rot // 2, generator=g) * 6.3
    start = torch.tensor([9, 0, 3, 30, 12][:B], dtype=torch.int32)
    slot = torch.tensor([33])
    args = lambda dev: (qkvg.to(dev).float() if dev == "cpu" else qkvg.to(dev), H, dim, vdim, rot, EPS, decay.to(dev),  # noqa: E731
                        state.to(dev).clone(), slot.to(dev), start.to(dev), ang.cos().to(dev), ang.sin().to(dev))
    a, b = args("cpu"), args("cuda")
    want, got = ops.retention.decode(*a, base=33), ops.retention.decode(*b, base=33)
    close(got, want, dtype)
    close(b[7], a[7], torch.float32)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rank", [16, 5])
@pytest.mark.parametrize("B,H,dim,vdim", SIZES)
def test_gla_step(B, H, dim, vdim, rank, dtype):
    g = torch.Generator().manual_seed(dim + vdim + rank)
    proj = torch.randn(B, 1, 2 * H * (dim + vdim) + rank, generator=g).to(dtype)
    a2, a2b, w = (t.to(dtype) for t in (torch.randn(H * dim, rank, generator=g) * 0.3, torch.randn(H * dim, generator=g),
                                         torch.randn(vdim, generator=g)))
    state = torch.randn(B, H, vdim, dim, generator=g)
    slot = torch.tensor([33])
    out = {}
    for dev in ("cpu", "cuda"):
        t = [x.to(dev).float() if dev == "cpu" else x.to(dev) for x in (proj, a2, a2b, w)]
        s = state.to(dev).clone()
        out[dev] = ops.gla.decode(*t, H, dim, vdim, 8.0, EPS, s, slot.to(dev), None, base=33), s
    close(out["cuda"][0], out["cpu"][0], dtype)
    close(out["cuda"][1], out["cpu"][1], torch.float32)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,H,dim,rot,vdim,R", [
    (33, 16, 128, 64, 128, 512),  # four rows a workgroup in the merge, a last group of one, two passes of query rows
    (5, 3, 64, 16, 40, 128), (2, 17, 256, 32, 32, 256),  # groups of heads that are not full, the smaller and largest tiles
    (3, 2, 24, 0, 20, 72), (2, 2, 20, 6, 33, 1000)])  # no rotated part; odd sizes, more than 512 columns
def test_latent_step(B, H, dim, rot, vdim, R, dtype):
    """bf16: queries in latent space and the result are rounded, scores and weights are not (one more 2^-8)."""
    g = torch.Generator().manual_seed(B + R)
    q = torch.randn(B, 1, H * (dim + rot), generator=g).to(dtype)
    latent = torch.randn(B, 150, R + rot, generator=g).to(dtype)
    up = (torch.randn(H * (dim + vdim), R, generator=g) * R ** -0.5).to(dtype)
    ang = torch.rand(150, rot // 2, generator=g) * 6.3
    start, slot = torch.randint(0, 60, (B,), generator=g).int(), torch.tensor([130])
    out = {}
    for dev in ("cpu", "cuda"):
        t = [x.to(dev).float() if dev == "cpu" else x.to(dev) for x in (q, latent, up)]
        out[dev] = ops.latent.decode(*t, H, dim, rot, vdim, (dim + rot) ** -0.5, 100, slot.to(dev), start.to(dev),
                                     ang.cos().to(dev), ang.sin().to(dev), base=130)
    want = out["cpu"].double()
    off = float((out["cuda"].cpu().double() - want).norm())
    assert off <= (8e-3 if dtype == torch.bfloat16 else 2e-5) * float(want.norm())
