"""The captured token step around the model: the row-split draw against the single-block one, the bookkeeping after it and
the cache position, against their forms in separate torch operations."""
import pytest
import torch

from distributed_llm_alignment_amd.ops import decode

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("V", [32768, 32776, 50304, 128256])
@pytest.mark.parametrize("top_k,top_p", [(0, 1.0), (0, 0.9), (40, 1.0), (40, 0.8), (7, 0.5)])
def test_split_draw_equals_single_block(V, top_k, top_p):
    """Rows with an odd stride take the single-block kernel: same thresholds, same random number. The two add the kept
    masses in different orders, so their running sums differ by some 2^-22 of the total, and a draw differs where it falls
    that close to the edge between two tokens: with `kept` edges, at most kept * 2 * 2^-22 of the draws."""
    g = torch.Generator(device=DEV).manual_seed(V + top_k)
    rows = 64
    logits = (torch.randn(rows, V, device=DEV, generator=g) * 3).bfloat16()
    logits[1] = -100.0  # one token holds the row
    logits[1, V - 1] = 5.0
    logits[2] = 1.0  # all equal
    odd = torch.empty(rows, V + 1, device=DEV, dtype=torch.bfloat16)[:, :V]
    odd.copy_(logits)
    differ = 0
    for step in range(16):
        rng = torch.tensor([9, step], dtype=torch.long, device=DEV)
        a, b = (decode.sample_tokens(x, 0.7, top_k, top_p, False, rng) for x in (logits, odd))
        differ += int((a != b).sum())
        assert int(a[1]) == V - 1
    assert differ <= 1 + 16 * rows * (top_k or V) * 2 ** -21


@pytest.mark.parametrize("rows", [1, 3, 256, 1000])
@pytest.mark.parametrize("eos,pad", [(5, 0), (5, 5), (None, 2), (-1, 0)])
def test_token_step(rows, eos, pad):
    g = torch.Generator().manual_seed(rows)
    cols = 4

    def state(dev):
        return (torch.zeros(rows, dtype=torch.bool, device=dev), torch.zeros((rows, 1), dtype=torch.long, device=dev),
                torch.full((rows, cols), pad, dtype=torch.long, device=dev), torch.zeros((rows, cols), dtype=torch.long, device=dev),
                torch.zeros(1, dtype=torch.long, device=dev), torch.tensor([7, 0], dtype=torch.long, device=dev))

    have, want = state(DEV), state("cpu")
    for _ in range(cols):
        nxt = torch.randint(0, 8, (rows,), generator=g)
        decode.token_step(nxt.to(DEV), *have, eos, pad)
        decode.token_step(nxt, *want, eos, pad)
        for a, b in zip(have, want):
            assert torch.equal(a.cpu(), b)
    before = [t.clone() for t in have[2:4]]
    decode.token_step(nxt.to(DEV), *have, eos, pad)  # past the last column: nothing is written there
    assert all(torch.equal(a, b) for a, b in zip(before, have[2:4]))


@pytest.mark.parametrize("rows", [1, 256, 257])
def test_kv_advance(rows):
    slot, n, pos = (torch.full((k,), 3, dtype=t, device=DEV) for k, t in ((1, torch.long), (1, torch.int32), (rows, torch.int32)))
    for _ in range(2):
        decode.kv_advance(slot, n, pos.view(-1, 1))
    assert int(slot) == 5 and int(n) == 5 and bool((pos == 5).all())
