"""Row movement on both sides of the size at which the sorted rows pass through the caches
without being kept (176 MB), and on both sides of 8 and 16 experts a token, where the kernels
hold positions and scores differently: permute and combine with their backward equal, bit for
bit, the same sums taken in torch, row by row in sorted order with each rounding."""

import pytest
import torch

from tests.conftest import banner

pytestmark = pytest.mark.gpu

# (tokens, dim, experts, top_k, dtype): up to 187 MB of sorted rows
CASES = [(37, 8, 8, 1, torch.bfloat16), (100, 520, 16, 8, torch.bfloat16), (61, 264, 32, 9, torch.float32),
         (300, 1000, 32, 17, torch.bfloat16), (5600, 2048, 64, 8, torch.bfloat16), (5700, 2048, 64, 8, torch.bfloat16),
         (5640, 1024, 16, 8, torch.float32), (5600, 1024, 16, 8, torch.float32)]


@pytest.mark.parametrize("scored", [True, False], ids=["scored", "plain"])
@pytest.mark.parametrize("n,d,e,k,dtype", CASES)
def test_rows_equal_torch(dev, n, d, e, k, dtype, scored):
    banner(f"rows {n}x{k}x{d} {dtype} scored {scored}")
    from torchtitan_amd import ops

    gen = torch.Generator(device=dev).manual_seed(n + d)
    idx = torch.rand(n, e, device=dev, generator=gen).topk(k).indices
    top = torch.rand(n, k, device=dev, generator=gen)
    scores, token_idx, _counts, _offs, slot_pos, tok_pos = ops.reorder(top, idx, e)
    x, shared, go = (torch.randn(n, d, device=dev, generator=gen).to(dtype) for _ in range(3))
    rows = torch.randn(n * k, d, device=dev, generator=gen).to(dtype)
    s = scores if scored else None

    def scaled(r, pos):
        return (r.float() * scores[pos][:, None]).to(dtype) if scored else r

    assert torch.equal(ops.permute(x, slot_pos, tok_pos, s), scaled(x[token_idx], slice(None)))

    acc, grad_x = shared, torch.zeros_like(x)
    for j in range(k):
        pos = tok_pos[:, j].long()
        acc = acc + scaled(rows[pos], pos)
        grad_x = grad_x + scaled(rows[pos], pos)
    assert torch.equal(ops.combine(shared, rows, slot_pos, tok_pos, s), acc)
    got_x, got_s = ops.permute_backward(rows, x, tok_pos, s, True)
    assert torch.equal(got_x, grad_x)
    got_r, got_cs = ops.combine_backward(go, rows, slot_pos, tok_pos, s)
    want_r = scaled(go[token_idx], slice(None))
    assert torch.equal(got_r, want_r)
    if scored:  # fp32 sums of d products in another order: d rounding steps of the sum of magnitudes
        for got, other in ((got_s, x[token_idx]), (got_cs, go[token_idx])):
            p = rows.double() * other.double()
            assert ((got.double() - p.sum(1)).abs() <= d * 2.0 ** -24 * p.abs().sum(1)).all()
