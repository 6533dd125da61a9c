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
         (5640, 1024, 16, 8, torch.float32), (5600, 1024, 16, 8, torch.float32),
         (50, 264, 32, 12, torch.bfloat16), (3072, 72, 32, 16, torch.bfloat16), (3073, 72, 32, 16, torch.bfloat16)]


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


def test_small_combine_keeps_its_rows(dev):
    """Below the streaming size the combine leaves its rows in the caches, where a scored
    backward that follows at once (a recomputed layer) finds them: it takes about as long as
    when its rows were just read by the backward itself. With rows read past the caches it
    took 1.5 times as long at this size (59 MB of rows)."""
    from torchtitan_amd import ops

    n, d, e, k = 512, 7168, 64, 8
    banner("combine of 59 MB of rows, then its scored backward")
    gen = torch.Generator(device=dev).manual_seed(3)
    idx = torch.rand(n, e, device=dev, generator=gen).topk(k).indices
    scores, _idx, _counts, _offs, slot_pos, tok_pos = ops.reorder(torch.rand(n, k, device=dev, generator=gen), idx, e)
    shared, go = (torch.randn(n, d, device=dev, generator=gen).bfloat16() for _ in range(2))
    rows = torch.randn(n * k, d, device=dev, generator=gen).bfloat16()
    flush = torch.empty(1 << 28, dtype=torch.int32, device=dev)

    def backward():
        ops.combine_backward(go, rows, slot_pos, tok_pos, scores)

    def timed(first):
        times = []
        for _ in range(9):
            flush.zero_()  # 1 GB: nothing of the rows is left in the caches
            first()
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            backward()
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return sorted(times)[4]

    timed(backward)
    own, after = timed(backward), timed(lambda: ops.combine(shared, rows, slot_pos, tok_pos, scores))
    assert after < 1.25 * own, (after, own)
