"""The transposing quantizers that run a block per 128 rows, at the edges of those chunks
(groups of 0, 1, 127 to 129 and several hundred rows, one group, more groups than a wave
scans, rows and columns past the last group), byte for byte against the quantizers that
work another way: the MX row quantizer on each group transposed and zero padded in torch,
and the fp8 ones that take their own amax in a pass over a whole group.
"""

import pytest
import torch

from tests.conftest import banner

pytestmark = pytest.mark.gpu

CASES = {  # rows of each group, rows past them, columns
    "edges": ([127, 128, 129, 0, 1, 0, 300], 0, 128),
    "one_group": ([130], 5, 64),
    "last_empty": ([5, 257, 0], 40, 192),
    "many_groups": ([(37 * i) % 141 for i in range(257)], 9, 64),
    "wave_of_groups": ([(53 * i) % 150 for i in range(256)], 0, 128),
}


@pytest.mark.parametrize("name", list(CASES))
def test_token_chunks(dev, name):
    from torchtitan_amd import _lib
    from torchtitan_amd._lib import call, ptr

    groups, rest, c = CASES[name]
    banner(f"token quantizers by chunks {name}")
    e, r = len(groups), sum(groups) + rest
    gen = torch.Generator(device=dev).manual_seed(5)
    x = (torch.randn(r, c, generator=gen, device=dev) * torch.randn(r, 1, generator=gen, device=dev).exp()).bfloat16()
    counts = torch.tensor(groups, dtype=torch.int64, device=dev)
    rpad = (int(_lib.lib().moe_mxfp8_padded_rows(r, e)) + 127) // 128 * 128
    st = torch.cuda.current_stream().cuda_stream

    def u8(*shape):
        return torch.full(shape, 0xA5, dtype=torch.uint8, device=dev)

    qr, sr, qt, s = u8(r, c), u8(r, c // 32), u8(c, rpad), u8(rpad // 32, c)
    call("moe_mxfp8_quant_dual_tokens", ptr(x), ptr(counts), r, e, c, rpad, ptr(qr), ptr(sr), ptr(qt), ptr(s), st)
    wr, ws = u8(r, c), u8(r, c // 32)
    call("moe_mxfp8_quant_rows", ptr(x), r, c, ptr(wr), ptr(ws), st)
    n = sum(groups)
    assert torch.equal(qr[:n], wr[:n]) and torch.equal(sr[:n], ws[:n])
    want_q, want_s = torch.zeros_like(qt), torch.zeros_like(s)
    start = pstart = 0
    for g in groups:
        pad = (g + 127) // 128 * 128
        if g:
            t = torch.zeros(c, pad, dtype=torch.bfloat16, device=dev)
            t[:, :g] = x[start:start + g].t()
            q1, s1 = u8(c, pad), u8(c, pad // 32)
            call("moe_mxfp8_quant_rows", ptr(t), c, pad, ptr(q1), ptr(s1), st)
            want_q[:, pstart:pstart + pad] = q1
            want_s[pstart // 32:(pstart + pad) // 32] = s1.t()
        start, pstart = start + g, pstart + pad
    assert torch.equal(qt, want_q) and torch.equal(s, want_s)

    # fp8: from the groups' known amax, and with its own amax pass
    amax = torch.zeros(e, c, device=dev)
    start = 0
    for i, g in enumerate(groups):
        if g:
            amax[i] = x[start:start + g].float().abs().amax(0)
        start += g
    outs = []
    for known in (True, False):
        q, sc = u8(c, rpad), torch.zeros(e, c, device=dev)
        if known:
            call("moe_fp8_quant_tokens_t_amax", ptr(x), ptr(amax), ptr(counts), r, e, c, rpad, ptr(q), ptr(sc), st)
        else:
            call("moe_fp8_quant_tokens_t", ptr(x), ptr(counts), r, e, c, rpad, ptr(q), ptr(sc), st)
        outs.append((q, sc))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])


def test_token_chunks_counts_past_the_rows(dev):
    """Counts that sum up to twice the rows make more chunks than the launch has blocks:
    the columns past the last group, whose rows all lie past R, are still cleared, and the
    first group's bytes are those of its rows alone."""
    from torchtitan_amd import _lib
    from torchtitan_amd._lib import call, ptr

    r, c = 1536, 128
    banner("MX token quantizer, counts past the rows")
    gen = torch.Generator(device=dev).manual_seed(8)
    x = torch.randn(r, c, generator=gen, device=dev).bfloat16()
    st = torch.cuda.current_stream().cuda_stream

    def quant(groups):
        e = len(groups)
        counts = torch.tensor(groups, dtype=torch.int64, device=dev)
        rpad = int(_lib.lib().moe_mxfp8_padded_rows(r, e))
        q, s = (torch.full(d, 0xA5, dtype=torch.uint8, device=dev) for d in ((c, rpad), (rpad // 32, c)))
        call("moe_mxfp8_quant_tokens_t", ptr(x), ptr(counts), r, e, c, rpad, ptr(q), ptr(s), st)
        return q, s

    q, s = quant([r, r])
    want_q, want_s = quant([r])
    assert torch.equal(q[:, :r], want_q[:, :r]) and torch.equal(s[:r // 32], want_s[:r // 32])
    assert q.shape[1] > r and not q[:, r:].any() and not s[r // 32:].any()


@pytest.mark.parametrize("a,b", [(32, 64), (128, 128), (160, 192), (352, 128)])
def test_weight_chunks(dev, a, b):
    from torchtitan_amd._lib import call, ptr

    banner(f"weight quantizers by chunks {a} x {b}")
    e = 3
    gen = torch.Generator(device=dev).manual_seed(6)
    x = (torch.randn(e, a, b, generator=gen, device=dev) * torch.randn(e, 1, b, generator=gen, device=dev).exp()).bfloat16()
    st = torch.cuda.current_stream().cuda_stream

    def u8(*shape):
        return torch.full(shape, 0xA5, dtype=torch.uint8, device=dev)

    q, s, qt, t = u8(e, a, b), u8(e, a, b // 32), u8(e, b, a), u8(e, b, a // 32)
    call("moe_mxfp8_quant_dual_cols", ptr(x), e, a, b, ptr(q), ptr(s), ptr(qt), a * b, a, ptr(t), b * (a // 32),
         a // 32, st)
    wq, ws, wqt, wt = u8(e, a, b), u8(e, a, b // 32), u8(e, b, a), u8(e, b, a // 32)
    xt = x.transpose(1, 2).contiguous()
    call("moe_mxfp8_quant_rows", ptr(x), e * a, b, ptr(wq), ptr(ws), st)
    call("moe_mxfp8_quant_rows", ptr(xt), e * b, a, ptr(wqt), ptr(wt), st)
    for got, want in ((q, wq), (s, ws), (qt, wqt), (t, wt)):
        assert torch.equal(got, want)
    q2, t2 = u8(e, b, a), u8(e, b, a // 32)
    call("moe_mxfp8_quant_cols_t", ptr(x), e, a, b, ptr(q2), a * b, a, ptr(t2), b * (a // 32), a // 32, st)
    assert torch.equal(q2, wqt) and torch.equal(t2, wt)
    amax = x.float().abs().amax(1).contiguous()
    f = [(u8(e, b, a), torch.zeros(e, b, device=dev)) for _ in range(2)]
    call("moe_fp8_quant_cols_t_amax", ptr(x), ptr(amax), e, a, b, ptr(f[0][0]), a * b, a, ptr(f[0][1]), b, st)
    call("moe_fp8_quant_cols_t", ptr(x), e, a, b, ptr(f[1][0]), a * b, a, ptr(f[1][1]), b, st)
    assert torch.equal(f[0][0], f[1][0]) and torch.equal(f[0][1], f[1][1])


def test_token_chunks_more_than_2_32_threads(dev):
    """8.4 million gathered rows of 16384 columns (137 GB of fp8) are 2^23 blocks and more,
    2^32 threads of one launch: columns of the first, the last and of slabs between against
    a small call on the 64 rows that all of them repeat."""
    from torchtitan_amd._lib import call, ptr

    c, n_src = 16384, 64
    r = (1 << 23) + n_src
    rpad = (r + 127) // 128 * 128 + 128
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < c * rpad + (8 << 30):
        pytest.skip("needs 146 GB of free device memory")
    banner("fp8 token quantizer, 2^23 + 64 rows of 16384")
    gen = torch.Generator(device=dev).manual_seed(7)
    src = torch.randn(n_src, c, generator=gen, device=dev).bfloat16()
    amax = src.float().abs().amax(0)[None].contiguous()
    st = torch.cuda.current_stream().cuda_stream

    def quant(rows, padded):
        idx = torch.arange(rows, device=dev) % n_src
        counts = torch.tensor([rows], dtype=torch.int64, device=dev)
        q = torch.empty(c, padded, dtype=torch.uint8, device=dev)
        s = torch.empty(1, c, device=dev)
        call("moe_fp8_quant_tokens_t_amax_gather", ptr(src), n_src, ptr(idx), None, ptr(amax), ptr(counts), rows, 1, c,
             padded, ptr(q), ptr(s), st)
        return q, s

    want, ws = quant(n_src, 256)
    q, s = quant(r, rpad)
    try:
        assert torch.equal(s, ws)
        for col in (0, 1, 127, 128, 8191, 8192, c - 129, c - 1):
            row = q[col, :r].view(-1, n_src)
            assert bool((row == want[col, :n_src]).all()), col
            assert not q[col, r:(r + 127) // 128 * 128].any(), col
    finally:
        del q
        torch.cuda.empty_cache()


@pytest.mark.parametrize("kind", ["fp8_known_amax", "fp8", "mx", "mx_dual", "fp8_more_than_2_32_threads"])
def test_weight_chunks_in_slices(dev, kind):
    """Launches of more than one slice of 65536 blocks, and one of 2^23 blocks (1024 experts
    of 144 x 524288, 154 GB of weights), which is 2^32 threads: every expert repeats 128
    columns, whose bytes are those of a small launch."""
    from torchtitan_amd._lib import call, ptr

    huge = kind == "fp8_more_than_2_32_threads"
    e, a, b = (1024, 144, 1 << 19) if huge else (3, 160, 128 * 21846 if kind == "fp8" else 128 * 10924)
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < e * b * (3 * a + 8) + (8 << 30):
        pytest.skip(f"needs {e * b * (3 * a + 8) >> 30} GB of free device memory")
    banner(f"weight quantizer {kind}, {e} x {a} x {b}")
    gen = torch.Generator(device=dev).manual_seed(9)
    src = torch.randn(a, 128, generator=gen, device=dev).bfloat16()
    st = torch.cuda.current_stream().cuda_stream

    def u8(*shape):
        return torch.full(shape, 0xA5, dtype=torch.uint8, device=dev)

    def quant(e, b):
        x = torch.empty(e, a, b, dtype=torch.bfloat16, device=dev)
        x.view(e, a, b // 128, 128).copy_(src[None, :, None, :])
        if kind.startswith("fp8"):
            q, s = u8(e, b, a), torch.zeros(e, b, device=dev)
            if kind == "fp8":
                call("moe_fp8_quant_cols_t", ptr(x), e, a, b, ptr(q), a * b, a, ptr(s), b, st)
            else:
                amax = src.float().abs().amax(0).repeat(e, b // 128)
                call("moe_fp8_quant_cols_t_amax", ptr(x), ptr(amax), e, a, b, ptr(q), a * b, a, ptr(s), b, st)
            return [(q, a), (s, 1)]
        t, ts = u8(e, b, a), u8(e, b, a // 32)
        args = (ptr(t), a * b, a, ptr(ts), a // 32 * b, a // 32, st)
        if kind == "mx":
            call("moe_mxfp8_quant_cols_t", ptr(x), e, a, b, *args)
            return [(t, a), (ts, a // 32)]
        q, s = u8(e, a, b), u8(e, a, b // 32)
        call("moe_mxfp8_quant_dual_cols", ptr(x), e, a, b, ptr(q), ptr(s), *args)
        return [(t, a), (ts, a // 32), (q, None), (s, None)]

    got = want = None
    try:
        want = quant(1, 128)
        got = quant(e, b)
        for (t, n), (w, _) in zip(got, want):
            for i in range(0, e, 73):
                if n is None:  # row-wise: 128 columns, or their four scales, repeat in each row
                    assert bool((t[i].view(a, -1, w.shape[2]) == w[0][:, None]).all())
                else:
                    assert bool((t[i].view(-1, 128, n) == w.view(128, n)).all()), i
            if n is not None:  # the last expert's last columns
                assert bool((t[-1].view(-1, 128, n)[-1] == w.view(128, n)).all())
    finally:
        del got, want
        torch.cuda.empty_cache()
