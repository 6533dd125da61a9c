"""The fp32 expert GEMMs at the edges of their 64 x 64 x 32 tiles (rows around a tile, one
row, empty experts, counts that leave rows over) and with operands that are not 16-byte
aligned, against 64-bit products on the device. fp32 sums of n terms in any order are
within n 2^-24 of the sum of magnitudes; over these n <= 1024 random terms that is far
below the bound of 2e-5 of the tensor's largest magnitude.
"""

import pytest
import torch

from tests.conftest import banner

pytestmark = pytest.mark.gpu

TOL = 2e-5

CASES = {  # D, H, counts, rows past the counts
    "tile_edges": (64, 128, [63, 64, 65, 1, 0, 128, 129], 0),
    "one_row": (128, 64, [0, 1, 0], 0),
    "rest": (192, 320, [10, 0, 100], 77),
    "all_rest": (64, 64, [0, 0], 70),
    "many_experts": (64, 64, [i % 7 for i in range(300)], 3),
    "wide": (512, 1024, [700, 33, 0, 450], 0),
    # at most 64 rows per expert: weight gradients with one stage, whole, half and several of them
    "few_per_expert": (128, 192, [100, 0, 16, 17, 32, 33, 15, 1, 0, 97], 5),
}


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("shift", [0, 1], ids=["aligned", "unaligned"])
def test_f32_tiles(dev, name, shift):
    from torchtitan_amd import ops

    d, h, counts, rest = CASES[name]
    banner(f"fp32 experts {name}, operands {4 * shift} bytes off")
    e, rows = len(counts), sum(counts) + rest
    gen = torch.Generator(device=dev).manual_seed(11)

    def rnd(*shape, std=1.0):
        n = 1
        for v in shape:
            n *= v
        return (torch.randn(n + shift, generator=gen, device=dev) * std)[shift:].view(*shape)

    x, dy = rnd(rows, d), rnd(rows, d)
    w1, w2, w3 = rnd(e, h, d, std=0.1), rnd(e, d, h, std=0.1), rnd(e, h, d, std=0.1)
    leaves = [t.requires_grad_(True) for t in (x, w1, w2, w3)]
    cnt = torch.tensor(counts, dtype=torch.int64, device=dev)
    y, g, u, hh = ops.grouped_swiglu_f32(*leaves, cnt)
    got = torch.autograd.grad(y, leaves, dy)

    ref = [t.detach().double().requires_grad_(True) for t in leaves]
    out, s = [], 0
    for i, c in enumerate(counts):
        xe = ref[0][s:s + c]
        out.append((torch.nn.functional.silu(xe @ ref[1][i].t()) * (xe @ ref[3][i].t())) @ ref[2][i].t())
        s += c
    out.append(torch.zeros(rest, d, dtype=torch.float64, device=dev))
    yr = torch.cat(out)
    want = torch.autograd.grad(yr, ref, dy.double(), allow_unused=True)
    for what, a, b in (("y", y, yr), *((f"gradient {i}", a, b) for i, (a, b) in enumerate(zip(got, want)))):
        b = torch.zeros_like(a, dtype=torch.float64) if b is None else b
        den = b.abs().max().item()
        err = (a.double() - b).abs().max().item() / (den if den > 0 else 1.0)
        assert err <= TOL, (what, err)
    for t in (y, g, u, hh, got[0]):
        assert not t[rows - rest:].any(), "rows past the counts are zero"


def test_f32_no_rows(dev):
    """No rows at all (x of zero rows, counts all zero): empty results and zero weight
    gradients, through the op and through GroupedExperts on the per-expert path, which
    cuts x to the rows that the counts cover."""
    from torchtitan_amd import GroupedExperts, ops

    d, h, e = 64, 128, 3
    banner("fp32 experts without rows")
    cnt = torch.zeros(e, dtype=torch.int64, device=dev)
    x = torch.empty(0, d, device=dev, requires_grad=True)
    ws = [torch.randn(*s, device=dev, requires_grad=True) for s in ((e, h, d), (e, d, h), (e, h, d))]
    y, g, u, hh = ops.grouped_swiglu_f32(x, *ws, cnt)
    assert y.shape == (0, d) and g.shape == u.shape == hh.shape == (0, h)
    got = torch.autograd.grad(y, [x, *ws], torch.empty_like(y))
    assert got[0].shape == (0, d)
    for w, gw in zip(ws, got[1:]):
        assert torch.equal(gw, torch.zeros_like(w))

    experts = GroupedExperts.Config(dim=d, hidden_dim=h, num_experts=e, use_grouped_mm=False).build().to(dev)
    with torch.no_grad():
        for p in experts.parameters():
            p.normal_()
    for rows in (0, 70):  # 70: rows that no count covers
        x = torch.randn(rows, d, device=dev, requires_grad=True)
        y = experts(x, cnt)
        assert y.shape == (0, d)
        got = torch.autograd.grad(y, [x, *experts.parameters()], torch.empty_like(y))
        for t, gt in zip([x, *experts.parameters()], got):
            assert torch.equal(gt, torch.zeros_like(t))


@pytest.mark.parametrize("mode", ["gate_up", "down", "bwd_dgu", "bwd_dx"])
def test_f32_rows_past_the_counts_are_cheap(dev, mode):
    """The row kernels on a buffer whose first eighth holds the experts' rows take about as
    long as on that eighth alone (1.1 to 1.4 times as measured): the tiles spread over all
    eight XCDs whatever the grid is sized for. An order over the grid put them on one, six
    times as long."""
    from torchtitan_amd import _lib

    d, h, e, used = 512, 1024, 8, 8192
    banner(f"fp32 {mode}, rows past the counts")
    cnt = torch.full((e,), used // e, dtype=torch.int64, device=dev)
    rows = 8 * used
    wide = [torch.zeros(rows, h, device=dev) for _ in range(4)]
    narrow = [torch.zeros(rows, d, device=dev) for _ in range(2)]
    w1, w3 = torch.zeros(e, h, d, device=dev), torch.zeros(e, h, d, device=dev)
    (g, u, o0, o1), (x, y) = [t.data_ptr() for t in wide], [t.data_ptr() for t in narrow]
    w1p, w3p, cp, st = w1.data_ptr(), w3.data_ptr(), cnt.data_ptr(), torch.cuda.current_stream().cuda_stream

    def launch(r):
        name = "moe_grouped_gemm_f32_" + mode
        if mode == "gate_up":
            _lib.call(name, x, w1p, w3p, cp, r, e, d, h, g, u, o0, st)
        elif mode == "down":
            _lib.call(name, g, w1p, cp, r, e, d, h, y, st)
        elif mode == "bwd_dgu":
            _lib.call(name, x, w1p, g, u, cp, r, e, d, h, o0, o1, st)
        else:
            _lib.call(name, g, u, w1p, w3p, cp, r, e, d, h, y, st)

    def fastest(r):
        best = float("inf")
        for _ in range(10):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            for _ in range(4):
                launch(r)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    launch(rows)
    alone, padded = fastest(used), fastest(rows)
    print(f"{mode}: {alone / 4 * 1e3:.0f} us alone, {padded / 4 * 1e3:.0f} us with rows past the counts", flush=True)
    assert padded < 3 * alone


def _tail_tensors(dev, rows, cols, shift):
    """[rows, cols] tensors of ones, `shift` floats off a 16-byte boundary, and their buffers."""
    bufs = [torch.ones(rows * c + shift + 4, device=dev) for c in cols]
    return bufs, [b[shift:shift + rows * c].view(rows, c) for b, c in zip(bufs, cols)]


@pytest.mark.parametrize("cols", [(64, 3, 1, 130), (5, 0, 0, 7)], ids=["four", "two"])
@pytest.mark.parametrize("shift", [0, 1, 2, 3])
@pytest.mark.parametrize("used", [0, 1, 36, 37, 60])
def test_f32_zero_rows_past(dev, cols, shift, used):
    """Exactly the rows past the counts are cleared, wherever they and their tensors begin
    and end between 16-byte boundaries, also where a count is negative or past the rows."""
    from torchtitan_amd import _lib

    rows = 37
    banner(f"fp32 rows past the counts: {cols}, {used} of {rows} used, {shift} floats off")
    cnt = torch.tensor([-5, used, 0], dtype=torch.int64, device=dev)
    bufs, ts = _tail_tensors(dev, rows, cols, shift)
    args = [v for t, c in zip(ts, cols) for v in ((t.data_ptr() if c else None), c)]
    _lib.call("moe_zero_rows_past_f32", cnt.data_ptr(), rows, 3, *args, torch.cuda.current_stream().cuda_stream)
    for b, c in zip(bufs, cols):
        want = torch.ones_like(b)
        want[shift + min(used, rows) * c:shift + rows * c] = 0
        assert torch.equal(b, want), c


@pytest.mark.parametrize("experts", [600, 1023])
def test_f32_zero_rows_past_sum_of_counts_in_64_bits(dev, experts):
    """Counts of more rows than there are cover every row: nothing is cleared, also where
    their sum is past 32 bits: E (2^22 + 2^13) as an int is negative for 600 experts and a
    little less than the rows for 1023."""
    from torchtitan_amd import _lib

    banner(f"fp32 rows past the counts, {experts} counts of all rows")
    rows = (1 << 22) + (1 << 13)
    cnt = torch.full((experts,), 1 << 40, dtype=torch.int64, device=dev)
    t = torch.ones(rows, device=dev)
    _lib.call("moe_zero_rows_past_f32", cnt.data_ptr(), rows, experts, t.data_ptr(), 1, None, 0, None, 0, None, 0,
              torch.cuda.current_stream().cuda_stream)
    assert bool((t == 1).all())


def test_f32_zero_rows_past_speed(dev):
    """Clearing many rows keeps about the pace of torch's fill (1.05 of its time as measured;
    4-byte stores of 64 blocks took 2.8 times as long)."""
    from torchtitan_amd import _lib

    banner("fp32 rows past the counts, speed")
    rows, cols = 65536, (1024, 1024, 1024, 512)
    cnt = torch.tensor([64], dtype=torch.int64, device=dev)
    ts = [torch.ones(rows, c, device=dev) for c in cols]
    args = [v for t, c in zip(ts, cols) for v in (t.data_ptr(), c)]
    st = torch.cuda.current_stream().cuda_stream

    def fastest(f):
        best = float("inf")
        for _ in range(10):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            a.record()
            f()
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    fill = fastest(lambda: [t.zero_() for t in ts])
    rest = fastest(lambda: _lib.call("moe_zero_rows_past_f32", cnt.data_ptr(), rows, 1, *args, st))
    print(f"fill {fill * 1e3:.0f} us, rows past the counts {rest * 1e3:.0f} us", flush=True)
    assert rest < 1.6 * fill


def test_f32_grid_slices(dev):
    """Grids of a little more than one slice of 65536 workgroups, every entry point:
    the same result as its parts launched alone (narrower weights, or fewer experts), whose
    grids are one slice; the sums are the same ones in the same order."""
    from torchtitan_amd import _lib

    banner("fp32 grids of two slices")
    gen = torch.Generator(device=dev).manual_seed(5)
    st = torch.cuda.current_stream().cuda_stream

    def rnd(*shape):
        return torch.randn(*shape, generator=gen, device=dev)

    def run(name, ins, dims, outs):
        _lib.call("moe_grouped_gemm_f32_" + name, *(t.data_ptr() for t in ins), *dims,
                  *(t.data_ptr() for t in outs), st)
        return outs

    rows, wide, k, e = 2112, 131072, 64, 2  # (33 + 2) x 2048 tiles
    cnt = torch.tensor([1000, 1112], dtype=torch.int64, device=dev)
    a, a2, w, w3 = rnd(rows, k), rnd(rows, k), rnd(e, wide, k), rnd(e, wide, k)
    gw, uw = rnd(rows, wide), rnd(rows, wide)
    half = wide // 2
    cut = [(lambda t, i=i: t[..., i * half:(i + 1) * half].contiguous()) for i in range(2)]
    cute = [(lambda t, i=i: t[:, i * half:(i + 1) * half].contiguous()) for i in range(2)]

    def new(n, cols):
        return [torch.full((rows, cols), float("nan"), device=dev) for _ in range(n)]

    got = run("gate_up", [a, w, w3, cnt], (rows, e, k, wide), new(3, wide))
    for i in range(2):
        part = run("gate_up", [a, cute[i](w), cute[i](w3), cnt], (rows, e, k, half), new(3, half))
        assert all(torch.equal(cut[i](x), y) for x, y in zip(got, part))
    got = run("down", [a, w, cnt], (rows, e, wide, k), new(1, wide))
    for i in range(2):
        assert torch.equal(cut[i](got[0]), run("down", [a, cute[i](w), cnt], (rows, e, half, k), new(1, half))[0])
    wt, w3t = w.view(e, k, wide), w3.view(e, k, wide)
    got = run("bwd_dgu", [a, wt, gw, uw, cnt], (rows, e, k, wide), new(2, wide))
    for i in range(2):
        part = run("bwd_dgu", [a, cut[i](wt), cut[i](gw), cut[i](uw), cnt], (rows, e, k, half), new(2, half))
        assert all(torch.equal(cut[i](x), y) for x, y in zip(got, part))
    got = run("bwd_dx", [a, a2, wt, w3t, cnt], (rows, e, wide, k), new(1, wide))
    for i in range(2):
        part = run("bwd_dx", [a, a2, cut[i](wt), cut[i](w3t), cnt], (rows, e, half, k), new(1, half))
        assert torch.equal(cut[i](got[0]), part[0])
    del got, part, w, w3, wt, w3t, gw, uw

    m, n, e, rows = 2048, 4096, 33, 660  # 33 x 2048 tiles a weight
    cnt = torch.full((e,), rows // e, dtype=torch.int64, device=dev)
    dg, du, h, x, dy = rnd(rows, n), rnd(rows, n), rnd(rows, n), rnd(rows, m), rnd(rows, m)

    def all3(lo, hi):
        s = slice(lo * rows // e, hi * rows // e)
        outs = [torch.full((hi - lo, *d), float("nan"), device=dev) for d in ((n, m), (n, m), (m, n))]
        ins = [t[s].contiguous() for t in (dg, du, dy, x, h)]
        run("bwd_dw_all", [*ins, cnt[lo:hi].contiguous()], ((hi - lo) * rows // e, hi - lo, m, n), outs)
        one = torch.full((hi - lo, n, m), float("nan"), device=dev)
        run("bwd_dw", [ins[0], ins[3], cnt[lo:hi].contiguous()], ((hi - lo) * rows // e, hi - lo, n, m), [one])
        return [*outs, one]

    got = all3(0, e)
    for lo, hi in ((0, 8), (8, 16), (16, 24), (24, 33)):
        assert all(torch.equal(x[lo:hi], y) for x, y in zip(got, all3(lo, hi)))


def test_f32_more_than_2_32_threads(dev):
    """8.4 million output rows of 4096 columns (137 GB) are 2^23 tiles and more, 2^32 threads
    of one launch: rows of the first, the last and of tiles between against 64 bits."""
    from torchtitan_amd import _lib

    d, h, rows = 4096, 64, (1 << 23) + 64
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < rows * (d + h) * 4 + (8 << 30):
        pytest.skip("needs 148 GB of free device memory")
    banner("fp32 down, 2^23 + 64 rows of 4096")
    gen = torch.Generator(device=dev).manual_seed(6)
    x = torch.randn(rows, h, generator=gen, device=dev)
    w2 = torch.randn(1, d, h, generator=gen, device=dev)
    cnt = torch.tensor([rows], dtype=torch.int64, device=dev)
    y = torch.empty(rows, d, device=dev)
    try:
        y[-64:].fill_(float("nan"))
        _lib.call("moe_grouped_gemm_f32_down", x.data_ptr(), w2.data_ptr(), cnt.data_ptr(), rows, 1, d, h,
                  y.data_ptr(), torch.cuda.current_stream().cuda_stream)
        for r in (0, 1 << 20, (1 << 22) - 64, 1 << 22, 1 << 23):
            want = x[r:r + 64].double() @ w2[0].double().t()
            err = (y[r:r + 64].double() - want).abs().max().item() / want.abs().max().item()
            assert err <= TOL, (r, err)
    finally:
        del y, x
        torch.cuda.empty_cache()


@pytest.mark.parametrize("shift", [0, 1], ids=["aligned", "unaligned"])
def test_f32_dw_alone(dev, shift):
    """bwd_dw for each weight by itself against bwd_dw_all, and the same experts among empty
    ones, which takes the kernel with one stage instead of two: bit for bit."""
    from torchtitan_amd import _lib

    d, h, counts = 192, 320, [300, 0, 33, 128, 50]
    banner(f"fp32 weight gradients alone, operands {4 * shift} bytes off")
    rows, st = sum(counts), torch.cuda.current_stream().cuda_stream
    gen = torch.Generator(device=dev).manual_seed(12)

    def rnd(*shape):
        return torch.randn(shape[0] * shape[1] + shift, generator=gen, device=dev)[shift:].view(*shape)

    dg, du, hh, x, dy = rnd(rows, h), rnd(rows, h), rnd(rows, h), rnd(rows, d), rnd(rows, d)
    ptrs = [t.data_ptr() for t in (dg, du, dy, x, hh)]

    def new(e, m, n):
        return torch.full((e, m, n), float("nan"), device=dev)

    want = None
    for empty in (0, 20):
        cnt = torch.tensor(counts + [0] * empty, dtype=torch.int64, device=dev)
        e = len(counts) + empty
        assert (rows <= 64 * e) == (empty > 0)
        got = [new(e, h, d), new(e, h, d), new(e, d, h)]
        _lib.call("moe_grouped_gemm_f32_bwd_dw_all", *ptrs, cnt.data_ptr(), rows, e, d, h, *(t.data_ptr() for t in got), st)
        want = want or got
        for a, b, m, n, all_ in ((dg, x, h, d, got[0]), (du, x, h, d, got[1]), (dy, hh, d, h, got[2])):
            one = new(e, m, n)
            _lib.call("moe_grouped_gemm_f32_bwd_dw", a.data_ptr(), b.data_ptr(), cnt.data_ptr(), rows, e, m, n,
                      one.data_ptr(), st)
            assert torch.equal(one, all_)
        for a, b in zip(got, want):
            assert torch.equal(a[:len(counts)], b[:len(counts)]) and not a[len(counts):].any()


def test_f32_dw_of_few_rows_is_bound_by_its_stores(dev):
    """250 rows on 64 experts (1024 / 704): the three weight gradients, 554 MB, take 1.7 times as
    long as torch's fill of as much (2.3 times with two stages and a scan behind barriers)."""
    from torchtitan_amd import _lib

    d, h, e, rows = 1024, 704, 64, 250
    banner("fp32 weight gradients of few rows")
    gen = torch.Generator(device=dev).manual_seed(13)
    cnt = torch.bincount(torch.randint(e, (rows,), generator=gen, device=dev), minlength=e)
    dg, du, hh = (torch.randn(rows, h, generator=gen, device=dev) for _ in range(3))
    x, dy = (torch.randn(rows, d, generator=gen, device=dev) for _ in range(2))
    outs = [torch.empty(s, device=dev) for s in ((e, h, d), (e, h, d), (e, d, h))]
    st = torch.cuda.current_stream().cuda_stream

    def kernel():
        _lib.call("moe_grouped_gemm_f32_bwd_dw_all", *(t.data_ptr() for t in (dg, du, dy, x, hh, cnt)), rows, e, d, h,
                  *(t.data_ptr() for t in outs), st)

    def fill():
        for o in outs:
            o.fill_(1.0)

    def timed(fn):
        times = []
        for _ in range(9):
            a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
            torch.cuda._sleep(500_000)
            a.record()
            fn()
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return sorted(times)[4]

    timed(kernel)
    t, f = timed(kernel), timed(fill)
    print(f"dw {t * 1e3:.1f} us, fill {f * 1e3:.1f} us, {t / f:.2f}")
    assert t < 2.0 * f, (t, f)
