"""The bf16 grouped GEMMs over the shapes at which the launch picks each of its tiles
(whole and partial last tiles, few, some and many rows per expert, empty experts; which
tile a shape takes on 256 CUs is asserted, without a GPU):

* outputs and gradients against fp32 per-expert products of the same bf16 inputs on the
  device. The bounds, relative to the tensor's largest magnitude, are the bf16 roundings
  (2^-9 of a value each) that can all fall one way where an element sums few rows. SwiGLU:
  g, u, silu, h and the result, five, 1e-2. gpt-oss: h1 and its bias sum, alpha g, the
  sigmoid, their product, u + 1, h and the result, eight, 2^-6.
* the same rows of an expert under every tile, bit for bit: each runs the same MFMAs in the
  same k order.
"""

import pytest
import torch

from tests.conftest import banner

gpu = pytest.mark.gpu

TOL = {False: 1e-2, True: 2.0 ** -6}
CUS = 256  # MI355X

# mode -> the tiles that it has, (rows, columns, workgroups per CU)
MODES = ("gate_up", "down", "dgu", "dx", "dw1", "dw2")
FWD, TALL, TWO = (128, 256, 1), (256, 256, 1), (128, 256, 2)
DX384, DX512, LOW, SMALL = (128, 384, 1), (128, 512, 1), (64, 256, 2), (128, 128, 2)
TILES = {"gate_up": {FWD, TALL}, "down": {FWD, TALL}, "dgu": {FWD, TWO, LOW}, "dx": {FWD, TWO, DX384, DX512},
         "dw1": {SMALL, TALL}, "dw2": {SMALL, TALL}}


def tiles_of(oss):
    return {**TILES, "dx": TILES["dx"] | {TALL}} if oss else TILES


def tile(mode, oss, e, d, h, rows):
    from torchtitan_amd import _lib

    t = _lib.lib().moe_grouped_gemm_tile(MODES.index(mode), int(oss), rows, e, d, h, CUS)
    assert t > 0, t
    return t // 10000, t % 10000 // 10, t % 10


CASES = {  # experts, D, H, rows, seed, the tiles that the case is there for (SwiGLU; gpt-oss where it differs)
    # fewer rows than experts, small dW tiles
    "few_rows": (24, 320, 192, 17, 1, dict(gate_up=FWD, dw1=SMALL, dw2=SMALL)),
    # one row in all
    "one_row": (4, 192, 320, 1, 2, dict(gate_up=FWD, down=FWD, dgu=FWD, dx=FWD)),
    # dW at half a chip of wide tiles and above it, partial both ways
    "dw_small_tail": (8, 448, 576, 1500, 3, dict(dw1=SMALL, dw2=SMALL)),
    "dw_wide_tail": (24, 832, 960, 3000, 4, dict(dw1=TALL, dw2=TALL)),
    # dgu on 64-row tiles; dx on 128 x 384 with a partial last tile
    "dgu_low": (32, 1472, 1472, 4096, 5, dict(dgu=LOW, dx=DX384)),
    # forward on partial 256 x 256 tiles, dx on two workgroups per CU and, gpt-oss, 256 x 256
    "dx_tall": (32, 1472, 1472, 16384, 6, dict(gate_up=TALL, down=TALL, dgu=TWO, dx=(TWO, TALL))),
    # dx on 128 x 384, an expert's rows in one tile
    "dx_384": (48, 1600, 832, 600, 7, dict(dgu=FWD, dx=DX384)),
    # dgu and dx with two workgroups per CU
    "two_per_cu": (48, 1600, 832, 24576, 8, dict(dgu=TWO, dx=TWO)),
    # 256 x 256 forward tiles, long and short contraction
    "tall": (8, 1088, 704, 9000, 9, dict(gate_up=TALL, down=TALL)),
    "long": (4, 4160, 320, 5000, 10, dict(gate_up=FWD, down=FWD)),
    "tall_long": (6, 4160, 320, 12000, 11, dict(gate_up=TALL, down=TALL)),
    # dx on 128 x 512 over whole tiles, and, gpt-oss, with a partial last one
    "dx_512": (24, 2048, 576, 6000, 12, dict(dx=DX512)),
    "dx_512_tail": (48, 1600, 832, 4000, 13, dict(dx=(None, DX512))),
}


@pytest.mark.parametrize("oss", [False, True], ids=["swiglu", "gptoss"])
def test_cases_take_their_tiles(oss):
    """Each case takes the tiles that it is there for, and the cases take every tile."""
    taken = {m: set() for m in MODES}
    for name, (e, d, h, rows, _, want) in CASES.items():
        for m in MODES:
            t = tile(m, oss, e, d, h, rows)
            taken[m].add(t)
            w = want.get(m)
            if isinstance(w, tuple) and not isinstance(w[-1], int):
                w = w[oss]
            if w is not None:
                assert t == w, (name, m, t)
    assert taken == tiles_of(oss)


@pytest.mark.parametrize("oss", [False, True], ids=["swiglu", "gptoss"])
@pytest.mark.parametrize("e,d,h", [(256, 2304, 1024), (64, 2048, 1408), (32, 7168, 2048), (128, 2880, 2880)])
def test_experts_without_a_row_do_not_change_the_tile(oss, e, d, h):
    """With no more rows than experts the row kernels take the tile of that many experts."""
    for rows in range(1, e):
        for m in MODES[:4]:
            assert tile(m, oss, e, d, h, rows) == tile(m, oss, rows, d, h, rows), (m, rows)


@pytest.mark.parametrize("e,d,h,rows", [(64, 3072, 1536, 6701), (256, 2304, 1024, 23480), (128, 1536, 768, 30816),
                                        (64, 2304, 1024, 600), (24, 1536, 320, 44073)])
def test_dx_on_whole_384_tiles(e, d, h, rows):
    """Where D is a multiple of 384 and rounds do not speak clearly for another tile, dx stays on
    128 x 384, measured 5 to 30 % faster at these shapes than the tiles that cost a little less
    by their rounds."""
    assert tile("dx", False, e, d, h, rows) == DX384


def _close(a, b, what, tol):
    den = b.abs().max().item()
    err = (a.float() - b).abs().max().item() / (den if den > 0 else 1.0)
    assert err <= tol, (what, err)


@gpu
@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("oss", [False, True], ids=["swiglu", "gptoss"])
def test_tiles(dev, name, oss):
    from torchtitan_amd import ops

    e, d, h, rows, seed, _ = CASES[name]
    banner(f"grouped GEMM tiles {name} {'gpt-oss' if oss else 'swiglu'}")
    gen = torch.Generator().manual_seed(seed)
    load = torch.rand(e, generator=gen) ** 2
    load[e // 2] = 0  # an empty expert
    counts = torch.bincount(torch.multinomial(load, rows, replacement=True, generator=gen), minlength=e)
    gd = torch.Generator(device=dev).manual_seed(seed)

    def rnd(*shape, std=1.0):
        return (torch.randn(*shape, generator=gd, device=dev) * std).bfloat16()

    x, dy = rnd(rows, d).requires_grad_(True), rnd(rows, d)
    if oss:
        ws = [rnd(e, 2 * h, d, std=0.02), rnd(e, 2 * h, std=0.02), rnd(e, d, h, std=0.02), rnd(e, d, std=0.02)]
    else:
        ws = [rnd(e, h, d, std=0.02), rnd(e, d, h, std=0.02), rnd(e, h, d, std=0.02)]
    ws = [w.requires_grad_(True) for w in ws]
    cnt = counts.to(dev)
    if oss:
        y = ops.grouped_swiglu_oss(x, *ws, cnt, 7.0)[0]
    else:
        y = ops.grouped_swiglu(x, *ws, cnt)[0]
    got = torch.autograd.grad(y, [x, *ws], dy)

    xr = x.detach().float().requires_grad_(True)
    wr = [w.detach().float().requires_grad_(True) for w in ws]
    out, s = [], 0
    for i, c in enumerate(counts.tolist()):
        xe, pe = xr[s:s + c], [w[i] for w in wr]
        s += c
        if oss:
            h1 = xe @ pe[0].t() + pe[1]
            glu, lin = h1[:, ::2].clamp(max=7.0), h1[:, 1::2].clamp(min=-7.0, max=7.0)
            out.append((glu * torch.sigmoid(1.702 * glu) * (lin + 1)) @ pe[2].t() + pe[3])
        else:
            out.append((torch.nn.functional.silu(xe @ pe[0].t()) * (xe @ pe[2].t())) @ pe[1].t())
    yr = torch.cat(out)
    ref = torch.autograd.grad(yr, [xr, *wr], dy.float())
    _close(y.detach(), yr.detach(), "y", TOL[oss])
    for i, (a, b) in enumerate(zip(got, ref)):
        _close(a, b, f"gradient {i}", TOL[oss])
        if i and a.dim() == 3:
            assert not a[e // 2].any(), "gradient of an empty expert's weights"


def _every_bf16(rows, cols):
    """bf16 bit patterns over [rows, cols]: those in the reciprocal form's range first."""
    bits = torch.arange(-32768, 32768, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    f = bits.float()
    fast = (f >= -40.0) & (f <= 3.38e38)
    v = torch.cat([bits[fast], bits[~fast]])
    return v.repeat((rows * cols + v.numel() - 1) // v.numel())[:rows * cols].view(rows, cols)


# D, H -> (experts, rows) that between them take every tile of every mode
SAME_ROWS = {
    (1536, 512): [(2, 500), (12, 28000), (48, 500), (48, 6000), (48, 14000)],
    (1600, 832): [(2, 500), (6, 8000), (48, 4000), (48, 6000), (48, 7000)],
    (2048, 576): [(2, 500), (6, 12000), (24, 3000), (48, 8000), (48, 20000)],
}


@pytest.mark.parametrize("oss", [False, True], ids=["swiglu", "gptoss"])
def test_same_rows_take_every_tile(oss):
    taken = {m: {tile(m, oss, e, d, h, rows) for (d, h), runs in SAME_ROWS.items() for e, rows in runs} for m in MODES}
    assert taken == tiles_of(oss)


@gpu
@pytest.mark.parametrize("d,h", list(SAME_ROWS))
@pytest.mark.parametrize("oss", [False, True], ids=["swiglu", "gptoss"])
def test_tiles_give_the_same_bits(dev, d, h, oss):
    """The first and the last expert with the same 100 and 150 rows and weights among
    more and fewer other experts and rows, so that each launch takes another tile: their
    rows of every result and their weight gradients are the same bits."""
    from torchtitan_amd import ops

    assert torch.cuda.get_device_properties(dev).multi_processor_count == CUS
    banner(f"grouped GEMM tiles, same bits {d} / {h} {'gpt-oss' if oss else 'swiglu'}")
    gd = torch.Generator(device=dev).manual_seed(21)

    def rnd(*shape, std=1.0):
        return (torch.randn(*shape, generator=gd, device=dev) * std).bfloat16()

    n0, n1 = 100, 150
    shapes = [(2 * h, d), (2 * h,), (d, h), (d,)] if oss else [(h, d), (d, h), (h, d)]
    fixed_x, fixed_dy, fixed_w = rnd(n0 + n1, d), rnd(n0 + n1, d), [rnd(2, *s, std=0.02) for s in shapes]
    first = None
    for e, rows in SAME_ROWS[d, h]:
        gen = torch.Generator().manual_seed(rows)
        rest = rows - n0 - n1 if e > 2 else 0
        mid = torch.bincount(torch.randint(max(e - 2, 1), (rest,), generator=gen), minlength=e - 2) if e > 2 else []
        counts = torch.tensor([n0, *mid, n1], dtype=torch.int64, device=dev)
        pad = rows - n0 - n1 - rest  # two experts: rows past the counts
        x, dy = ([f[:n0], rnd(rest, d), f[n0:], rnd(pad, d)] for f in (fixed_x, fixed_dy))
        x, dy = torch.cat(x).requires_grad_(True), torch.cat(dy)
        ws = [torch.cat([f[:1], rnd(e - 2, *s, std=0.02), f[1:]]).requires_grad_(True) for f, s in zip(fixed_w, shapes)]
        out = ops.grouped_swiglu_oss(x, *ws, counts, 7.0) if oss else ops.grouped_swiglu(x, *ws, counts)
        got = torch.autograd.grad(out[0], [x, *ws], dy)
        own = [t.detach() for t in (*out, got[0]) if t.dim() == 2 and t.shape[0] == rows]
        assert len(own) == 5
        own = [torch.cat([t[:n0], t[n0 + rest:n0 + rest + n1]]) for t in own]
        own += [torch.stack([t[0], t[-1]]) for t in got[1:] if t.dim() == 3]
        if first is None:
            first = own
        for i, (a, b) in enumerate(zip(first, own)):
            assert torch.equal(a, b), (e, rows, i)


@gpu
def test_gptoss_epilogues_every_bf16(dev):
    """The gpt-oss epilogues on every bf16 value of g (infinities and NaNs included)
    against torch's bf16 ops and their autograd: h from the g and u that gate_up returns,
    and du from a one-hot dy, whose dh is mlp2's entries exactly, bit for bit; dg up to the
    order of the three factors of torch's sigmoid backward, which can move the bf16 rounding
    of that term, its product with alpha and the sum by one place (up to 2^-7) each."""
    from torchtitan_amd import _lib

    banner("gpt-oss epilogues, every bf16 g")
    rows, d, h, limit, alpha = 256, 256, 256, 7.0, 1.702
    gen = torch.Generator().manual_seed(13)
    gt = _every_bf16(rows, h).to(dev)
    u = (torch.randn(rows, h, generator=gen) * 4).bfloat16().to(dev)
    counts = torch.tensor([rows], dtype=torch.int64, device=dev)
    eye = torch.eye(rows, d, dtype=torch.bfloat16, device=dev)
    st = torch.cuda.current_stream().cuda_stream

    def act(g, v):
        xg, xl = g.clamp(max=limit), v.clamp(min=-limit, max=limit)
        return xg * torch.sigmoid(alpha * xg) * (xl + 1)

    def same(a, b):
        ok = (a.view(torch.int16) == b.view(torch.int16)) | (torch.isnan(a) & torch.isnan(b))
        assert bool(ok.all()), int((~ok).sum())

    w2 = (torch.randn(1, d, h, generator=gen) * 2).bfloat16().to(dev)
    dgu = torch.empty(rows, 2 * h, dtype=torch.bfloat16, device=dev)
    _lib.call("moe_grouped_gemm_oss_bwd_dgu", eye.data_ptr(), w2.data_ptr(), gt.data_ptr(), u.data_ptr(),
              counts.data_ptr(), rows, 1, d, h, limit, dgu.data_ptr(), st)
    gr, ur = gt.clone().requires_grad_(True), u.clone().requires_grad_(True)
    act(gr, ur).backward(w2[0])
    same(dgu[:, h:], ur.grad)
    dg, want, gf = dgu[:, :h].float(), gr.grad.float(), gt.float()
    assert torch.equal(torch.isfinite(dg), torch.isfinite(want))
    xg, xl = gf.clamp(max=limit), u.float().clamp(min=-limit, max=limit)
    sig = torch.sigmoid(alpha * xg)
    term = (alpha * w2[0].float() * (xl + 1) * xg * sig * (1 - sig)).abs()
    ok = (dg - want).abs() <= 2.0 ** -7 * (2 * torch.nan_to_num(term) + want.abs()) + 1e-30
    assert bool((ok | ~torch.isfinite(want)).all()), int((~ok & torch.isfinite(want)).sum())

    fin = torch.where(torch.isfinite(gt.float()), gt, torch.zeros_like(gt))
    w1 = torch.stack([fin.t(), u.t()], dim=1).reshape(1, 2 * h, d).contiguous()  # glu 2 j, linear 2 j + 1
    b1 = torch.randn(1, 2 * h, generator=gen).bfloat16().to(dev)
    g2, u2, h2 = (torch.empty(rows, h, dtype=torch.bfloat16, device=dev) for _ in range(3))
    _lib.call("moe_grouped_gemm_oss_gate_up", eye.data_ptr(), w1.data_ptr(), b1.data_ptr(), counts.data_ptr(), rows, 1,
              d, h, limit, g2.data_ptr(), u2.data_ptr(), h2.data_ptr(), st)
    same(h2, act(g2, u2))
