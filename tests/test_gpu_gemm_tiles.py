"""The bf16 grouped GEMMs over the shapes at which the launch picks each of its tiles
(whole and partial last tiles, few, some and many rows per expert, empty experts):
outputs and gradients against fp32 per-expert products of the same bf16 inputs on the
device. The bounds, relative to the tensor's largest magnitude, are the bf16 roundings
(2^-9 of a value each) that can all fall one way where an element sums few rows. SwiGLU:
g, u, silu, h and the result, five, 1e-2. gpt-oss: h1 and its bias sum, alpha g, the
sigmoid, their product, u + 1, h and the result, eight, 2^-6.
"""

import pytest
import torch

from tests.conftest import banner

pytestmark = pytest.mark.gpu

TOL = {False: 1e-2, True: 2.0 ** -6}

CASES = {  # experts, D, H, rows, seed
    # fewer rows than experts, small dW tiles
    "few_rows": (24, 320, 192, 17, 1),
    # one row in all
    "one_row": (4, 192, 320, 1, 2),
    # dW at half a chip of wide tiles and above it: 128 x 128 and 256 x 256, partial both ways
    "dw_small_tail": (8, 448, 576, 1500, 3),
    "dw_wide_tail": (24, 832, 960, 3000, 4),
    # dgu on 64-row tiles; dx on 128 x 384 with a partial last tile
    "dgu_low": (32, 1472, 1472, 4096, 5),
    # dx on 128 x 512, partial, and on 128 x 256
    "dx_wide": (32, 1472, 1472, 16384, 6),
    "dx_narrow": (48, 1600, 832, 600, 7),
    # dgu and dx with two workgroups per CU
    "two_per_cu": (48, 1600, 832, 24576, 8),
    # 256 x 256 forward tiles, long and short contraction
    "tall": (8, 1088, 704, 9000, 9),
    "tall_long": (4, 4160, 320, 5000, 10),
}


def _close(a, b, what, tol):
    den = b.abs().max().item()
    err = (a.float() - b).abs().max().item() / (den if den > 0 else 1.0)
    assert err <= tol, (what, err)


@pytest.mark.parametrize("name", list(CASES))
@pytest.mark.parametrize("oss", [False, True], ids=["swiglu", "gptoss"])
def test_tiles(dev, name, oss):
    from torchtitan_amd import ops

    e, d, h, rows, seed = CASES[name]
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
