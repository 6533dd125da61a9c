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
