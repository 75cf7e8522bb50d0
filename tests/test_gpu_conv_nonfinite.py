"""A value that is not finite changes the outputs it reaches, in every kernel
that adds such outputs up a second time: the small-map kernel, fp32 operands
in bf16 parts (whole and split), and layers on padded copies. An infinity
times ordinary values is not finite, so the outputs to change are exactly
those with a pair on it. Of the others, those in the column of a weight or
gradient that is not finite may be sums in another order (their rows' missing
neighbours are multiplied with it first): 2^-24 or 2^-8 per rounding, up to
2,000 of them at random, is under 1e-5 or 2e-2 of the largest; all others keep
their bits."""
import numpy as np
import pytest
import torch

import oracle
from riemannengine_amd import abi
from helpers import DEV, gpu_tables_and_map, random_coords

pytestmark = pytest.mark.gpu


def _map(n, span, ks=3):
    c, _, _ = oracle.insert_and_map(random_coords(np.random.default_rng(n), 4 * n + 8, 3, span))
    assert len(c) >= n
    return gpu_tables_and_map(c[:n], c[:n], oracle.region_offsets(3, ks), same=True)[2]


def _same_but(clean, got, hit, column=None):
    assert torch.isfinite(clean).all()
    assert torch.equal(torch.isfinite(got), ~hit)
    if column is not None:
        a, b, m = (t[..., column].float() for t in (clean, got, hit))
        tol = 1e-5 if clean.dtype == torch.float32 else 2e-2
        assert float((a - b)[m == 0].abs().max()) <= tol * float(a.abs().max())
        hit[..., column] = True
    assert torch.equal(clean[~hit], got[~hit])


@pytest.mark.parametrize("n,span,cin,cout,dtype,kernel", [
    (300, 5, 64, 64, torch.float32, "small"), (77, 4, 32, 48, torch.float32, "small"),
    (300, 5, 64, 64, torch.bfloat16, "small"), (100, 4, 96, 32, torch.bfloat16, "small"),
    (6000, 12, 64, 64, torch.float32, "parts split"),
    (5000, 11, 96, 192, torch.float32, "parts split"),
    (15001, 15, 256, 256, torch.float32, "parts"), (58000, 24, 64, 64, torch.float32, "parts"),
    (300, 5, 24, 40, torch.float32, "padded"), (300, 5, 24, 64, torch.bfloat16, "padded"),
    (400, 5, 64, 20, torch.bfloat16, "padded"), (6000, 12, 40, 40, torch.float32, "padded")])
def test_other_outputs_keep_their_bits(n, span, cin, cout, dtype, kernel):
    km = _map(n, span)
    for cred, ncols, dx in ((cin, cout, False), (cout, cin, True)):
        name, splits = abi.conv_plan(dtype, 27, cred, ncols, n, n, dx)
        assert name + (" split" if splits > 1 else "") == kernel
    g = torch.Generator(DEV).manual_seed(n)
    x, gy, w = (torch.randn(s, generator=g, device=DEV).to(dtype)
                for s in ((n, cin), (n, cout), (27, cin, cout)))
    print(f"nonfinite n={n} {cin}->{cout} {dtype} {kernel}", flush=True)
    ir, orr = km.in_rows.long(), km.out_rows.long()
    on = slice(int(km.offsets_host[4]), int(km.offsets_host[5]))  # offset 4's pairs
    inf = float("inf")

    def hits(rows, cols, r, c):
        m = torch.zeros(rows, cols, dtype=torch.bool, device=DEV)
        m[r, c] = True
        return m

    y, gx = abi.conv_forward(x, w, km), abi.conv_backward_input(gy, w, km)
    wb, xb, gb = w.clone(), x.clone(), gy.clone()
    wb[4, 2, 9], xb[n // 2, 3], gb[n // 3, 5] = inf, -inf, inf
    _same_but(y, abi.conv_forward(x, wb, km), hits(n, cout, orr[on], 9), 9)
    _same_but(gx, abi.conv_backward_input(gy, wb, km), hits(n, cin, ir[on], 2), 2)
    _same_but(y, abi.conv_forward(xb, w, km), hits(n, cout, orr[ir == n // 2], slice(None)))
    _same_but(gx, abi.conv_backward_input(gb, w, km),
              hits(n, cin, ir[orr == n // 3], slice(None)))
    if kernel == "padded":  # dW on padded copies: the offsets that pair the row, its column
        gw = abi.conv_weight_grad(x, gy, km, 27)
        ks = torch.repeat_interleave(torch.arange(27, device=DEV),
                                     torch.as_tensor(np.diff(km.offsets_host)).to(DEV))
        hit = torch.zeros(27, cin, cout, dtype=torch.bool, device=DEV)
        hit[ks[orr == n // 3].unique(), :, 5] = True
        _same_but(gw, abi.conv_weight_grad(x, gb, km, 27), hit, 5)
