"""Layers whose channel counts are not multiples of 16 against the oracle:
forward with bias, input gradient and weight gradient at the edges of the
thin kernels' tiles (64 positions, 96 im2col columns, 16 / 32 / 64 output
columns; rows of 2-, 4- and 16-byte pieces) and of the padded widths (32, 64,
128, 192, 256; copies that run on the small-map kernel, on larger maps and on
more than 32 offsets on the tiled ones), on stride-2 maps, and with weights or
gradients that are not finite. Tolerance: norm-wise rel 1e-4 for fp32 and 2e-2
for bf16 (helpers.TOL)."""
import numpy as np
import pytest
import torch

import oracle
from riemannengine_amd import abi
from helpers import (DEV, TOL, assert_rel, gpu_tables_and_map, random_coords, reference_passes,
                     to_dev)


def test_ragged_weight_gradient_query_without_a_gpu():
    q = abi.lib().rhip_conv_backward_weight_ragged_supported
    assert q(abi.F32, 3, 32, 27, 1000, 1000) == 1 and q(abi.BF16, 64, 20, 1, 1000, 1000) == 1
    assert q(abi.BF16, 64, 48, 27, 1000, 1000) == 0  # the tiled kernels' shapes
    assert q(abi.F32, 40, 8, 27, 1000, 1000) == 1    # padded
    assert q(abi.F32, 40, 8, 129, 1000, 1000) == 0   # neither thin nor at most 128 offsets
    assert q(7, 3, 32, 27, 1000, 1000) == 0 and q(abi.F32, 3, 32, 27, -1, 1000) == 0


@pytest.mark.gpu
def test_a_pair_list_weight_gradient_asks_for_no_ragged_kernel(monkeypatch):
    """Neither thin nor padded (216 offsets of 40 channels): the query says so,
    and no call is made to be refused."""
    km, lib = _map(60, 6, seed=3, span=3), abi.lib()
    x, gy = (to_dev(np.ones((60, c), np.float32)) for c in (40, 8))

    def refused(*args):
        raise AssertionError("called for a shape its query refuses")

    monkeypatch.setattr(lib, "rhip_conv_backward_weight_ragged", refused)
    got = abi.conv_weight_grad(x, gy, km, km.K)
    pairs = torch.from_numpy(np.diff(km.offsets_host).astype(np.float32))
    assert torch.equal(got.cpu(), pairs[:, None, None].expand(km.K, 40, 8))


def _map(n, ks, seed, span=7):
    c, _, _ = oracle.insert_and_map(random_coords(np.random.default_rng(seed), 4 * n + 8, 3, span))
    c = c[:n]
    assert len(c) == n
    return gpu_tables_and_map(c, c, oracle.region_offsets(3, ks), same=True)[2]


def _reference(km, x, w, gy):
    kofs = km.offsets_host
    ir, orr = km.in_rows.cpu().numpy(), km.out_rows.cpu().numpy()
    y = oracle.conv_forward(x, w, kofs, ir, orr, km.n_out)
    return (y, *oracle.conv_backward(x, gy, w, kofs, ir, orr))


def _ragged_dw(x, gy, km):
    """rhip_conv_backward_weight_ragged itself (no fallback)."""
    dt = abi._dtype_code(x.dtype)
    gw = torch.empty((km.K, x.shape[1], gy.shape[1]), dtype=x.dtype, device=DEV)
    ws = abi._conv_ws(km.K, x.shape[1], gy.shape[1], dt, DEV, km)
    abi._check(abi.lib().rhip_conv_backward_weight_ragged(
        abi._ptr(x), km.n_in, x.shape[1], abi._ptr(gy), km.n_out, gy.shape[1], km.K,
        abi._ptr(km.nbr), abi._ptr(km.out_order), abi._ptr(gw), dt, abi._ptr(ws), ws.numel(),
        abi._stream(DEV)), "rhip_conv_backward_weight_ragged")
    return gw


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,ks,cin,cout", [
    (1, 3, 3, 32), (63, 3, 1, 16), (64, 3, 2, 33), (65, 3, 3, 64), (700, 3, 3, 32),
    (700, 3, 4, 80), (129, 3, 6, 13), (300, 5, 1, 20), (300, 5, 6, 40), (257, 1, 64, 20),
    (1000, 1, 256, 10), (500, 1, 13, 21), (200, 2, 12, 100), (130, 3, 24, 24), (90, 3, 37, 5),
    (400, 3, 64, 20), (400, 3, 20, 64), (257, 3, 33, 65), (129, 2, 40, 129), (300, 3, 200, 72),
    (200, 5, 24, 40), (150, 3, 300, 8), (3000, 3, 40, 40), (5000, 3, 72, 129),
    (5001, 3, 24, 100)])
def test_ragged_layers_match_oracle(n, ks, cin, cout, dtype):
    km = _map(n, ks, seed=n + ks)
    rng = np.random.default_rng(cin * 31 + cout)
    x, gy = rng.standard_normal((n, cin)), rng.standard_normal((n, cout))
    w = rng.standard_normal((km.K, cin, cout)) / np.sqrt(cin * km.K)
    b = rng.standard_normal(cout).astype(np.float32)
    xt, wt, gyt = (to_dev(a.astype(np.float32), dtype) for a in (x, w, gy))
    print(f"ragged n={n} ks={ks} {cin}->{cout} {dtype}", flush=True)
    assert all(abi.conv_plan(dtype, km.K, *s, n, n)[0] in ("thin", "padded")
               for s in ((cin, cout), (cout, cin)))
    y = abi.conv_forward(xt, wt, km, bias=to_dev(b))
    gx = abi.conv_backward_input(gyt, wt, km)
    ry, rgx, rgw = _reference(km, *(t.float().cpu().numpy() for t in (xt, wt, gyt)))
    assert_rel(y.float().cpu().numpy(), ry + b, TOL[dtype], "Y")
    assert_rel(gx.float().cpu().numpy(), rgx, TOL[dtype], "dX")
    if not (cin % 16 == 0 and cout % 16 == 0):
        gw = _ragged_dw(xt, gyt, km)
        assert_rel(gw.float().cpu().numpy(), rgw, TOL[dtype], "dW")
        assert torch.equal(gw, _ragged_dw(xt, gyt, km))
        assert torch.equal(gw, abi.conv_weight_grad(xt, gyt, km, km.K))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("offset", [1, 3])
@pytest.mark.parametrize("c", [4, 24])
def test_ragged_layers_on_views_off_the_piece_alignment(dtype, offset, c):
    """Feature rows that start off 4 or 16 bytes (a contiguous view into a
    longer buffer) go in smaller pieces or are copied."""
    km = _map(200, 3, seed=9)
    rng = np.random.default_rng(5)
    flat = to_dev(rng.standard_normal(200 * c + offset).astype(np.float32), dtype)
    x = flat[offset:].view(200, c)
    w = to_dev(rng.standard_normal((27, c, c)).astype(np.float32) / 18, dtype)
    y, gw = abi.conv_forward(x, w, km), _ragged_dw(x, x, km)
    xc = x.clone()
    assert torch.equal(y, abi.conv_forward(xc, w, km))
    assert torch.equal(gw, _ragged_dw(xc, xc, km))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
@pytest.mark.parametrize("cin,cout", [(3, 20), (24, 20), (64, 40)])
def test_ragged_layers_keep_non_finite_values_to_their_pairs(cin, cout, dtype, bad):
    """A weight or gradient that is not finite reaches the outputs its pairs
    reach and no others, as in the pair sums (a missing neighbour is no 0 *
    inf), and a feature row's only the rows that gather it."""
    n = 400
    km = _map(n, 3, seed=4, span=5)
    rng = np.random.default_rng(8)
    x, gy = (rng.standard_normal((n, c)).astype(np.float32) for c in (cin, cout))
    w = rng.standard_normal((27, cin, cout)).astype(np.float32)
    xb, wb, gb = x.copy(), w.copy(), gy.copy()
    xb[17, 1], wb[5, 2, 7], gb[33, 4] = bad, bad, bad
    for xs, ws, gs in ((x, wb, gb), (xb, w, gy)):
        xt, wt, gt = (to_dev(a, dtype) for a in (xs, ws, gs))
        got = (abi.conv_forward(xt, wt, km), abi.conv_backward_input(gt, wt, km),
               _ragged_dw(xt, gt, km))
        with np.errstate(invalid="ignore"):
            ref = _reference(km, xs, ws, gs)
        for name, a, r in zip(("Y", "dX", "dW"), got, ref):
            a = a.float().cpu().numpy()
            assert np.array_equal(np.isfinite(a), np.isfinite(r)), name
            m = np.isfinite(r)
            assert m.any(), name
            assert_rel(a[m], r[m], TOL[dtype], name)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,cin,cout,fwd,dx", [
    (700, 13, 13, "rows", "rows"), (3000, 20, 24, "rows", "rows"), (900, 48, 20, "rows", "rows"),
    (900, 3, 40, "thin", "rows"), (20000, 24, 40, "padded", "rows"),
    (20000, 40, 64, "padded", "padded"), (700, 6, 12, "thin", "thin")])
def test_ragged_layers_on_stride_maps(n, cin, cout, fwd, dx, dtype):
    """2^3 stride-2 maps: with little work one lane per output, else thin or
    padded, in both directions."""
    rng = np.random.default_rng(n + cin)
    side = int(np.ceil(n ** (1 / 3)))
    grid = np.indices((1, side, side, side)).reshape(4, -1).T[:n]
    c = rng.permutation(grid).astype(np.int32)
    out = np.unique(oracle.stride(c, [2, 2, 2]), axis=0).astype(np.int32)
    km = gpu_tables_and_map(c, out, oracle.region_offsets(3, 2))[2]
    m = km.n_out
    assert km.n_in == n and 8 * m < 4 * n
    assert (abi.conv_plan(dtype, 8, cin, cout, n, m)[0],
            abi.conv_plan(dtype, 8, cout, cin, m, n, True)[0]) == (fwd, dx)
    x, gy = (to_dev(rng.standard_normal(s).astype(np.float32), dtype) for s in ((n, cin), (m, cout)))
    w = to_dev((rng.standard_normal((8, cin, cout)) / 4).astype(np.float32), dtype)
    print(f"ragged stride n={n} {cin}->{cout} {dtype}", flush=True)
    got = (abi.conv_forward(x, w, km), abi.conv_backward_input(gy, w, km),
           abi.conv_weight_grad(x, gy, km, 8))
    for name, a, ref in zip(("Y", "dX", "dW"), got, reference_passes(km, x, gy, w)):
        assert_rel(a.float().cpu().numpy(), ref.cpu().numpy(), TOL[dtype], name)
