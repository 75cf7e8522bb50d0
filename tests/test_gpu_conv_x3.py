"""fp32 forward and input gradient on three-part bf16 operands: against 64-bit
sums at the edges of its tiles (128 or 64 rows, 64 or 32 columns, one to four
mask words, split and whole offset axes), and with values no bf16 part can
hold. Tolerance: the sums round once per 32 channels and offset to fp32 (2^-24
of a partial sum, at random: under 4e-7 of the result's 2-norm for 27 x 256
products), the operands' parts lose under 2^-24 of a product: 1e-6."""
import numpy as np
import pytest
import torch

import oracle
from riemannengine_amd import abi
from helpers import DEV, gpu_tables_and_map, random_coords, to_dev

pytestmark = pytest.mark.gpu


def _map(n, off, seed, span):
    c, _, _ = oracle.insert_and_map(random_coords(np.random.default_rng(seed), 6 * n + 8, 3, span))
    assert len(c) >= n
    return gpu_tables_and_map(c[:n], c[:n], off, same=True)[2]


def _sums(rows_in, rows_out, kofs, x, w, n_out, transpose):
    """sum over pairs in float64; w [K, a, b], transposed for the gradient."""
    y = torch.zeros(n_out, w.shape[1] if transpose else w.shape[2], dtype=torch.float64)
    for k in range(w.shape[0]):
        s = slice(int(kofs[k]), int(kofs[k + 1]))
        wk = w[k].double().T if transpose else w[k].double()
        y.index_add_(0, rows_out[s].long(), x.double()[rows_in[s].long()] @ wk)
    return y


@pytest.mark.parametrize("n,ks,cin,cout,span", [
    (1, 3, 64, 64, 9), (127, 3, 64, 64, 4), (128, 3, 64, 96, 4), (129, 3, 96, 64, 4),
    (700, 3, 128, 128, 6), (300, 3, 192, 64, 5), (333, 3, 256, 160, 5), (260, 1, 64, 64, 5),
    (500, 2, 64, 128, 5), (200, 4, 64, 64, 4), (150, 5, 96, 96, 4), (12000, 3, 64, 64, 14)])
def test_x3_matches_64_bit_sums(n, ks, cin, cout, span):
    km = _map(n, oracle.region_offsets(3, ks), seed=n + ks, span=span)
    g = torch.Generator().manual_seed(cin + cout)
    x, gy = torch.randn(n, cin, generator=g), torch.randn(n, cout, generator=g)
    x *= torch.exp2(torch.randint(-20, 20, x.shape, generator=g).float())
    w = torch.randn(km.K, cin, cout, generator=g)
    b = torch.randn(cout, generator=g)
    print(f"x3 n={n} ks={ks} {cin}->{cout}", flush=True)
    y = abi.conv_forward(x.to(DEV), w.to(DEV), km, bias=b.to(DEV)).double().cpu()
    gx = abi.conv_backward_input(gy.to(DEV), w.to(DEV), km).double().cpu()
    ir, orr, kofs = km.in_rows.cpu(), km.out_rows.cpu(), km.offsets_host
    ry = _sums(ir, orr, kofs, x, w, n, False) + b.double()
    rgx = _sums(orr, ir, kofs, gy, w, n, True)
    assert (y - ry).norm() <= 1e-6 * ry.norm()
    assert (gx - rgx).norm() <= 1e-6 * rgx.norm()


@pytest.mark.parametrize("n,span", [(300, 5), (20000, 17)])  # split, whole
@pytest.mark.parametrize("where", ["x", "w"])
@pytest.mark.parametrize("bad", [float("inf"), float("nan"), 3.4e38])
def test_x3_keeps_values_that_are_not_finite(bad, where, n, span):
    """Infinities, NaN and magnitudes that round to infinity in bf16 give what
    fp32 sums over the pairs give: the same outputs finite, infinite and NaN,
    and the finite ones as close as ever."""
    km = _map(n, oracle.region_offsets(3, 3), seed=3, span=span)
    g = torch.Generator().manual_seed(7)
    x, w = torch.randn(n, 64, generator=g), torch.randn(27, 64, 64, generator=g) / 64
    if where == "x":
        x[n // 2, 3], x[5, 60] = bad, -bad
    else:
        w[4, 2, 9] = bad
    y = abi.conv_forward(x.to(DEV), w.to(DEV), km).cpu()
    ref = _sums(km.in_rows.cpu(), km.out_rows.cpu(), km.offsets_host, x, w, n, False).float()
    assert torch.equal(torch.isnan(y), torch.isnan(ref))
    inf = torch.isinf(ref)
    assert torch.equal(torch.isinf(y), inf) and torch.equal(y[inf], ref[inf])
    m = torch.isfinite(ref)
    assert (~m).any() or bad == 3.4e38
    scale = ref.abs().clamp(max=1e30)[m & (ref.abs() < 1e30)].norm()
    small = m & (ref.abs() < 1e30)
    assert (y[small] - ref[small]).norm() <= 1e-5 * scale
    big = m & ~small
    assert torch.allclose(y[big], ref[big], rtol=1e-5)


def _device_sums(km, x, w, transpose=False):
    """_sums on the device, in float64."""
    rin, rout = (km.out_rows, km.in_rows) if transpose else (km.in_rows, km.out_rows)
    y = torch.zeros(km.n_out, w.shape[1] if transpose else w.shape[2], dtype=torch.float64,
                    device=DEV)
    for k in range(w.shape[0]):
        s = slice(int(km.offsets_host[k]), int(km.offsets_host[k + 1]))
        wk = w[k].double()
        y.index_add_(0, rout[s].long(),
                     x[rin[s].long()].double() @ (wk.t().contiguous() if transpose else wk))
    return y


@pytest.mark.parametrize("n,cout", [(5000, 64), (14000, 256)])  # split, whole
@pytest.mark.parametrize("ex,ew", [(-112, 0), (-118, 0), (-124, 12), (-130, 20), (-140, 24),
                                   (0, -112), (10, -124), (20, -130), (-60, -50), (60, -100)])
def test_x3_keeps_the_bits_of_small_operands(n, cout, ex, ew):
    """Features, gradients and weights down to fp32's denormals (the inputs as
    fp32 holds them) give sums as exact as ordinary ones."""
    km = _map(n, oracle.region_offsets(3, 3), seed=n, span=18 if n > 9000 else 13)
    kernel, splits = abi.conv_plan(torch.float32, 27, 64, cout, n, n)
    assert kernel == "parts" and (splits > 1) == (n == 5000)
    g = torch.Generator(DEV).manual_seed(ex * 7 + ew)
    x, gy, w = (torch.randn(s, generator=g, device=DEV) for s in
                ((n, 64), (n, cout), (27, 64, cout)))
    x, gy, w = (torch.ldexp(t, torch.tensor(e, device=DEV)) for t, e in
                ((x, ex), (gy, ex), (w, ew)))
    assert all(bool((t != 0).float().mean() > 0.99) for t in (x, gy, w))
    print(f"x3 small n={n} cout={cout} 2^{ex} 2^{ew}", flush=True)
    for got, ref in ((abi.conv_forward(x, w, km), _device_sums(km, x, w)),
                     (abi.conv_backward_input(gy, w, km), _device_sums(km, gy, w, True))):
        assert float(ref.norm()) > 0
        # fp32's smallest step where the sums are that small
        step = 2.0 ** -149 * ref.numel() ** 0.5
        assert float((got.double() - ref).norm()) <= 1e-6 * float(ref.norm()) + step
