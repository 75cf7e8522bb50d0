"""fp32 forward and input gradient on three-part bf16 operands: against 64-bit
sums at the edges of its tiles (128 rows up to 32 offsets, else 64; 64 or 32
columns; one, three or four mask words), every reduction width, split and
whole offset axes, down to fp32's smallest values, and with values no bf16 part
can hold. Each case names the kernel it is meant for (rhip_conv_plan). Some
cases below its row limit run on the small-map kernel instead, on fp32 sums.
Tolerance: the sums round once per 32 channels and offset to fp32 (2^-24 of a
partial sum, at random: under 4e-7 of the result's 2-norm for 27 x 256
products), the operands' parts lose under 2^-24 of a product: 1e-6."""
import numpy as np
import pytest
import torch

import oracle
from riemannengine_amd import abi
from helpers import DEV, gpu_tables_and_map, random_coords


def _map(n, off, seed, span):
    c, _, _ = oracle.insert_and_map(random_coords(np.random.default_rng(seed), 6 * n + 8, 3, span))
    assert len(c) >= n
    return gpu_tables_and_map(c[:n], c[:n], off, same=True)[2]


def _device_sums(km, x, w, transpose=False):
    """The sums over the pairs in float64; transposed: the input gradient's."""
    rin, rout = (km.out_rows, km.in_rows) if transpose else (km.in_rows, km.out_rows)
    y = torch.zeros(km.n_out, w.shape[1] if transpose else w.shape[2], dtype=torch.float64,
                    device=DEV)
    for k in range(w.shape[0]):
        s = slice(int(km.offsets_host[k]), int(km.offsets_host[k + 1]))
        wk = w[k].double()
        y.index_add_(0, rout[s].long(),
                     x[rin[s].long()].double() @ (wk.t().contiguous() if transpose else wk))
    return y


def _kernel(K, cred, ncols, n, dx=False):
    name, splits = abi.conv_plan(torch.float32, K, cred, ncols, n, n, dx)
    return name + (" split" if splits > 1 else "")


# fwd, dx: the kernels of the forward and of the input gradient
@pytest.mark.gpu
@pytest.mark.parametrize("n,ks,cin,cout,span,fwd,dx", [
    # split: rows at and around a 128-row tile's edges, both column tiles, every width
    (3711, 3, 64, 64, 11, "parts split", "parts split"),
    (3712, 3, 64, 96, 11, "parts split", "parts split"),
    (3713, 3, 96, 64, 11, "parts split", "parts split"),
    (1023, 3, 128, 128, 8, "parts split", "parts split"),
    (1281, 3, 192, 64, 8, "parts split", "parts split"),
    (257, 3, 256, 256, 5, "parts split", "parts split"),
    (640, 3, 256, 160, 7, "parts split", "tiled split"),
    (1000, 3, 160, 128, 8, "tiled split", "parts split"),
    (6145, 2, 64, 128, 13, "parts split", "parts split"),
    (11009, 3, 64, 160, 15, "parts split", "tiled split"),
    (18303, 3, 192, 96, 17, "parts split", "parts"),
    # whole
    (55041, 3, 64, 64, 24, "parts", "parts"), (22017, 3, 96, 160, 18, "parts", "tiled"),
    (36481, 3, 96, 192, 21, "parts", "parts"), (13825, 3, 128, 256, 15, "parts", "parts split"),
    (13697, 3, 192, 256, 15, "parts", "parts split"), (13696, 3, 256, 256, 15, "parts", "parts"),
    (98433, 1, 128, 128, 29, "parts", "parts"),
    # three and four mask words: 64-row tiles
    (191, 4, 64, 64, 5, "parts split", "parts split"),
    (192, 4, 128, 64, 5, "parts split", "parts split"),
    (193, 4, 64, 96, 5, "parts split", "parts split"),
    (27457, 4, 64, 64, 19, "parts", "parts"),
    (63, 5, 64, 192, 4, "parts split", "parts split"),
    (150, 5, 96, 96, 4, "parts split", "parts split"),
    (129, 5, 256, 64, 4, "parts split", "parts split"),
    # small maps
    (1, 3, 64, 64, 9, "small", "small"), (129, 3, 96, 64, 4, "small", "small"),
    (260, 1, 64, 64, 5, "small", "small"), (300, 3, 192, 64, 5, "small", "small")])
def test_x3_matches_64_bit_sums(n, ks, cin, cout, span, fwd, dx):
    km = _map(n, oracle.region_offsets(3, ks), seed=n + ks, span=span)
    assert (_kernel(km.K, cin, cout, n), _kernel(km.K, cout, cin, n, True)) == (fwd, dx)
    g = torch.Generator(DEV).manual_seed(cin + cout)
    x, gy, w, b = (torch.randn(s, generator=g, device=DEV) for s in
                   ((n, cin), (n, cout), (km.K, cin, cout), (cout,)))
    x *= torch.exp2(torch.randint(-20, 20, x.shape, generator=g, device=DEV).float())
    print(f"x3 n={n} ks={ks} {cin}->{cout} {fwd} / {dx}", flush=True)
    y = abi.conv_forward(x, w, km, bias=b).double()
    gx = abi.conv_backward_input(gy, w, km).double()
    ry, rgx = _device_sums(km, x, w) + b.double(), _device_sums(km, gy, w, True)
    # the fp32 matrix cores round once per 4 channels and offset
    tol = [1e-6 if k.startswith("parts") else 4e-6 for k in (fwd, dx)]
    assert float((y - ry).norm()) <= tol[0] * float(ry.norm())
    assert float((gx - rgx).norm()) <= tol[1] * float(rgx.norm())


@pytest.mark.gpu
@pytest.mark.parametrize("n,span,kernel", [(300, 5, "small"), (20000, 17, "parts split"),
                                           (55041, 24, "parts")])
@pytest.mark.parametrize("where", ["x", "w"])
@pytest.mark.parametrize("bad", [float("inf"), float("nan"), 3.4e38])
def test_x3_keeps_values_that_are_not_finite(bad, where, n, span, kernel):
    """Infinities, NaN and magnitudes that round to infinity in bf16 give what
    fp32 sums over the pairs give: the same outputs finite, infinite and NaN,
    and the finite ones as close as ever."""
    km = _map(n, oracle.region_offsets(3, 3), seed=3, span=span)
    assert _kernel(27, 64, 64, n) == kernel
    g = torch.Generator().manual_seed(7)
    x, w = torch.randn(n, 64, generator=g), torch.randn(27, 64, 64, generator=g) / 64
    if where == "x":
        x[n // 2, 3], x[5, 60] = bad, -bad
    else:
        w[4, 2, 9] = bad
    y = abi.conv_forward(x.to(DEV), w.to(DEV), km).cpu()
    ref = _device_sums(km, x.to(DEV), w.to(DEV)).float().cpu()
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


@pytest.mark.gpu
@pytest.mark.parametrize("n,cout", [(5000, 64), (14000, 256)])  # split, whole
@pytest.mark.parametrize("ex,ew", [(-112, 0), (-118, 0), (-124, 12), (-130, 20), (-140, 24),
                                   (0, -112), (10, -124), (20, -130), (-60, -50), (60, -100)])
def test_x3_keeps_the_bits_of_small_operands(n, cout, ex, ew):
    """Features, gradients and weights down to fp32's denormals (the inputs as
    fp32 holds them) give sums as exact as ordinary ones."""
    km = _map(n, oracle.region_offsets(3, 3), seed=n, span=18 if n > 9000 else 13)
    assert _kernel(27, 64, cout, n) == ("parts split" if n == 5000 else "parts")
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


def test_x3_dispatch_without_a_gpu():
    """Where the three-part kernel stops: narrow layers, part-empty column tiles
    on large maps, stride-2 maps and 1^3 layers with little work."""
    f32 = torch.float32

    def name(*a):
        return abi.conv_plan(f32, *a)[0]

    assert name(27, 64, 64, 10000, 10000) == "parts" and name(27, 32, 64, 10000, 10000) != "parts"
    assert name(27, 64, 48, 99999, 99999) != "parts"
    assert name(27, 64, 96, 20480, 20480) == "parts" and name(27, 64, 96, 20481, 20481) != "parts"
    assert name(27, 96, 96, 99999, 99999) == "parts" and name(27, 160, 64, 9999, 9999) != "parts"
    # a stride-2 map and its transpose: channels, work, one neighbour a row
    assert name(8, 128, 128, 48231, 10850) == "parts" and name(8, 64, 128, 48231, 10850) != "parts"
    assert name(8, 128, 128, 23086, 5100) != "parts"
    assert name(8, 256, 128, 10850, 48231) == "parts" and name(8, 256, 128, 8663, 37452) != "parts"
    assert name(8, 192, 192, 5100, 23086) == "parts" != name(8, 192, 192, 5100, 23086, True)
    assert name(1, 128, 128, 50000, 50000) == "parts" and name(1, 64, 64, 409553, 409553) != "parts"
    assert name(8, 64, 64, 50000, 50000) == "parts"  # 2^3 at stride 1: several pairs a row
