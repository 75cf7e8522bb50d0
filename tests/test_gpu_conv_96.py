"""bf16 layers of 96 and 192 channels: 96-column tiles with one, two and three
chunks per stage, 96-channel stages with every column tile, and the shared-row
dW with a last chunk or tile part empty, at the edges of their tiles (64 and
128 rows), split and whole offset axes, one and three mask words. Each case
names the kernels it is meant for (rhip_conv_plan); the padded and the odd
reductions into 96 columns run on the general kernel, small maps on their own.
Against fp32 products per offset; tolerance: norm-wise rel 2e-2 (helpers.TOL)."""
import numpy as np
import pytest
import torch

import oracle
from riemannengine_amd import abi
from helpers import TOL, assert_rel, gpu_tables_and_map, random_coords, reference_passes, to_dev


def _kernel(K, cred, ncols, n, dx=False):
    name, splits = abi.conv_plan(torch.bfloat16, K, cred, ncols, n, n, dx)
    return name + (" split" if splits > 1 else "")


@pytest.mark.gpu
@pytest.mark.parametrize("n,ks,cin,cout,fwd,dx", [
    # split, 3^3: rows at and around 64- and 128-row tiles
    (1343, 3, 96, 96, "lds split", "lds split"), (1344, 3, 96, 96, "lds split", "lds split"),
    (1409, 3, 96, 96, "lds split", "lds split"), (3905, 3, 32, 96, "lds split", "lds split"),
    (2048, 3, 64, 96, "lds split", "lds split"), (2047, 3, 96, 64, "lds split", "lds split"),
    (500, 3, 192, 192, "lds split", "lds split"), (1025, 3, 64, 192, "lds split", "lds split"),
    (1088, 3, 128, 96, "lds split", "lds split"), (640, 3, 256, 96, "lds split", "lds split"),
    (2113, 3, 192, 32, "lds split", "lds split"), (7745, 3, 16, 96, "tiled split", "lds split"),
    (2177, 2, 96, 192, "lds split", "lds split"),
    # whole
    (54657, 3, 96, 96, "lds", "lds"), (54655, 3, 128, 96, "lds", "lds"),
    (54656, 3, 64, 96, "lds", "lds"), (27329, 3, 32, 96, "lds", "lds"),
    (27327, 3, 192, 192, "lds", "lds"), (13697, 3, 32, 192, "lds", "lds split"),
    (35009, 1, 96, 96, "lds", "lds"), (54657, 3, 192, 128, "lds", "lds"),
    (27329, 3, 192, 256, "lds", "lds"),
    # three mask words
    (200, 4, 96, 96, "lds split", "lds split"), (129, 4, 192, 64, "lds split", "lds split"),
    # padded and odd reductions into 96 columns
    (5000, 3, 48, 96, "tiled split", "lds split"), (9104, 3, 80, 96, "tiled", "lds"),
    (900, 3, 160, 96, "tiled split", "lds split"), (9105, 3, 160, 96, "tiled", "lds"),
    # small maps
    (1, 3, 96, 96, "small", "small"), (129, 3, 96, 96, "small", "small"),
    (64, 3, 96, 32, "small", "small"), (300, 3, 96, 16, "small", "tiled split")])
def test_96_channel_layers_match_products(n, ks, cin, cout, fwd, dx):
    rng = np.random.default_rng(n + cin)
    span = max(4, int(round((2 * n) ** (1 / 3))))
    c, _, _ = oracle.insert_and_map(random_coords(rng, 4 * n + 8, 3, span))
    km = gpu_tables_and_map(c[:n], c[:n], oracle.region_offsets(3, ks), same=True)[2]
    assert km.n_in == n
    assert (_kernel(km.K, cin, cout, n), _kernel(km.K, cout, cin, n, True)) == (fwd, dx)
    x, gy, w = (to_dev(rng.standard_normal(s).astype(np.float32), torch.bfloat16)
                for s in ((n, cin), (n, cout), (km.K, cin, cout)))
    print(f"96 n={n} ks={ks} {cin}->{cout} {fwd} / {dx}", flush=True)
    got = (abi.conv_forward(x, w, km), abi.conv_backward_input(gy, w, km),
           abi.conv_weight_grad(x, gy, km, km.K))
    for name, a, ref in zip(("Y", "dX", "dW"), got, reference_passes(km, x, gy, w)):
        assert_rel(a.float().cpu().numpy(), ref.cpu().numpy(), TOL[torch.bfloat16], name)


@pytest.mark.gpu
@pytest.mark.parametrize("n,cin,cout", [
    (66001, 96, 96), (30000, 192, 96), (5000, 224, 160), (40001, 80, 224), (30001, 160, 96),
    (9000, 96, 96), (70000, 64, 96)])
def test_weight_gradient_with_part_empty_tiles(n, cin, cout):
    """Channel counts that are no multiples of 64, on either side of where the
    shared-row kernel takes over, against the pair-list kernel (the same
    products in another order; both sum in fp32, the result rounds to bf16
    once: 2^-8)."""
    rng = np.random.default_rng(1)
    c, _, _ = oracle.insert_and_map(random_coords(rng, 100000, 3, 30))
    km = gpu_tables_and_map(c[:n], c[:n], oracle.region_offsets(3, 3), same=True)[2]
    x, gy = (to_dev(rng.standard_normal((n, k)).astype(np.float32), torch.bfloat16)
             for k in (cin, cout))
    got, ref = abi.conv_weight_grad(x, gy, km, 27), abi.conv_backward_weight(x, gy, km, 27)
    assert_rel(got.float().cpu().numpy(), ref.float().cpu().numpy(), 2 ** -8, "dW")
    assert torch.equal(got, abi.conv_weight_grad(x, gy, km, 27))


def test_96_column_tiles_without_a_gpu():
    """Short reductions take the narrower tiles where 96-column ones would be
    split; 192 columns that the kernel with 96-column tiles does not take run
    in 64-column ones."""
    bf16 = torch.bfloat16
    for n in (10000, 23086):
        assert abi.conv_plan(bf16, 27, 32, 96, n, n) == ("lds", 1)
    assert abi.conv_plan(bf16, 27, 64, 96, 23086, 23086) == ("lds", 1)
    assert abi.conv_plan(bf16, 27, 96, 96, 10000, 10000)[1] > 1
    assert abi.conv_plan(bf16, 27, 64, 192, 10000, 10000)[1] > 1
    for cred, ncols in ((192, 96), (96, 192), (192, 192)):  # a transposed stride-2 map
        assert abi.conv_plan(bf16, 8, cred, ncols, 5100, 23086) == ("lds", 1)
    assert abi.conv_plan(bf16, 27, 48, 192, 5036, 5036) == ("tiled", 3)
