"""bf16 layers of 96 and 192 channels: 96-column tiles, 96-channel stages and
the shared-row dW with a last chunk or tile part empty, against the oracle at
the edges of their tiles (64 and 128 rows), whole and split offset axes, one
and three mask words. Tolerance: norm-wise rel 2e-2 (helpers.TOL)."""
import numpy as np
import pytest
import torch

import oracle
from riemannengine_amd import abi
from helpers import TOL, assert_rel, gpu_tables_and_map, random_coords, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ks,cin,cout", [
    (1, 3, 96, 96), (64, 3, 96, 32), (65, 3, 32, 96), (128, 3, 96, 64), (129, 3, 96, 96),
    (500, 3, 192, 192), (700, 3, 64, 192), (300, 3, 128, 96), (257, 3, 96, 128), (300, 2, 96, 192),
    (200, 4, 96, 96), (400, 1, 96, 96), (300, 3, 160, 96), (300, 3, 96, 16)])
def test_96_channel_layers_match_oracle(n, ks, cin, cout):
    rng = np.random.default_rng(n + cin)
    c, _, _ = oracle.insert_and_map(random_coords(rng, 4 * n + 8, 3, 6))
    km = gpu_tables_and_map(c[:n], c[:n], oracle.region_offsets(3, ks), same=True)[2]
    x, gy, w = (to_dev(rng.standard_normal(s).astype(np.float32), torch.bfloat16)
                for s in ((n, cin), (n, cout), (km.K, cin, cout)))
    kofs, ir, orr = km.offsets_host, km.in_rows.cpu().numpy(), km.out_rows.cpu().numpy()
    xs, gs, ws = (t.float().cpu().numpy() for t in (x, gy, w))
    rgx, rgw = oracle.conv_backward(xs, gs, ws, kofs, ir, orr)
    print(f"96 n={n} ks={ks} {cin}->{cout}", flush=True)
    for name, got, ref in (
            ("Y", abi.conv_forward(x, w, km), oracle.conv_forward(xs, ws, kofs, ir, orr, n)),
            ("dX", abi.conv_backward_input(gy, w, km), rgx),
            ("dW", abi.conv_weight_grad(x, gy, km, km.K), rgw)):
        assert_rel(got.float().cpu().numpy(), ref, TOL[torch.bfloat16], name)


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
