"""Maps with few rows: forward with bias and input gradient of the kernel
whose waves share out a 16-row tile's stages, against the oracle at its edges
(16 rows, 16 / 32 / 64 columns, one chunk or several, fewer stages than waves,
1 to 32 offsets, both weight layouts; in bf16 1^D layers and directions that
reduce an odd multiple of 16 channels run on others). Tolerance: norm-wise rel 1e-4 for fp32
and 2e-2 for bf16 (helpers.TOL)."""
import numpy as np
import pytest
import torch

import oracle
from riemannengine_amd import abi
from helpers import TOL, assert_rel, gpu_tables_and_map, random_coords, to_dev


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,off,cin,cout", [
    (1, (3, 3), 32, 16), (15, (3, 3), 16, 32), (16, (3, 1), 64, 64), (17, (3, 3), 32, 48),
    (33, (3, 3), 96, 32), (200, (3, 2), 32, 64), (500, (3, 3), 64, 64), (900, (2, 5), 32, 32),
    (130, (5, 2), 32, 80), (700, (3, 3), 256, 16), (2100, (3, 3), 32, 32)])
def test_small_map_layers_match_oracle(n, off, cin, cout, dtype):
    D, ks = off
    rng = np.random.default_rng(n + cin)
    span = 30 if D == 2 else (3 if D == 5 else 6)
    c, _, _ = oracle.insert_and_map(random_coords(rng, 6 * n + 8, D, span))
    km = gpu_tables_and_map(c[:n], c[:n], oracle.region_offsets(D, ks), same=True)[2]
    x, gy = (to_dev(rng.standard_normal((n, k)).astype(np.float32), dtype) for k in (cin, cout))
    w = to_dev((rng.standard_normal((km.K, cin, cout)) / 20).astype(np.float32), dtype)
    b = rng.standard_normal(cout).astype(np.float32)
    plans = [abi.conv_plan(dtype, km.K, cin, cout, n, n)[0],
             abi.conv_plan(dtype, km.K, cout, cin, n, n, True)[0]]
    odd = [dtype == torch.bfloat16 and c % 32 != 0 for c in (cin, cout)]
    small = "lds" if dtype == torch.bfloat16 and km.K < 8 else "small"
    assert plans == ["tiled" if o else small for o in odd]
    print(f"small n={n} K={km.K} {cin}->{cout} {dtype}", flush=True)
    y, gx = abi.conv_forward(x, w, km, bias=to_dev(b)), abi.conv_backward_input(gy, w, km)
    kofs, ir, orr = km.offsets_host, km.in_rows.cpu().numpy(), km.out_rows.cpu().numpy()
    xs, gs, ws = (t.float().cpu().numpy() for t in (x, gy, w))
    assert_rel(y.float().cpu().numpy(), oracle.conv_forward(xs, ws, kofs, ir, orr, n) + b,
               TOL[dtype], "Y")
    assert_rel(gx.float().cpu().numpy(), oracle.conv_backward(xs, gs, ws, kofs, ir, orr)[0],
               TOL[dtype], "dX")
    assert torch.equal(y, abi.conv_forward(x, w, km, bias=to_dev(b)))


def test_small_map_dispatch_without_a_gpu():
    """Where the small-map kernel stops: rows, the weights its workgroups read
    together, and 1^D layers, which have no chain of stages to share out."""
    def name(dtype, *a):  # of the forward and the input gradient
        f, dx = abi.conv_plan(dtype, *a)[0], abi.conv_plan(dtype, *a, True)[0]
        return f if f == dx else (f, dx)

    f32, bf16 = torch.float32, torch.bfloat16
    assert name(f32, 27, 32, 32, 10000, 10000) == "small" == name(bf16, 27, 32, 32, 10000, 10000)
    assert name(f32, 27, 16, 16, 40000, 40000) == "small" != name(f32, 27, 16, 16, 40001, 40001)
    assert name(f32, 27, 64, 64, 4900, 4900) != "small" != name(bf16, 27, 64, 64, 4900, 4900)
    assert name(f32, 1, 192, 192, 3113, 3113) == "small" == name(f32, 1, 32, 32, 20000, 20000)
    assert name(f32, 1, 64, 64, 20000, 20000)[0] == "small" != name(f32, 1, 64, 64, 20000, 20000)[1]
    assert name(f32, 1, 128, 64, 48231, 48231) != "small"
    assert name(bf16, 1, 32, 32, 1000, 1000) == "lds"
    assert name(f32, 8, 64, 64, 48231, 10850) == "small"
    assert name(f32, 8, 16, 16, 12000, 60000) == ("small", "lds")
