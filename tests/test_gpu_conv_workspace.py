"""The workspace of a convolution's forward and input gradient holds what the
launches write: the split partial sums of every channel count, among them bf16
reductions of 16 more than a multiple of 32 (padded by 16, so that the width
the stages are counted in is not the layer's), and nothing is written past its
end. Outputs against fp32 products per offset at helpers.TOL."""
import numpy as np
import pytest
import torch

import oracle
from riemannengine_amd import abi
from helpers import DEV, TOL, gpu_tables_and_map, random_coords, to_dev

WIDTHS = (16, 32, 48, 64, 80, 96, 112, 128, 144, 160, 176, 192, 240, 256, 288, 384)


def _forward_bytes(K, cin, cout, dt, n_in, n_out):
    return abi._sizeq(abi.lib().rhip_conv_forward_workspace_bytes, K, cin, cout, dt, n_in, n_out)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_workspace_holds_the_split_sums(dtype):
    dt = abi._dtype_code(dtype)
    for K in (8, 27, 125):
        for cin in WIDTHS:
            for cout in WIDTHS:
                for n in (500, 8000, 20000, 30000, 50000, 90000):
                    m = n // 3
                    room = _forward_bytes(K, cin, cout, dt, n, m)
                    for n_rows, cred, ncols, n_x in ((m, cin, cout, n), (n, cout, cin, m)):
                        _, sp = abi.conv_plan(dtype, K, cred, ncols, n_x, n_rows)
                        assert sp == 1 or sp * n_rows * ncols * 4 <= room, (K, cin, cout, n)


def test_workspace_counts_the_padded_reduction():
    """112 channels run as 128: 13 stages per split instead of 6, so eight
    splits of 8,000 rows."""
    assert _forward_bytes(27, 112, 128, abi.BF16, 8000, 8000) >= 8 * 8000 * 128 * 4
    assert abi.conv_plan(torch.bfloat16, 27, 112, 128, 8000, 8000) == ("tiled", 8)
    # 96 columns of a padded reduction run in 32-column tiles: enough of them
    assert abi.conv_plan(torch.bfloat16, 27, 48, 96, 30000, 30000) == ("tiled", 1)


@pytest.mark.gpu
@pytest.mark.parametrize("n,cin,cout", [
    (8000, 48, 96), (20000, 48, 96), (30000, 48, 96), (50000, 48, 96), (20000, 48, 192),
    (8000, 112, 128), (20000, 112, 128), (9000, 80, 96), (9000, 176, 96), (5000, 240, 256)])
def test_padded_reductions_stay_in_their_workspace(n, cin, cout):
    rng = np.random.default_rng(n + cin)
    c, _, _ = oracle.insert_and_map(random_coords(rng, 4 * n, 3, int(round((2 * n) ** (1 / 3)))))
    km = gpu_tables_and_map(c[:n], c[:n], oracle.region_offsets(3, 3), same=True)[2]
    assert km.n_in == n
    x, gy, w = (to_dev(rng.standard_normal(s).astype(np.float32), torch.bfloat16)
                for s in ((n, cin), (n, cout), (27, cin, cout)))
    print(f"workspace n={n} {cin}->{cout}", flush=True)
    room = _forward_bytes(27, cin, cout, abi.BF16, n, n)
    buf = torch.full((room + (64 << 20),), 0xA5, dtype=torch.uint8, device=DEV)
    L, st = abi.lib(), abi._stream(DEV)
    y, gx = torch.empty(n, cout, **_bf16()), torch.empty(n, cin, **_bf16())
    abi._check(L.rhip_conv_forward(abi._ptr(x), n, cin, abi._ptr(w), 27, cout, None,
                                   abi._ptr(km.nbr), abi._ptr(km.out_order), n, abi._ptr(y),
                                   abi.BF16, abi._ptr(buf), room, st), "forward")
    assert bool((buf[room:] == 0xA5).all())
    abi._check(L.rhip_conv_backward_input(abi._ptr(gy), n, cout, abi._ptr(w), 27, cin,
                                          abi._ptr(km.nbr), abi._ptr(km.partner),
                                          abi._ptr(km.out_order), n, abi._ptr(gx), abi.BF16,
                                          abi._ptr(buf), room, st), "input gradient")
    assert bool((buf[room:] == 0xA5).all())
    ry, rgx = (torch.zeros(n, k, device=DEV) for k in (cout, cin))
    for k in range(27):
        s = slice(int(km.offsets_host[k]), int(km.offsets_host[k + 1]))
        ir, orr, wk = km.in_rows[s].long(), km.out_rows[s].long(), w[k].float()
        ry.index_add_(0, orr, x[ir].float() @ wk)
        rgx.index_add_(0, ir, gy[orr].float() @ wk.t().contiguous())
    for got, ref in ((y, ry), (gx, rgx)):
        assert float((got.float() - ref).abs().max()) <= TOL[torch.bfloat16] * float(
            ref.abs().max())


def _bf16():
    return {"dtype": torch.bfloat16, "device": DEV}
