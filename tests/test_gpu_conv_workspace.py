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
from helpers import DEV, TOL, gpu_tables_and_map, random_coords, reference_passes, to_dev

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
                    for dx, n_rows, cred, ncols, n_x in ((False, m, cin, cout, n),
                                                         (True, n, cout, cin, m)):
                        _, sp = abi.conv_plan(dtype, K, cred, ncols, n_x, n_rows, dx)
                        assert sp == 1 or sp * n_rows * ncols * 4 <= room, (K, cin, cout, n)


def test_workspace_counts_the_padded_reduction():
    """112 channels run as 128: 13 stages per split instead of 6, so eight
    splits of 8,000 rows."""
    assert _forward_bytes(27, 112, 128, abi.BF16, 8000, 8000) >= 8 * 8000 * 128 * 4
    assert abi.conv_plan(torch.bfloat16, 27, 112, 128, 8000, 8000) == ("tiled", 8)
    # 96 columns of a padded reduction run in 32-column tiles: enough of them
    assert abi.conv_plan(torch.bfloat16, 27, 48, 96, 30000, 30000) == ("tiled", 1)


def _pass_bytes(passes, K, cin, cout, dt, n_in, n_out):
    return abi._sizeq(abi.lib().rhip_conv_pass_workspace_bytes, passes, K, cin, cout, dt, n_in,
                      n_out, n_out)


def test_workspace_reserves_only_what_the_call_uses():
    # a first layer's forward and its weight gradient need no padded copies
    stem = _pass_bytes(abi.PASS_FORWARD, 27, 3, 32, abi.F32, 10**7, 10**7)
    assert stem <= 1024
    assert _pass_bytes(abi.PASS_WEIGHT_GRAD, 27, 3, 32, abi.F32, 10**7, 10**7) < 8 << 20
    # no pass of a 1^3 classifier does
    head = abi._sizeq(abi.lib().rhip_conv_workspace_bytes, 1, 64, 20, abi.F32, 10**6, 10**6, 10**6)
    assert head < 8 << 20
    # 30,000 rows of 32 channels are not split
    assert abi.conv_plan(torch.float32, 27, 32, 64, 30000, 30000)[1] == 1
    assert _forward_bytes(27, 32, 64, abi.F32, 30000, 30000) < 1 << 20
    # the bias gradient: 256 chunk sums whatever the layer
    assert _pass_bytes(abi.PASS_BIAS_GRAD, 1, 1, 20, abi.F32, 0, 10**6) <= 256 * 20 * 4 + 1024
    # the queries for several passes cover each
    for shape in ((27, 24, 40), (27, 64, 64), (1, 64, 20), (27, 48, 96), (8, 64, 128)):
        for dt in (abi.F32, abi.BF16):
            one = [_pass_bytes(p, *shape, dt, 30000, 20000) for p in (1, 2, 4, 8)]
            assert _pass_bytes(15, *shape, dt, 30000, 20000) == max(one)
            full = abi._sizeq(abi.lib().rhip_conv_workspace_bytes, *shape, dt, 30000, 20000, 20000)
            assert full >= max(one) and _forward_bytes(*shape, dt, 30000, 20000) >= max(one[:3])
    st = abi.lib().rhip_conv_pass_workspace_bytes(16, 27, 3, 32, abi.F32, 1, 1, 1,
                                                  abi.ctypes.byref(abi.ctypes.c_size_t(0)))
    assert st != 0


F32, BF16 = torch.float32, torch.bfloat16


@pytest.mark.gpu
@pytest.mark.parametrize("n,cin,cout,dtype,kernel", [
    (8000, 48, 96, BF16, "tiled"), (20000, 48, 96, BF16, "tiled"), (30000, 48, 96, BF16, "tiled"),
    (50000, 48, 96, BF16, "tiled"), (20000, 48, 192, BF16, "tiled"),
    (8000, 112, 128, BF16, "tiled"), (20000, 112, 128, BF16, "tiled"),
    (9000, 80, 96, BF16, "tiled"), (9000, 176, 96, BF16, "tiled"), (5000, 240, 256, BF16, "tiled"),
    (9000, 96, 96, BF16, "lds"), (9000, 160, 96, BF16, "tiled"), (9000, 128, 128, BF16, "lds"),
    (900, 3, 32, F32, "thin"), (900, 24, 40, F32, "padded"), (900, 40, 64, BF16, "padded"),
    (20000, 64, 40, F32, "padded"), (900, 32, 32, F32, "small"), (900, 32, 64, BF16, "small"),
    (9000, 64, 96, F32, "parts"), (9000, 48, 48, F32, "tiled"), (60000, 64, 64, F32, "parts")])
def test_calls_stay_in_their_workspace(n, cin, cout, dtype, kernel):
    """Each pass in a workspace of its own size, the bytes behind it kept."""
    rng = np.random.default_rng(n + cin)
    c, _, _ = oracle.insert_and_map(random_coords(rng, 4 * n, 3, int(round((2 * n) ** (1 / 3)))))
    km = gpu_tables_and_map(c[:n], c[:n], oracle.region_offsets(3, 3), same=True)[2]
    assert km.n_in == n and abi.conv_plan(dtype, 27, cin, cout, n, n)[0] == kernel
    x, gy, w = (to_dev(rng.standard_normal(s).astype(np.float32), dtype)
                for s in ((n, cin), (n, cout), (27, cin, cout)))
    dt, L, st, p = abi._dtype_code(dtype), abi.lib(), abi._stream(DEV), abi._ptr
    print(f"workspace n={n} {cin}->{cout} {dtype}", flush=True)
    y, gx, gw = torch.empty_like(gy), torch.empty_like(x), torch.empty_like(w)

    def call(passes, fn, args):
        room = abi._sizeq(L.rhip_conv_pass_workspace_bytes, passes, 27, cin, cout, dt, n, n,
                          km.n_pairs)
        buf = torch.full((room + (64 << 20),), 0xA5, dtype=torch.uint8, device=DEV)
        rc = fn(*args, dt, p(buf), room, st)
        assert bool((buf[room:] == 0xA5).all())
        return rc

    table, perm, order = p(km.nbr), p(km.partner), p(km.out_order)
    abi._check(call(abi.PASS_FORWARD, L.rhip_conv_forward,
                    (p(x), n, cin, p(w), 27, cout, None, table, order, n, p(y))), "forward")
    abi._check(call(abi.PASS_INPUT_GRAD, L.rhip_conv_backward_input,
                    (p(gy), n, cout, p(w), 27, cin, table, perm, order, n, p(gx))), "dX")
    dw = (p(x), n, cin, p(gy), n, cout, 27, table, order, p(gw))
    rc = call(abi.PASS_WEIGHT_GRAD, L.rhip_conv_backward_weight_rows, dw)
    if rc == abi.RHIP_ERR_UNSUPPORTED:
        rc = call(abi.PASS_WEIGHT_GRAD, L.rhip_conv_backward_weight_ragged, dw)
    if rc == abi.RHIP_ERR_UNSUPPORTED:
        rc = call(abi.PASS_WEIGHT_GRAD, L.rhip_conv_backward_weight,
                  (p(x), n, cin, p(gy), n, cout, 27, p(km.offsets), km.n_pairs, p(km.in_rows),
                   p(km.out_rows), p(gw)))
    abi._check(rc, "dW")
    for got, ref in zip((y, gx, gw), reference_passes(km, x, gy, w)):
        assert float((got.float() - ref).abs().max()) <= TOL[dtype] * float(ref.abs().max())
