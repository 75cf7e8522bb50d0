"""Every tile of a map runs once whatever the run length the workgroups are
dealt to the XCDs in: the mapping itself for all small tile counts (on the
host), and convolutions with 16-, 64- and 128-row tiles and stride-map pooling
at row counts around each change of the run, 16 * 2^i tiles, where the padded
grid reaches the next one. A missing or doubled tile leaves rows of the
NaN-filled output or misplaces them."""
import os
import subprocess

import numpy as np
import pytest
import torch

from riemannengine_amd import abi
from riemannengine_amd import build as rbuild
from helpers import DEV, to_dev

TILES = (1, 2, 7, 8, 9, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 513,
         1100)


@pytest.mark.skipif(not os.path.exists(rbuild.HIPCC), reason="needs the compiler")
def test_mapping_is_a_bijection(tmp_path):
    """xcd_tile over the xcd_grid of 1 to 5,000 tiles: every tile once, the
    rest past the last, as a program of its own (host code only)."""
    src = tmp_path / "runs.cpp"
    src.write_text("""
#include <cstdio>
#include <vector>
#include "rhip_internal.hpp"
int main() {
  for (int64_t tiles = 1; tiles <= 5000; ++tiles) {
    const int64_t grid = rhip::xcd_grid(tiles);
    std::vector<int> seen(static_cast<size_t>(grid), 0);
    for (int64_t b = 0; b < grid; ++b) {
      const int64_t t = rhip::xcd_tile(static_cast<uint32_t>(b), static_cast<uint32_t>(grid));
      if (t < 0 || t >= grid || seen[static_cast<size_t>(t)]++) {
        std::printf("%lld tiles: id %lld\\n", (long long)tiles, (long long)b);
        return 1;
      }
    }
  }
  return 0;
}
""")
    exe = tmp_path / "runs"
    subprocess.run([rbuild.HIPCC, "-x", "hip", "--offload-host-only", "-std=c++17", "-O1", "-w",
                    "-I" + rbuild.INCLUDE, "-I" + rbuild.CSRC, str(src), "-o", str(exe)],
                   check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout


def _rows(n, step=1):
    c = np.zeros((n, 4), np.int32)
    c[:, 1], c[:, 2] = step * (np.arange(n) % 512), step * (np.arange(n) // 512)
    return c


# one offset finds every row itself, the others (out of the plane) nothing
@pytest.mark.gpu
@pytest.mark.parametrize("K,rows,width,dtype,kernels", [
    (33, 64, 16, torch.float32, ("tiled", "lds")), (33, 64, 16, torch.bfloat16, ("tiled",)),
    (33, 64, 32, torch.bfloat16, ("lds",)), (1, 16, 16, torch.float32, ("small",)),
    (33, 64, 64, torch.float32, ("parts",)), (1, 128, 128, torch.float32, ("parts",))])
def test_every_tile_of_a_convolution_runs_once(K, rows, width, dtype, kernels):
    offsets = np.zeros((K, 3), np.int32)
    offsets[:, 2] = np.arange(K)
    for tiles in TILES if rows < 128 else (1023, 1024, 1025):
        n = rows * tiles - 3
        assert abi.conv_plan(dtype, K, width, width, n, n)[0] in kernels
        t = abi.hash_build(to_dev(_rows(n)))
        km = abi.kernel_map(t, t, to_dev(offsets))
        # whole values: every product and sum is exact
        g = torch.Generator(DEV).manual_seed(tiles)
        x = torch.randint(-8, 9, (n, width), device=DEV, generator=g).to(dtype)
        w = torch.randint(-1, 2, (K, width, width), device=DEV, generator=g).to(dtype)
        y = torch.full((n, width), float("nan"), dtype=dtype, device=DEV)
        dt = abi._dtype_code(dtype)
        ws = abi._pass_ws(abi.PASS_FORWARD, K, width, width, dt, DEV, n, n)
        print(f"tile runs K={K} rows={rows} {width} {dtype} tiles={tiles}", flush=True)
        abi._check(abi.lib().rhip_conv_forward(
            abi._ptr(x), n, width, abi._ptr(w), K, width, None, abi._ptr(km.nbr),
            abi._ptr(km.out_order), n, abi._ptr(y), dt, abi._ptr(ws), ws.numel(),
            abi._stream(DEV)), "rhip_conv_forward")
        assert torch.equal(y, (x.double() @ w[0].double()).to(dtype)), tiles


@pytest.mark.gpu
def test_every_tile_of_a_pooling_runs_once():
    """Four fp32 channels: one lane a row, 256 rows a tile; every row is its
    own cell of the stride map."""
    for tiles in TILES:
        n = 256 * tiles - 3
        c = to_dev(_rows(n, step=2))
        tin = abi.hash_build(c)
        tout = abi.hash_build(abi.stride_coords(c, [2, 2, 2]))
        assert tin.n == tout.n == n
        sm = abi.stride_map(tin, tout, [2, 2, 2])
        x = torch.randn(n, 4, device=DEV)
        print(f"tile runs pooling tiles={tiles}", flush=True)
        for mode in ("sum", "max"):
            y = torch.full((n, 4), float("nan"), device=DEV)
            gx = torch.full((n, 4), float("nan"), device=DEV)
            counts = torch.full((n,), -1, dtype=torch.int32, device=DEV)
            m, st = abi._pool_mode(mode), abi._stream(DEV)
            abi._check(abi.lib().rhip_pool_forward(
                abi._ptr(x), n, 4, abi._ptr(sm.nbr), sm.nbr.shape[0], abi._ptr(sm.out_order), n, m,
                abi._ptr(y), abi._ptr(counts), abi.F32, st), "rhip_pool_forward")
            assert torch.equal(y, x) and bool((counts == 1).all()), tiles
            ws = torch.empty(abi._sizeq(abi.lib().rhip_pool_workspace_bytes, n, 4, m),
                             dtype=torch.uint8, device=DEV)
            abi._check(abi.lib().rhip_pool_backward(
                abi._ptr(x), abi._ptr(y), abi._ptr(x), n, 4, abi._ptr(sm.nbr), sm.nbr.shape[0],
                abi._ptr(sm.out_order), abi._ptr(sm.nbr_t), sm.nbr_t.shape[0],
                abi._ptr(sm.in_order), n, abi._ptr(counts), m, abi._ptr(gx), abi.F32,
                abi._ptr(ws), ws.numel(), st), "rhip_pool_backward")
            assert torch.equal(gx, x), tiles
