"""Every tile of a map runs once whatever the run length the workgroups are
dealt to the XCDs in: 1^3 layers (one offset, every row its own neighbour)
and stride-map pooling at row counts around each change of the run, where
the padded grid reaches the next one. A missing or doubled tile leaves rows
of the poisoned output or misplaces them."""
import numpy as np
import pytest
import torch

from riemannengine_amd import abi
from helpers import DEV, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tiles", [1, 2, 7, 8, 9, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511,
                                   513, 1023, 1024, 1025, 1100])
def test_every_tile_runs_once(tiles):
    n = 64 * tiles - 3
    c = np.zeros((n, 4), np.int32)
    c[:, 1], c[:, 2] = np.arange(n) % 512, np.arange(n) // 512
    t = abi.hash_build(to_dev(c))
    km = abi.kernel_map(t, t, to_dev(np.zeros((1, 3), np.int32)))
    # whole values below 2^8: every product and sum is exact
    x = torch.randint(-8, 9, (n, 16), device=DEV, generator=torch.Generator(DEV).manual_seed(tiles))
    w = torch.randint(-3, 4, (1, 16, 16), device=DEV)
    for dtype in (torch.float32, torch.bfloat16):
        y = abi.conv_forward(x.to(dtype), w.to(dtype), km)
        ref = (x.double() @ w[0].double()).to(dtype)
        assert torch.equal(y, ref), (tiles, dtype)
        torch.full_like(y, float("nan"))  # the next output's memory, poisoned
