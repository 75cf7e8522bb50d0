"""Kernel maps over tables without a brick grid (coordinates too spread for
one), whose neighbours the mask pass keeps and a permutation reads back:
bit-exact pairs and tables against the oracle for the strides of the kept rows
(1 to 32 offsets), strided and symmetric maps, two rows to several waves."""
import ctypes

import numpy as np
import pytest

import oracle
from riemannengine_amd import abi
from helpers import gpu_canonical, gpu_tables_and_map, random_coords


def _spread(c, D):
    """Clusters of the cloud moved far apart: no grid within 16 entries a row."""
    far = c.copy()
    far[:, 1:] += (np.arange(len(c))[:, None] % 3) * 40000
    return np.unique(far, axis=0).astype(np.int32)


@pytest.mark.gpu
@pytest.mark.parametrize("D,ks,n", [(3, 3, 2), (3, 3, 63), (3, 3, 700), (3, 2, 300), (2, 3, 300),
                                    (2, 5, 200), (1, 3, 65), (5, 2, 129), (4, 2, 64), (3, 1, 100)])
def test_spread_clouds_match_oracle(D, ks, n):
    rng = np.random.default_rng(n + D)
    c = _spread(random_coords(rng, n, D, 5), D)
    off = oracle.region_offsets(D, ks)
    kofs, ir, orr = oracle.kernel_map(c, c, off)
    _, _, km = gpu_tables_and_map(c, c, off, same=True)
    np.testing.assert_array_equal(gpu_canonical(km), oracle.canonical_pairs(kofs, ir, orr))
    nbr, order = km.nbr.cpu().numpy(), km.out_order.cpu().numpy()
    assert np.array_equal(np.sort(order), np.arange(len(c)))
    got = sorted((k, int(nbr[k, p]), int(order[p])) for k in range(km.K)
                 for p in range(len(c)) if nbr[k, p] >= 0)
    want = sorted((k, int(i), int(o)) for k in range(km.K)
                  for i, o in zip(ir[kofs[k]:kofs[k + 1]], orr[kofs[k]:kofs[k + 1]]))
    assert got == want


@pytest.mark.gpu
@pytest.mark.parametrize("stride", [2, 3])
def test_spread_strided_maps_match_oracle(stride):
    rng = np.random.default_rng(stride)
    c = _spread(random_coords(rng, 500, 3, 6), 3)
    out = oracle.stride(c, [stride] * 3)
    off = oracle.region_offsets(3, stride)
    kofs, ir, orr = oracle.kernel_map(c, out, off)
    _, _, km = gpu_tables_and_map(c, out, off)
    np.testing.assert_array_equal(gpu_canonical(km), oracle.canonical_pairs(kofs, ir, orr))


def test_tables_with_bricks_reserve_no_kept_neighbours():
    """Host sizes only: 28 entries a row less for 27 offsets where the table has a
    brick grid, and the general query covers both."""
    def ws(fn, *a):
        return abi._sizeq(getattr(abi.lib(), fn), *a)

    t = abi.RhipTable()
    t.n_unique, t.ncol = 100000, 4
    plain = ws("rhip_kmap_table_workspace_bytes", ctypes.byref(t), 50000, 27)
    assert plain <= ws("rhip_kmap_workspace_bytes", 100000, 50000, 27)
    t.n_unique = 1000  # the second phase, sized by the input rows, no longer the larger
    plain = ws("rhip_kmap_table_workspace_bytes", ctypes.byref(t), 50000, 27)
    t.bricks = 256  # any address: not read
    bricks = ws("rhip_kmap_table_workspace_bytes", ctypes.byref(t), 50000, 27)
    assert plain - bricks >= 28 * 4 * 50000 - 4096
