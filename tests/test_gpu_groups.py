"""Unions inside groups of tiles (continuous volumes of at least 4,096 row tiles)
at every connectivity and voxel width: ragged last groups, and a region of
distinct values whose groups hold more local roots than the group's table.
Bit for bit."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(66, 505, 250), (3, 509, 512), (18, 512, 505)])
@pytest.mark.parametrize("connectivity", [6, 18, 26])
@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.uint32, np.uint64, np.float64])
def test_groups(gpu, shape, connectivity, dtype):
  import cc3d
  rng = np.random.default_rng(sum(shape) + connectivity)
  print(shape, connectivity, np.dtype(dtype).name, flush=True)
  side = 11
  cells = 80 * rng.integers(0, 4, size=[-(-s // side) for s in shape])
  vol = np.kron(cells, np.ones((side, side, side), np.int64))[:shape[0], :shape[1], :shape[2]]
  vol = np.where(vol > 0, vol - rng.integers(0, 15, size=shape), 0)  # tones within 15 of each other
  part = vol[:, 40:120, 30:100]  # values that no neighbour is near: as many local roots as voxels
  x, y, z = np.meshgrid(*[np.arange(s) for s in part.shape], indexing="ij")
  part[:] = 20 + 28 * ((x & 1) + 2 * (y & 1) + 4 * (z & 1))
  vol = np.asfortranarray(vol.astype(dtype))
  exp, en = oracle.connected_components(vol, connectivity=connectivity, delta=16, return_N=True, out_dtype=np.uint32)
  got, n = cc3d.connected_components(vol, connectivity=connectivity, delta=16, return_N=True, out_dtype=np.uint32)
  assert n == en and np.array_equal(got, exp)
