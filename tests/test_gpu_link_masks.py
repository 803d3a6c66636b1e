"""Continuous volumes whose voxels keep more links than a wave's queue holds
(csrc/rows.hpp): noise, whose waves list what leaves the tile, and a lattice
that leaves more than the list holds, whose waves store their links as masks.
Bit for bit."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _lattice(shape, dtype):
  """Voxels linked across planes but not along their rows: 8.5 kept links a
  voxel at 26-connectivity (at delta = 10).  Columns 16 to 31 are one value,
  so that their waves keep a list; a few voxels link to nothing."""
  x, y, z = np.meshgrid(*[np.arange(s) for s in shape], indexing="ij")
  vol = np.where(z & 1, np.where(x & 1, 91, 109), np.where(x & 1, 115, 100))
  if shape[0] > 40:
    vol[16:32] = 100
  rng = np.random.default_rng(sum(shape))
  vol[rng.random(shape) < 0.02] = 200
  vol[rng.random(shape) < 0.02] = 0
  return np.asfortranarray(vol.astype(dtype))


def _check(vol, **kw):
  import cc3d
  print(vol.shape, vol.dtype, kw, flush=True)
  exp, en = oracle.connected_components(vol, return_N=True, **kw)
  got, n = cc3d.connected_components(vol, return_N=True, **kw)
  assert n == en and np.array_equal(got, exp)


@pytest.mark.parametrize("connectivity", [18, 26])
@pytest.mark.parametrize("shape", [(130, 17, 18), (20, 17, 18), (16, 9, 26), (66, 505, 250)])
def test_noise(gpu, shape, connectivity):
  rng = np.random.default_rng(sum(shape) + connectivity)
  vol = np.asfortranarray((1 + 100 * rng.random(shape)).astype(np.float32))
  _check(vol, connectivity=connectivity, delta=25, out_dtype=np.uint32)
  vol[:33] = 7  # waves with few links beside waves with many
  _check(vol, connectivity=connectivity, delta=8, out_dtype=np.uint32)
  vol = np.asfortranarray(1 + rng.integers(0, 8, size=shape).astype(np.uint16))
  _check(vol, connectivity=connectivity, delta=2, out_dtype=np.uint32)


@pytest.mark.parametrize("connectivity", [18, 26])
@pytest.mark.parametrize("dtype", [np.uint8, np.uint64, np.float32, np.float64])
@pytest.mark.parametrize("shape", [(130, 17, 18), (64, 8, 8), (33, 20, 9), (20, 17, 18), (16, 9, 26), (1, 40, 40)])
def test_masks(gpu, shape, dtype, connectivity):
  _check(_lattice(shape, dtype), connectivity=connectivity, delta=10, out_dtype=np.uint32)


@pytest.mark.parametrize("connectivity", [18, 26])
@pytest.mark.parametrize("shape", [(66, 505, 250), (2, 512, 512), (18, 509, 506)])
def test_masks_in_groups(gpu, shape, connectivity):
  """4,096 tiles and more: the listed links inside a group of tiles are settled
  there, the masks stay."""
  _check(_lattice(shape, np.float32), connectivity=connectivity, delta=10, out_dtype=np.uint32)


def test_masks_in_batches(gpu):
  import cc3d
  import torch
  vols = [_lattice(s, np.float32) for s in ((130, 17, 18), (20, 17, 18), (50, 30, 9), (64, 64, 1))]
  dev = [torch.from_numpy(np.ravel(v, order="F").copy()).to(gpu).as_strided(v.shape, (1, v.shape[0], v.shape[0] * v.shape[1]))
         for v in vols]
  conns = [26, 18, 6, 26]
  res = cc3d.connected_components_batch(dev, connectivity=conns, return_N=True, out_dtype=np.uint32, delta=10)
  for v, c, (lab, n) in zip(vols, conns, res):
    exp, en = oracle.connected_components(v, connectivity=c, return_N=True, out_dtype=np.uint32, delta=10)
    assert n == en and np.array_equal(lab.cpu().numpy(), exp), (v.shape, c)
