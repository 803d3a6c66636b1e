"""Narrow volumes (up to 32 columns) keep rows of 16 or 32 entries per tile
row in scratch: every width at which that changes, several tiles in y and z,
tiles of few and of more than 255 roots, full request lists.  Bit for bit."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

WIDTHS = [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 64]


def _check(vol, tag, **kw):
  import cc3d
  try:
    exp, en = oracle.connected_components(vol, return_N=True, **kw)
  except RuntimeError as e:  # more provisional labels than the reference's table holds
    with pytest.raises(RuntimeError, match=str(e)):
      cc3d.connected_components(vol, return_N=True, **kw)
    return
  got, n = cc3d.connected_components(vol, return_N=True, **kw)
  assert n == en and np.array_equal(got, exp), tag


@pytest.mark.parametrize("connectivity", [6, 18, 26])
@pytest.mark.parametrize("sx", WIDTHS)
def test_widths(gpu, sx, connectivity):
  rng = np.random.default_rng(100 * sx + connectivity)
  shape = (sx, 21, 26)
  print(shape, connectivity, flush=True)
  noise = np.asfortranarray(rng.integers(0, 9, size=shape).astype(np.uint32))  # > 255 roots from 16 columns on
  cells = np.asfortranarray(np.kron(rng.integers(0, 4, size=(-(-sx // 5), 5, 6)), np.ones((5, 5, 5), int))[:sx, :21, :26]
                            .astype(np.uint64))
  x, y, z = np.meshgrid(*[np.arange(s) for s in shape], indexing="ij")
  board = np.asfortranarray(1 + ((x + y + z) & 1).astype(np.uint8))
  for name, vol in (("noise", noise), ("cells", cells), ("board", board), ("mask", (noise > 5).astype(np.uint8))):
    _check(vol, name, connectivity=connectivity, out_dtype=np.uint32)
    _check(vol, name + " binary", connectivity=connectivity, binary_image=True, out_dtype=np.uint32)
    if connectivity == 6:
      _check(vol, name + " periodic", connectivity=6, periodic_boundary=True, out_dtype=np.uint32)
  tones = np.asfortranarray((rng.integers(0, 7, size=shape) * 2 + rng.random(shape)).astype(np.float32))
  for vol in (tones, noise, cells.astype(np.float64) * 3):
    _check(vol, "continuous", connectivity=connectivity, delta=2, out_dtype=np.uint32)


@pytest.mark.parametrize("connectivity", [4, 8])
@pytest.mark.parametrize("sx", WIDTHS)
def test_plane_widths(gpu, sx, connectivity):
  rng = np.random.default_rng(200 * sx + connectivity)
  vol = np.asfortranarray(rng.integers(0, 4, size=(sx, 150)).astype(np.uint16))
  print(vol.shape, connectivity, flush=True)
  for kw in ({}, {"binary_image": True}, {"periodic_boundary": True}, {"delta": 1}):
    _check(vol, str(kw), connectivity=connectivity, out_dtype=np.uint32, **kw)


@pytest.mark.parametrize("widest", [16, 32, 33])
def test_batch_widths(gpu, widest):
  """A batch's rows are as wide as its widest volume needs."""
  import cc3d
  import torch
  rng = np.random.default_rng(widest)
  shapes = [(sx, 9 + sx % 13, 20) for sx in WIDTHS if sx <= widest]
  print(shapes, flush=True)
  vols = [rng.integers(0, 4, size=s).astype(np.uint32) for s in shapes]
  conns = [(26, 18, 6)[k % 3] for k in range(len(vols))]
  dev = [torch.from_numpy(np.ravel(v, order="F").view(np.int32)).to(gpu).as_strided(v.shape, (1, v.shape[0], v.shape[0] * v.shape[1]))
         for v in vols]
  for kw in ({}, {"binary_image": True}, {"delta": 1}):
    res = cc3d.connected_components_batch(dev, connectivity=conns, return_N=True, out_dtype=np.uint32, **kw)
    for v, c, (lab, n) in zip(vols, conns, res):
      exp, en = oracle.connected_components(np.asfortranarray(v), connectivity=c, return_N=True, out_dtype=np.uint32, **kw)
      assert n == en and np.array_equal(lab.cpu().numpy(), exp), (v.shape, c, kw)
