"""Scratch of one labelling call (cc3d_amd_workspace_bytes plans on the host
alone): no shape needs more than 32 x 8 x 8 voxel tiles took."""
import pytest

# J and requests of one such tile, and its counters
VOXEL_TILE = 3 * 2048 + 4 * 1012 + 32
WIDTHS = list(range(1, 132)) + [160, 161, 192, 193, 255, 256, 257, 320, 512]


def _scratch(sx, sy, sz, connectivity, binary=0, flags=0):
  from cc3d import _lib as L
  got = int(L.lib().cc3d_amd_workspace_bytes(sx, sy, sz, connectivity, binary, flags))
  assert got > 0
  return got


def _voxel_tiles(sx, sy, sz):
  V = sx * sy * sz
  tiles = -(-sx // 32) * -(-sy // 8) * -(-sz // 8)
  return 8 * V + V // 4 + tiles * VOXEL_TILE + 32768  # forest, bitmask and its prefix, tiles, alignment


def _check(sx, sy, sz, connectivity, binary=0, flags=0):
  """Two row tiles stand for three voxel tiles where 65 to 96 columns are wide:
  the one place where they take more, 3 % on ordinary volumes and up to 6.5 %
  where a tile holds a row or two."""
  limit = _voxel_tiles(sx, sy, sz) * (1.065 if 65 <= sx <= 96 else 1.0)
  got = _scratch(sx, sy, sz, connectivity, binary, flags)
  assert got <= limit, (sx, sy, sz, connectivity, binary, flags, got / limit)


@pytest.mark.parametrize("connectivity", [6, 18, 26])
@pytest.mark.parametrize("binary", [0, 1])
def test_volumes(connectivity, binary):
  for sx in WIDTHS:
    for sy, sz in ((2, 2), (7, 100), (64, 64), (100, 3), (333, 2000), (1, 5000), (5000, 5)):
      _check(sx, sy, sz, connectivity, binary)


def test_narrow_batches():
  """Volumes of at most 32 columns in one call keep narrow rows; a wider one
  among them widens the rows of all."""
  from cc3d import _lib as L
  lib = L.lib()
  n = 12
  table = (L.Volume * n)(*[L.Volume(4096, 2 + i, 200, 200, 26) for i in range(n)])
  voxels = sum((2 + i) * 200 * 200 for i in range(n))
  tiles = n * 25 * 25
  for mode in (L.BATCH_MULTILABEL, L.BATCH_BINARY):
    got = lib.cc3d_amd_batch_workspace_bytes(table, n, mode)
    assert 0 < got <= 8.25 * voxels + tiles * VOXEL_TILE + (1 << 20)
  table[n - 1].sx = 33
  assert lib.cc3d_amd_batch_workspace_bytes(table, n, L.BATCH_MULTILABEL) > got + tiles * 8192


@pytest.mark.parametrize("connectivity", [6, 18, 26])
def test_continuous_volumes(connectivity):
  from cc3d import _lib as L
  for sx in WIDTHS:
    for sy, sz in ((2, 2), (7, 100), (64, 64), (100, 3), (333, 2000), (1, 5000), (5000, 5)):
      _check(sx, sy, sz, connectivity, 0, L.FLAG_CONTINUOUS)
