"""The tuner's rule against the library's default tile family (CPU)."""
import pytest


@pytest.mark.parametrize("connectivity", [6, 18, 26])
def test_rows_are_the_default(connectivity):
  """A key missing from the table is labelled on row tiles, so a measurement
  replaces them only with a family that is MARGIN faster."""
  from cc3d import _lib as L
  from cc3d import _tune
  m = _tune.MARGIN
  assert _tune.default_family(connectivity) == "rows"
  assert _tune.decide(connectivity, {"voxels": 1.0, "tall": 1.0, "rows": 1.0 - m / 2}) == "rows"
  assert _tune.decide(connectivity, {"voxels": 1.0 - m / 2, "tall": 1.0 - m / 2, "rows": 1.0}) == "rows"
  assert _tune.decide(connectivity, {"voxels": 1.0 - 2 * m, "tall": 1.0, "rows": 1.0}) == "voxels"
  # the default of the library itself: the same scratch as rows asked for by name
  size = L.lib().cc3d_amd_workspace_bytes
  assert size(100, 90, 80, connectivity, 0, 0) == size(100, 90, 80, connectivity, 0, L.FLAG_TILES_ROWS)
  assert size(100, 90, 80, connectivity, 0, 0) != size(100, 90, 80, connectivity, 0, L.FLAG_TILES_VOXELS)
