"""Work that small calls do not pay for: a launch to narrow a few boxes, and
labels of a single row that are written twice."""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [5, 7998, 7999, 8000, 12000])
def test_boxes_of_small_tables(gpu, n, monkeypatch):
  """Boxes of up to 48,000 coordinates are narrowed on the host, where that
  takes less than a launch: the same table on both sides of the line."""
  import cc3d
  from cc3d import _follow
  calls = []
  lib = _follow._bind()
  real = lib.cc3d_amd_narrow_boxes
  monkeypatch.setattr(lib, "cc3d_amd_narrow_boxes", lambda *a: calls.append(1) or real(*a))
  ids = np.random.default_rng(n).integers(1, n + 1, size=40 * 30 * 20).astype(np.uint32)
  ids[0] = n
  vol = ids.reshape((40, 30, 20), order="F")
  got = cc3d.statistics(vol, no_slice_conversion=True)
  counts, boxes, centroids = oracle.statistics_raw(vol)
  assert bool(calls) == (6 * (n + 1) > 48000)
  assert got["bounding_boxes"].dtype == np.uint16
  assert np.array_equal(got["voxel_counts"], counts)
  assert np.array_equal(got["bounding_boxes"], np.minimum(boxes, 65535))
  assert np.array_equal(got["centroids"], centroids, equal_nan=True)


@pytest.mark.parametrize("fill", ["runs", "empty", "binary"])
def test_single_row(gpu, fill):
  """A single row is labelled by its runs: stage 2 runs only where that rule does
  not apply (no foreground, or a mask)."""
  import cc3d
  from cc3d import _lib as L
  lib = L.lib()
  lib.cc3d_amd_profile_enable.argtypes, lib.cc3d_amd_profile_enable.restype = [ctypes.c_int], None
  lib.cc3d_amd_profile_collect.restype = ctypes.c_int
  names, ms, counts = ctypes.create_string_buffer(64 * 64), (ctypes.c_double * 64)(), (ctypes.c_int * 64)()
  row = np.random.default_rng(1).integers(0, 3, size=70000).astype(np.uint32)
  if fill == "empty":
    row[:] = 0
  kw = {"return_N": True, "out_dtype": np.uint32, "binary_image": fill == "binary"}
  exp, en = oracle.connected_components(row, **kw)
  lib.cc3d_amd_profile_enable(1)
  got, n = cc3d.connected_components(row, **kw)
  lib.cc3d_amd_profile_enable(0)
  k = lib.cc3d_amd_profile_collect(names, 64, ms, counts, 64)
  launched = {names.raw[64 * i:64 * i + 64].split(b"\0", 1)[0] for i in range(k)}
  assert n == en and np.array_equal(got, exp)
  assert (b"k_finalize" in launched) == (fill != "runs")
