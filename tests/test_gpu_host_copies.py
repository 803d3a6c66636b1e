"""Results handed to numpy: where dust writes, and boxes narrowed to 16 bits."""
import numpy as np
import pytest

import cc3d

pytestmark = pytest.mark.gpu


def _two_boxes(order, dtype=np.uint32):
  img = np.zeros((9, 8, 7), dtype=dtype, order=order)
  img[1:3, 1:3, 1:3] = 5  # 8 voxels
  img[5:9, 4:8, 3:7] = 7  # 64 voxels
  return img


@pytest.mark.parametrize("dtype", [np.uint8, np.int64, np.float32])
@pytest.mark.parametrize("layout", ["C", "F", "strided", "memmap"])
def test_dust_in_place(layout, dtype, tmp_path):
  img = _two_boxes("F" if layout == "F" else "C", dtype)
  want = img.copy()
  want[1:3, 1:3, 1:3] = 0
  if layout == "strided":
    big = np.full((18, 8, 7), 9, dtype=dtype)
    big[::2] = img
    img = big[::2]
  elif layout == "memmap":
    mm = np.memmap(tmp_path / "img.bin", dtype=dtype, mode="w+", shape=img.shape)
    mm[:] = img
    img = mm
  out = cc3d.dust(img, 20, in_place=True)
  assert np.array_equal(img, want) and np.array_equal(out, want)
  if layout == "strided":
    assert (big[1::2] == 9).all()


@pytest.mark.parametrize("order", ["C", "F"])
def test_dust_read_only(order):
  img = _two_boxes(order)
  img.flags.writeable = False
  with pytest.raises(ValueError):
    cc3d.dust(img, 20, in_place=True)
  assert (img[1:3, 1:3, 1:3] == 5).all()
  assert (cc3d.dust(img, 20)[1:3, 1:3, 1:3] == 0).all()


@pytest.mark.parametrize("n", [1, 4, 5, 65535, 65536])
def test_boxes(n):
  """Label 3 of 1..4 is absent; sides on both sides of the 16-bit limit."""
  lab = np.zeros((n, 2, 3), dtype=np.uint32)
  lab[0, 0, 0], lab[n - 1, 1, 2], lab[n // 2, 1, 0] = 1, 2, 4
  got = cc3d.statistics(lab, no_slice_conversion=True)["bounding_boxes"]
  top = np.iinfo(np.uint32 if n > 65535 else np.uint16).max
  background = [f(axis) for axis in np.nonzero(lab == 0) for f in (np.min, np.max)]
  want = np.array([background, [0, 0, 0, 0, 0, 0], [n - 1, n - 1, 1, 1, 2, 2],
                   [top, 0, top, 0, top, 0], [n // 2, n // 2, 1, 1, 0, 0]])
  assert got.dtype == (np.uint32 if n > 65535 else np.uint16)
  assert np.array_equal(got, want)
