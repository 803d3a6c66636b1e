"""Long thin volumes: a component is a chain of one entry per tile, which the
unions and stage 2 must not walk entry by entry."""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _times(lib, call, reps=5):
  """Least time of each kernel over some calls."""
  names, ms, counts = ctypes.create_string_buffer(64 * 64), (ctypes.c_double * 64)(), (ctypes.c_int * 64)()
  best = {}
  for _ in range(reps):
    lib.cc3d_amd_profile_enable(1)
    call()
    lib.cc3d_amd_profile_enable(0)
    n = lib.cc3d_amd_profile_collect(names, 64, ms, counts, 64)
    for i in range(n):
      k = names.raw[64 * i:64 * i + 64].split(b"\0", 1)[0].decode()
      best[k] = min(best.get(k, float("inf")), ms[i])
  return best


@pytest.mark.parametrize("shape,p,connectivity,binary", [
  ((16, 8, 100000), 1.0, 6, False), ((8, 8, 30000), 0.3, 26, False), ((64, 30000, 8), 1.0, 6, True),
  ((64, 300000), 0.5, 8, True), ((64, 300000), 0.5, 8, False), ((16, 300000), 1.0, 4, True)])
def test_long_volumes(gpu, shape, p, connectivity, binary):
  import cc3d
  import torch
  from cc3d import _lib as L
  lib = L.lib()
  lib.cc3d_amd_profile_enable.argtypes, lib.cc3d_amd_profile_enable.restype = [ctypes.c_int], None
  lib.cc3d_amd_profile_collect.restype = ctypes.c_int
  rng = np.random.default_rng(len(shape) + connectivity)
  vol = np.asfortranarray((rng.random(shape) < p).astype(np.uint8))
  kw = {"connectivity": connectivity, "binary_image": binary, "out_dtype": np.uint32, "return_N": True}
  strides = np.cumprod((1,) + shape[:-1])
  dev = torch.from_numpy(np.ravel(vol, order="F")).to(gpu).as_strided(shape, tuple(int(s) for s in strides))
  print(shape, p, connectivity, binary, flush=True)
  got, n = cc3d.connected_components(dev, **kw)
  exp, en = oracle.connected_components(vol, **kw)
  assert n == en and np.array_equal(got.cpu().numpy(), exp)
  t = _times(lib, lambda: cc3d.connected_components(dev, **kw))
  print({k: round(1e3 * v) for k, v in t.items()}, "us", flush=True)
  # the forest of a few thousand entries costs no more than a few passes over the volume
  assert t["k_requests"] + t["k_finalize"] < 6 * t["k_local"]
