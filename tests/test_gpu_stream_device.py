"""A job on a stream of another device than the calling thread's current one."""
import ctypes

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _label(vol, device, current):
  import torch
  from cc3d import _lib as L
  lib = L.lib()
  with torch.cuda.device(device):
    dev = torch.from_numpy(np.ravel(vol, order="F")).to(f"cuda:{device}")
    out = torch.zeros(vol.size, dtype=torch.int32, device=f"cuda:{device}")
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
  sx, sy, sz = vol.shape
  n = int(lib.cc3d_amd_workspace_bytes(sx, sy, sz, 6, 0, 0))
  ws = torch.empty(n, dtype=torch.uint8, device=f"cuda:{device}")
  job, st, delta = ctypes.c_void_p(0), L.Stats(), ctypes.c_uint64(0)
  with torch.cuda.device(current):
    L.check(lib.cc3d_amd_label_begin(ctypes.byref(job), ctypes.c_void_p(dev.data_ptr()), L.DT_U8, sx, sy, sz, 6,
                                     ctypes.byref(delta), 0, 0, 0, ctypes.c_void_p(ws.data_ptr()), n,
                                     ctypes.c_void_p(stream.cuda_stream)))
    L.check(lib.cc3d_amd_label_finish(job, ctypes.c_void_p(out.data_ptr()), L.DT_U32))
    L.check(lib.cc3d_amd_job_stats(job, ctypes.byref(st)))
    lib.cc3d_amd_job_free(job)
    assert torch.cuda.current_device() == current
  stream.synchronize()
  return out.cpu().numpy().view(np.uint32).reshape(vol.shape, order="F"), int(st.N)


@pytest.mark.parametrize("device,current", [(0, 0), (1, 0), (0, 1)])
def test_stream_device(gpu, device, current):
  import torch
  if torch.cuda.device_count() <= max(device, current):
    pytest.skip("needs a second GPU")
  vol = np.asfortranarray(np.random.default_rng(3).integers(0, 3, size=(70, 20, 18)).astype(np.uint8))
  exp, en = oracle.connected_components(vol, connectivity=6, return_N=True, out_dtype=np.uint32)
  for _ in range(2):  # a new buffer, and one of the pool
    got, n = _label(vol, device, current)
    assert n == en and np.array_equal(got, exp)
