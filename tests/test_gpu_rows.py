"""Row tiles (csrc/rows.hpp) where they can go wrong: sides around the tile
(64 x 8 x 8) and the 16-voxel segment, every voxel width, links that fill a
wave's queue past its capacity, and the scratch limit that sends a volume back
to the voxel tiles.  Labels and N are whole numbers: bit for bit."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

SIDES = [(1, 9, 8), (15, 8, 9), (16, 7, 17), (17, 16, 3), (63, 9, 2), (64, 8, 8), (65, 17, 9), (130, 10, 16)]


def _check(vol, tag, **kw):
  import cc3d
  print(tag, vol.shape, vol.dtype, kw, flush=True)
  try:
    exp, en = oracle.connected_components(vol, return_N=True, **kw)
  except RuntimeError as e:  # more provisional labels than the reference's table holds
    with pytest.raises(RuntimeError, match=str(e)):
      cc3d.connected_components(vol, return_N=True, **kw)
    return
  got, n = cc3d.connected_components(vol, return_N=True, **kw)
  assert n == en and np.array_equal(got, exp), tag


@pytest.mark.parametrize("connectivity", [6, 18, 26])
@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.uint32, np.uint64, np.float32, np.float64])
def test_edges_of_tile_and_segment(gpu, dtype, connectivity):
  rng = np.random.default_rng(connectivity + np.dtype(dtype).itemsize)
  for k, shape in enumerate(SIDES):
    vol = rng.integers(0, 3, size=shape).astype(dtype)
    vol = np.asfortranarray(vol) if k & 1 else vol
    _check(vol, f"multilabel {k}", connectivity=connectivity)
    _check(vol, f"binary {k}", connectivity=connectivity, binary_image=True)


@pytest.mark.parametrize("connectivity", [18, 26])
@pytest.mark.parametrize("binary", [False, True])
def test_more_links_than_a_queue_holds(gpu, connectivity, binary):
  """A checkerboard: no face links, three kept edge links per foreground voxel."""
  x, y, z = np.meshgrid(*[np.arange(s) for s in (130, 17, 18)], indexing="ij")
  vol = np.asfortranarray(((x + y + z) & 1).astype(np.uint32))
  _check(vol, "checkerboard", connectivity=connectivity, binary_image=binary)
  vol = np.asfortranarray(1 + ((x + y + z) & 1).astype(np.uint8))  # both colours labelled
  _check(vol, "two colours", connectivity=connectivity, binary_image=binary)


@pytest.mark.parametrize("connectivity", [6, 18, 26])
@pytest.mark.parametrize("dtype", [np.uint8, np.uint16, np.uint32, np.uint64, np.float32, np.float64])
def test_continuous_edges(gpu, dtype, connectivity):
  """Chains of values within delta of each other but not of all: no link may
  stand for another unless their own pair is linked."""
  rng = np.random.default_rng(7 * connectivity + np.dtype(dtype).itemsize)
  for k, shape in enumerate(SIDES):
    vol = (rng.integers(0, 7, size=shape) * 2).astype(dtype)
    if np.dtype(dtype).kind == "f":
      vol[vol != 0] += rng.random(size=np.count_nonzero(vol)).astype(dtype) * dtype(0.5)
    vol = np.asfortranarray(vol) if k & 1 else vol
    _check(vol, f"continuous {k}", connectivity=connectivity, delta=2)


def test_continuous_special_values(gpu):
  """inf - inf is NaN (no link, except to the equal voxel below at 26), NaN
  links to nothing, and a negative delta leaves only that one rule (where the
  reference's label table holds one label per voxel)."""
  rng = np.random.default_rng(11)
  pool = np.array([0.0, -0.0, np.nan, np.inf, -np.inf, 1.0, 2.5, -1.0], np.float32)
  for dt in (np.float32, np.float64):
    vol = pool[rng.integers(0, len(pool), size=(70, 9, 11))].astype(dt)
    for conn in (6, 18, 26):
      for delta in (1.5, np.inf, -1.0):
        _check(vol, f"special values {delta}", connectivity=conn, delta=delta)


PLANES = [(1, 64), (15, 65), (16, 127), (17, 128), (63, 66), (64, 64), (65, 129), (130, 71)]


@pytest.mark.parametrize("connectivity", [4, 8, 6, 26])
@pytest.mark.parametrize("dtype", [np.uint8, np.uint32, np.uint64, np.float32])
def test_plane_edges(gpu, dtype, connectivity):
  """Planes on 64 x 64 tiles in every mode, with the block numbering of
  binary 8 and the first-row rule of binary 4 (values of one image differ)."""
  rng = np.random.default_rng(13 * connectivity + np.dtype(dtype).itemsize)
  for k, shape in enumerate(PLANES):
    vol = rng.integers(0, 3, size=shape).astype(dtype)
    vol = np.asfortranarray(vol) if k & 1 else np.ascontiguousarray(vol.T)
    _check(vol, f"multilabel {k}", connectivity=connectivity)
    _check(vol, f"binary {k}", connectivity=connectivity, binary_image=True)
    if connectivity in (4, 8, 6):
      _check(vol, f"periodic {k}", connectivity=connectivity, periodic_boundary=True)
      _check(vol, f"periodic binary {k}", connectivity=connectivity, periodic_boundary=True, binary_image=True)
    many = (rng.integers(0, 7, size=shape) * 2).astype(dtype)
    many = np.asfortranarray(many) if k & 1 else np.ascontiguousarray(many.T)
    _check(many, f"continuous {k}", connectivity=connectivity, delta=2)


@pytest.mark.parametrize("connectivity", [18, 26])
def test_groups_of_tiles(gpu, connectivity):
  """Volumes large enough for unions inside groups of tiles: ragged sides (the
  last groups are partly outside), and a region of distinct voxels whose groups
  hold more local roots than the group's table."""
  import synth
  vol = synth.voronoi((1250, 157, 163), 4000, seed=21)
  vol[600:760, 40:110, 30:80] = np.arange(1, 160 * 70 * 50 + 1, dtype=np.uint32).reshape(160, 70, 50)
  _check(vol, "multilabel groups", connectivity=connectivity, out_dtype=np.uint32)
  tones = synth.tones((700, 160, 170), 700, seed=22)
  tones[300:400, 60:120, 40:90] = np.arange(100 * 60 * 50, dtype=np.float32).reshape(100, 60, 50) * 50 + 1000
  _check(tones, "continuous groups", connectivity=connectivity, delta=20, out_dtype=np.uint32)


def test_special_float_values(gpu):
  """NaN equals nothing (not even itself), infinities and signed zeros follow ==."""
  rng = np.random.default_rng(5)
  pool = np.array([0.0, -0.0, np.nan, np.inf, -np.inf, 1.0, 1e-42], np.float32)
  for dt in (np.float32, np.float64):
    vol = pool[rng.integers(0, len(pool), size=(70, 9, 11))].astype(dt)
    for conn in (6, 18, 26):
      _check(vol, "special values", connectivity=conn)


def test_scratch_limit_keeps_ragged_volumes(gpu):
  """A volume whose row tiles exceed the fixed scratch is labelled on the voxel
  tiles: 65 columns leave a second row tile nearly empty."""
  import ctypes
  import torch
  from cc3d import _lib as L
  lib = L.lib()
  f = lib.cc3d_amd_connected_components3d_noalloc
  f.restype = ctypes.c_int
  f.argtypes = lib.cc3d_amd_connected_components3d.argtypes
  sx, sy, sz = 65, 512, 504
  limit = 256 << 20
  assert lib.cc3d_amd_workspace_bytes(sx, sy, sz, 26, 0, 0) > limit
  assert lib.cc3d_amd_workspace_bytes(sx, sy, sz, 26, 0, L.FLAG_TILES_VOXELS) <= limit
  g = torch.Generator().manual_seed(3)
  vol = torch.randint(0, 3, (sx * sy * sz,), generator=g, dtype=torch.int32).to(gpu)
  exp, en = torch.empty_like(vol), ctypes.c_uint64(0)
  got, gn = torch.empty_like(vol), ctypes.c_uint64(0)
  d = np.zeros(1, np.uint32)
  s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
  for fn, out, n in ((lib.cc3d_amd_connected_components3d, exp, en), (f, got, gn)):
    rc = fn(ctypes.c_void_p(vol.data_ptr()), L.DT_U32, sx, sy, sz, vol.numel(), 26, d.ctypes.data,
            ctypes.c_void_p(out.data_ptr()), L.DT_U32, ctypes.byref(n), 0, 0, s)
    assert rc == L.OK
  torch.cuda.synchronize()
  assert en.value == gn.value and torch.equal(exp, got)


@pytest.mark.parametrize("shape", [(1, 1, 1), (64, 64, 1023), (64, 64, 1024), (64, 64, 1025), (1, 1, 131072),
                                   (1, 1, 131073), (64, 2048, 1), (64, 2049, 1)])
def test_one_launch_scan_limits(gpu, shape):
  """Bitmasks of up to 32 blocks of 131,072 voxels and up to 16,384 tiles are
  ranked, and their counters folded, in one launch."""
  vol = np.asfortranarray(np.random.default_rng(len(str(shape))).integers(0, 3, size=shape).astype(np.uint16))
  _check(vol, "scan", connectivity=6)
  _check(vol, "scan", connectivity=26, binary_image=True)


@pytest.mark.parametrize("shape", [(16, 1, 1), (48, 3, 1), (16, 9, 17), (80, 65, 1), (112, 8, 9), (144, 5, 8),
                                   (96, 96, 96)])
def test_stored_root_bits(gpu, shape):
  """Rows of whole segments: the root bitmask is stored, not cleared first, an
  odd last half-word included. The scratch is filled with ones before."""
  import torch
  rng = np.random.default_rng(sum(shape))
  vol = np.asfortranarray(rng.integers(0, 3, size=shape).astype(np.uint32))
  for kw in ({"connectivity": 6}, {"connectivity": 26}, {"connectivity": 18, "binary_image": True}):
    junk = torch.full((1 << 24,), -1, dtype=torch.int32, device="cuda")
    del junk
    _check(vol, "bits", **kw)
  if shape[2] == 1:
    for conn in (4, 8):
      _check(vol[:, :, 0], "bits 2D", connectivity=conn)
      _check(vol[:, :, 0], "bits 2D binary", connectivity=conn, binary_image=True)


@pytest.mark.parametrize("pattern", ["comb", "chain", "sponge", "cells"])
def test_unions_that_meet_at_one_root(gpu, pattern):
  """Links of a wave that would hang the same root: one component over every
  tile joined at one end, along a path, and at random; and many small ones."""
  rng = np.random.default_rng(len(pattern))
  vol = np.zeros((200, 70, 68), dtype=np.uint32, order="F")
  if pattern == "comb":
    vol[::2, :, ::2] = 1
    vol[:, -1, ::2] = 1
    vol[0, 0, :] = 1
  elif pattern == "chain":
    vol[:, ::2, ::2] = 1
    vol[-1, 1::4, ::2] = vol[0, 3::4, ::2] = 1
    vol[-1, 69, 1::4] = vol[-1, 0, 3::4] = 1
    vol[-1, 68:, ::2] = 1
  elif pattern == "sponge":
    vol[:] = rng.random(vol.shape) < 0.35
  else:
    vol[:] = np.repeat(np.repeat(np.repeat(rng.integers(1, 5, (40, 14, 17)), 5, 0), 5, 1), 4, 2)
  for connectivity in (6, 18, 26):
    _check(vol, pattern, connectivity=connectivity, out_dtype=np.uint32)
    _check(vol, pattern, connectivity=connectivity, out_dtype=np.uint32, binary_image=True)


@pytest.mark.parametrize("connectivity,binary,shape", [(26, 0, (96, 70, 50)), (8, 1, (200, 131, 1)), (6, 1, (64, 64, 64))])
def test_captured_job(gpu, connectivity, binary, shape):
  """Both stages recorded in a graph: every replay equals the eager labels,
  whatever the scratch held, with other calls between the replays."""
  import ctypes
  import cc3d
  import torch
  from cc3d import _lib as L
  lib = L.lib()
  sx, sy, sz = shape
  rng = np.random.default_rng(connectivity)
  vol = torch.from_numpy(rng.integers(0, 3, size=(sz, sy, sx)).astype(np.uint8)).cuda()
  out = torch.zeros(sx * sy * sz, dtype=torch.int32, device="cuda")
  ws = torch.empty(64 << 20, dtype=torch.uint8, device="cuda")
  delta = ctypes.c_uint64(0)
  stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()

  def both_stages():
    job = ctypes.c_void_p(0)
    L.check(lib.cc3d_amd_label_begin(ctypes.byref(job), ctypes.c_void_p(vol.data_ptr()), L.DT_U8, sx, sy, sz,
                                     connectivity, ctypes.byref(delta), 0, 0, binary,
                                     ctypes.c_void_p(ws.data_ptr()), ws.numel(), ctypes.c_void_p(stream.cuda_stream)))
    L.check(lib.cc3d_amd_label_finish(job, ctypes.c_void_p(out.data_ptr()), L.DT_U32))
    return job

  torch.cuda.synchronize()
  lib.cc3d_amd_job_free(both_stages())
  torch.cuda.synchronize()
  eager = out.clone()
  with torch.cuda.graph(graph, stream=stream):
    job = both_stages()
  lib.cc3d_amd_job_free(job)
  for rep in range(4):
    out.zero_()
    ws.fill_(255)
    graph.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, eager), rep
    _, n = cc3d.connected_components(vol[0].cpu().numpy(), connectivity=8, return_N=True)
    assert n == oracle.connected_components(vol[0].cpu().numpy(), connectivity=8, return_N=True)[1]
