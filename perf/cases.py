"""The calls whose speed counts, over the range that a user of cc3d makes them in.

Every case is one call through the package's public functions on an input that
the program already holds: a device tensor for the labelling calls and
`statistics` (a segmentation pipeline keeps its volumes in HBM), a numpy array
for `dust`, which takes nothing else.

Inputs follow the repository's own workloads:

  multi     segment ids: a Voronoi partition with one seed per ~8,000-11,000
            voxels, 80 % of the region boundary removed as membrane, 2 % salt
  binary    a mask of independent foreground voxels (probability p), or, with
            "blobs", the foreground of a thresholded Voronoi partition
  tones     an image of three grey levels plus noise, labelled with a delta
  segments  labels as connected_components returns them: large regions and
            many single-voxel components, numbered without gaps

`shape` is (sx, sy, sz) with x fastest in memory; `order` "F" hands the call an
(x, y, z) tensor, "C" the same memory as a (z, y, x) tensor.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = os.path.join(_ROOT, "connected-components-3d_amd")
if _PKG not in sys.path:
  sys.path.insert(0, _PKG)

import cc3d  # noqa: E402

_DEV = "cuda"
_OUT = {"u16": np.uint16, "u32": np.uint32, "u64": np.uint64, "auto": None}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
  return [
    # one small crop, labelled on its own: an interactive tool, or a loop over objects
    dict(name="crop_u32_26", op="label", kind="multi", bits=32, shape="64x64x64", conn=26, out="u32", order="C"),
    # an ordinary block of a chunked pipeline
    dict(name="block_u32_26", op="label", kind="multi", bits=32, shape="256x256x256", conn=26, out="u32", order="F"),
    # the headline volume: a whole cutout
    dict(name="cutout_u32_26", op="label", kind="multi", bits=32, shape="512x512x512", conn=26, out="u32", order="F"),
    # 64-bit segment ids, face connectivity, output dtype chosen by the library
    dict(name="cutout_u64_6", op="label", kind="multi", bits=64, shape="512x512x512", conn=6, out="auto", order="F"),
    # a ragged block of narrow ids, 18-connected
    dict(name="ragged_u16_18", op="label", kind="multi", bits=16, shape="301x275x203", conn=18, out="u32", order="C"),
    # a thresholded, noisy probability map: many voxels, one dominant component
    dict(name="mask_p30_26", op="label", kind="binary", p=0.3, shape="512x512x512", conn=26, out="u32", order="F"),
    # the hardest density for face connectivity, odd sides
    dict(name="mask_p50_6", op="label", kind="binary", p=0.5, shape="383x401x367", conn=6, out="u32", order="C"),
    # a whole-slide mask
    dict(name="slide_p50_8", op="label", kind="binary", p=0.5, shape="16384x16384x1", conn=8, out="u32", order="C"),
    # grey levels with noise: labelling within a tolerance
    dict(name="tones_f32_26", op="label", kind="tones", bits=32, shape="512x512x512", conn=26, out="u32", order="F"),
    # many uneven volumes in one call
    dict(name="batch_u32", op="batch", count=32, side_lo=64, side_hi=256, out="u32"),
    # per-object tables of a labelled block
    dict(name="statistics_256", op="statistics", shape="256x256x256", bits=32),
    # removal of small components from an array in host memory
    dict(name="dust_256", op="dust", shape="256x256x192", bits=32, conn=26, threshold=100),
  ]


def _log(rng, lo, hi):
  return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _box(rng, lo, hi):
  """Sides of a box of lo..hi voxels (log-uniform), uneven and often odd."""
  n = _log(rng, lo, hi)
  a = math.exp(rng.uniform(-0.5, 0.5))
  b = math.exp(rng.uniform(-0.5, 0.5))
  s = n ** (1.0 / 3.0)
  sx, sy = max(1, int(s * a)), max(1, int(s * b))
  sz = max(1, int(n / (sx * sy)))
  return f"{sx}x{sy}x{sz}"


def draw(rng):
  op = rng.choice(["multi"] * 5 + ["binary"] * 3 + ["plane"] * 2 + ["tones", "batch", "statistics", "dust"])
  order = rng.choice(["C", "F"])
  if op == "multi":
    bits = rng.choice([16, 32, 32, 64])
    return dict(op="label", kind="multi", bits=bits, shape=_box(rng, 30_000, 120_000_000),
                conn=rng.choice([26, 26, 18, 6]), out=rng.choice(["u32", "auto"]), order=order)
  if op == "binary":
    kind = rng.choice(["binary", "blobs"])
    c = dict(op="label", kind=kind, shape=_box(rng, 30_000, 120_000_000), conn=rng.choice([26, 18, 6]),
             out=rng.choice(["u32", "auto"]), order=order)
    c["p"] = round(rng.uniform(0.05, 0.7), 3)
    return c
  if op == "plane":
    n = _log(rng, 60_000, 250_000_000)
    sx = max(16, int(math.sqrt(n) * math.exp(rng.uniform(-0.5, 0.5))))
    shape = f"{sx}x{max(1, n // sx)}x1"
    if rng.random() < 0.5:
      return dict(op="label", kind="binary", p=round(rng.uniform(0.2, 0.7), 3), shape=shape,
                  conn=rng.choice([8, 4]), out="u32", order=order)
    return dict(op="label", kind="multi", bits=rng.choice([16, 32]), shape=shape, conn=rng.choice([8, 4]),
                out="u32", order=order)
  if op == "tones":
    return dict(op="label", kind="tones", bits=32, shape=_box(rng, 30_000, 60_000_000),
                conn=rng.choice([26, 18, 6]), out="u32", order=order)
  if op == "batch":
    return dict(op="batch", count=rng.randint(4, 40), side_lo=rng.randint(30, 64), side_hi=rng.randint(70, 230),
                out="u32")
  if op == "statistics":
    return dict(op="statistics", shape=_box(rng, 100_000, 16_000_000), bits=rng.choice([32, 64]))
  return dict(op="dust", shape=_box(rng, 100_000, 12_000_000), bits=rng.choice([8, 32]),
              conn=rng.choice([26, 6]), threshold=rng.randint(5, 300))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _shape(case):
  return tuple(int(s) for s in case["shape"].split("x"))


def _gen(seed):
  g = torch.Generator(device=_DEV)
  g.manual_seed(int(seed))
  return g


def _chance(n, p, g):
  """n independent booleans, true with probability p (one random byte pair each)."""
  return torch.randint(0, 65536, (n,), generator=g, device=_DEV, dtype=torch.int32) < int(p * 65536)


def _regions(shape, g, per_seed=9500.0):
  """Voronoi region of every voxel (flat, x fastest) and the number of
  regions: one seed in every cell of a regular grid, at a random place of it."""
  sx, sy, sz = shape
  flat = sz == 1
  c = per_seed ** (1.0 / 2.0 if flat else 1.0 / 3.0)
  if flat:
    c = c / 2.0
  cx, cy, cz = (max(1, int(math.ceil(s / c))) for s in shape)
  n = cx * cy * cz
  jit = torch.rand((3, n), generator=g, device=_DEV)
  idx = torch.arange(n, device=_DEV)
  px = ((idx % cx).float() + jit[0]) * c
  py = ((idx // cx % cy).float() + jit[1]) * c
  pz = ((idx // (cx * cy)).float() + jit[2]) * (0.0 if flat else c)
  out = torch.empty(sx * sy * sz, dtype=torch.int32, device=_DEV)
  x = torch.arange(sx, device=_DEV)
  gx = (x.float() / c).long()
  rows = sy * sz
  step = max(1, (8 << 20) // sx)
  for r0 in range(0, rows, step):
    r = torch.arange(r0, min(rows, r0 + step), device=_DEV)
    y, z = r % sy, r // sy
    gy, gz = (y.float() / c).long(), (z.float() / c).long()
    best = torch.full((r.numel(), sx), 3.0e38, device=_DEV)
    arg = torch.zeros((r.numel(), sx), dtype=torch.int32, device=_DEV)
    for dz in ((0,) if flat else (-1, 0, 1)):
      for dy in (-1, 0, 1):
        qy, qz = gy + dy, gz + dz
        okr = (qy >= 0) & (qy < cy) & (qz >= 0) & (qz < cz)
        base = qy.clamp(0, cy - 1) * cx + qz.clamp(0, cz - 1) * (cx * cy)
        for dx in (-1, 0, 1):
          qx = gx + dx
          cell = base[:, None] + qx.clamp(0, cx - 1)[None, :]
          d = (px[cell] - x) ** 2 + (py[cell] - y[:, None]) ** 2 + (pz[cell] - z[:, None]) ** 2
          ok = okr[:, None] & ((qx >= 0) & (qx < cx))[None, :] & (d < best)
          best = torch.where(ok, d, best)
          arg = torch.where(ok, cell.int(), arg)
    out[r0 * sx:(r0 + r.numel()) * sx] = arg.reshape(-1)
  return out, n


def _boundary(reg, shape):
  """Voxels with a voxel of another region among their 26 neighbours."""
  sx, sy, sz = shape
  lo = reg.view(sz, sy, sx)
  hi = lo
  for axis in range(3):
    n = lo.shape[axis]
    if n == 1:
      continue
    a, b = lo.clone(), hi.clone()
    for s, d in ((slice(0, n - 1), slice(1, n)), (slice(1, n), slice(0, n - 1))):
      at = [slice(None)] * 3
      af = [slice(None)] * 3
      at[axis], af[axis] = d, s
      a[tuple(at)] = torch.minimum(a[tuple(at)], lo[tuple(af)])
      b[tuple(at)] = torch.maximum(b[tuple(at)], hi[tuple(af)])
    lo, hi = a, b
  return (lo != hi).reshape(-1)


def _ids(n, bits, g):
  if bits == 64:
    return torch.randint(1, 2 ** 63 - 1, (n,), generator=g, device=_DEV, dtype=torch.int64)
  hi = {8: 2 ** 8, 16: 2 ** 16, 32: 2 ** 31}[bits]
  return torch.randint(1, hi, (n,), generator=g, device=_DEV, dtype=torch.int64)


_SIGNED = {8: torch.uint8, 16: torch.int16, 32: torch.int32, 64: torch.int64}
_UNSIGNED = {8: torch.uint8, 16: torch.uint16, 32: torch.uint32, 64: torch.uint64}


def _narrow(v, bits):
  """int64 ids as unsigned integers of `bits` bits."""
  if bits == 64:
    return v.view(torch.uint64)
  if bits == 16:
    v = torch.where(v >= 32768, v - 65536, v)
  return v.to(_SIGNED[bits]).view(_UNSIGNED[bits])


def _multi(shape, bits, g):
  reg, n = _regions(shape, g)
  ids = _ids(n, bits, g)
  total = reg.numel()
  out = ids[reg.long()]
  out[_boundary(reg, shape) & _chance(total, 0.8, g)] = 0
  salt = _chance(total, 0.02, g).nonzero().reshape(-1)
  out[salt] = ids[torch.randint(0, n, (salt.numel(),), generator=g, device=_DEV)]
  return _narrow(out, bits)


def _segments(shape, bits, g):
  """Labels of regions with membranes; one voxel in every 50 is salt, each a
  label of its own (their number belongs to the shape, as N does)."""
  reg, n = _regions(shape, g)
  total = reg.numel()
  out = reg.long() + 1
  out[_boundary(reg, shape) & _chance(total, 0.8, g)] = 0
  salt = torch.arange(total // 50, device=_DEV) * 50
  salt += torch.randint(0, 50, (salt.numel(),), generator=g, device=_DEV)
  out[salt] = torch.arange(n + 1, n + 1 + salt.numel(), device=_DEV)
  return _narrow(out, bits)


def _flat_input(case, shape, g):
  kind = case["kind"]
  total = shape[0] * shape[1] * shape[2]
  if kind == "multi":
    return _multi(shape, case["bits"], g)
  if kind == "binary":
    out = torch.empty(total, dtype=torch.uint8, device=_DEV)
    step = 1 << 26
    for a in range(0, total, step):
      b = min(total, a + step)
      out[a:b] = _chance(b - a, case["p"], g)
    return out
  if kind == "blobs":
    reg, n = _regions(shape, g)
    on = _chance(n, case["p"], g)
    return (on[reg.long()] ^ _chance(total, 0.01, g)).to(torch.uint8)
  reg, n = _regions(shape, g, per_seed=27000.0)
  tone = torch.randint(0, 3, (n,), generator=g, device=_DEV).float() * 100.0
  return tone[reg.long()] + (torch.rand((total,), generator=g, device=_DEV) * 10.0 - 5.0)


def _view(flat, shape, order):
  """The tensor a program passes: the array with its own axes, 2D for one plane."""
  sx, sy, sz = shape
  dims = [sx, sy] if sz == 1 else [sx, sy, sz]
  if order == "C":
    return flat.view(tuple(reversed(dims)))
  strides = [1, sx] if sz == 1 else [1, sx, sx * sy]
  return flat.as_strided(tuple(dims), tuple(strides))


def prepare(case, seed):
  g = _gen(seed)
  op = case["op"]
  state = {"case": dict(case)}
  if op == "label":
    shape = _shape(case)
    state["data"] = _view(_flat_input(case, shape, g), shape, case["order"])
  elif op == "batch":
    # sides and connectivities belong to the case, the contents to the seed
    rng = np.random.default_rng([case["count"], case["side_lo"], case["side_hi"]])
    vols, conns = [], []
    for _ in range(case["count"]):
      shape = tuple(int(s) for s in rng.integers(case["side_lo"], case["side_hi"] + 1, size=3))
      vols.append(_view(_multi(shape, 32, g), shape, "F"))
      conns.append(int(rng.choice([6, 26])))
    state["data"], state["conns"] = vols, conns
  elif op == "statistics":
    shape = _shape(case)
    state["data"] = _view(_segments(shape, case["bits"], g), shape, "F")
  else:
    shape = _shape(case)
    flat = _multi(shape, case["bits"], g).cpu().numpy()
    state["data"] = flat.reshape(shape, order="F")
  torch.cuda.synchronize()
  return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _plain(result):
  """(labels, N) with the labels seen as the signed type of their width:
  torch has no indexing for the wider unsigned ones."""
  labels, n = result
  signed = {2: torch.int16, 4: torch.int32, 8: torch.int64}[labels.element_size()]
  return labels.view(signed), n


def run(state):
  case = state["case"]
  op = case["op"]
  if op == "label":
    kw = {"connectivity": case["conn"], "return_N": True, "out_dtype": _OUT[case["out"]]}
    if case["kind"] in ("binary", "blobs"):
      kw["binary_image"] = True
    elif case["kind"] == "tones":
      kw["delta"] = 20
    return _plain(cc3d.connected_components(state["data"], **kw))
  if op == "batch":
    res = cc3d.connected_components_batch(state["data"], connectivity=state["conns"], return_N=True,
                                          out_dtype=_OUT[case["out"]])
    return [_plain(r) for r in res]
  if op == "statistics":
    return cc3d.statistics(state["data"], no_slice_conversion=True)
  return cc3d.dust(state["data"], threshold=case["threshold"], connectivity=case["conn"])


def work(case):
  """Bytes: every input voxel read once and every output element written once."""
  op = case["op"]
  if op == "batch":
    rng = np.random.default_rng([case["count"], case["side_lo"], case["side_hi"]])
    n = 0
    for _ in range(case["count"]):
      n += int(np.prod(rng.integers(case["side_lo"], case["side_hi"] + 1, size=3)))
      rng.choice([6, 26])
    return {"bytes": 8 * n, "flops": 0}
  sx, sy, sz = _shape(case)
  n = sx * sy * sz
  if op == "label":
    size_in = 1 if case["kind"] in ("binary", "blobs") else case["bits"] // 8
    return {"bytes": n * (size_in + 4), "flops": 0}
  if op == "statistics":
    # about one label per 45 voxels: a count, a box of 6 uint16 and 3 float64 each
    return {"bytes": n * case["bits"] // 8 + (n // 45) * (4 + 12 + 24), "flops": 0}
  return {"bytes": 2 * n * case["bits"] // 8, "flops": 0}


def exact(case, seed):
  """Statistics in float64 and whole numbers; labels are whole numbers and
  have no rounding to compare."""
  if case["op"] != "statistics":
    return None
  sx, sy, sz = _shape(case)
  lab = prepare(case, seed)["data"]
  flat = lab.as_strided((sx * sy * sz,), (1,)).cpu().numpy().astype(np.int64)
  n = int(flat.max()) + 1
  count = np.bincount(flat, minlength=n)
  i = np.arange(flat.size, dtype=np.int64)
  axes = [i % sx, i // sx % sy, i // (sx * sy)]
  cen = np.empty((n, 3), np.float64)
  box = np.empty((n, 6), np.int64)
  for a, pos in enumerate(axes):
    total = np.bincount(flat, weights=pos.astype(np.float64), minlength=n)
    with np.errstate(invalid="ignore", divide="ignore"):
      cen[:, a] = total / count
    lo = np.full(n, np.iinfo(np.uint16).max, np.int64)
    hi = np.zeros(n, np.int64)
    np.minimum.at(lo, flat, pos)
    np.maximum.at(hi, flat, pos)
    box[:, 2 * a], box[:, 2 * a + 1] = lo, hi
  return {"voxel_counts": count.astype(np.uint32), "bounding_boxes": box.astype(np.uint16), "centroids": cen}
