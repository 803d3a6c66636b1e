"""What the service reserves for a batch is what the batch takes: its volumes
share tiles as wide as the widest of them needs, and request lists as long as
the largest neighbourhood's."""
import pytest

pytestmark = pytest.mark.gpu


def _batch_bytes(requests):
  from cc3d import _lib as L
  from cc3d import _serve
  table = (L.Volume * len(requests))(*[L.Volume(r.volume.data_ptr(), *_serve._dims(r.volume), r.connectivity)
                                       for r in requests])
  return int(L.lib().cc3d_amd_batch_workspace_bytes(table, len(requests), L.BATCH_MULTILABEL))


def _volume(shape):
  import torch
  sx, sy, sz = shape
  return torch.ones(sx * sy * sz, dtype=torch.int32, device="cuda").as_strided(shape, (1, sx, sx * sy))


@pytest.mark.parametrize("name,work", [
  ("connectivities", [((128, 96, 100), 6)] * 5 + [((128, 96, 100), 26)]),
  ("widths", [((16, 120, 128), 26)] * 5 + [((130, 120, 64), 26), ((20, 64, 64), 18)]),
  ("planes", [((512, 500, 1), 26)] * 4),
  ("alike", [((100, 90, 80), 26)] * 4)])
def test_reserved_for_batches(gpu, name, work):
  from cc3d import _serve
  server = _serve.LabelServer(hbm_budget=1 << 34, workers=0)
  requests = [server.submit(_volume(s), c) for s, c in work]
  outputs = sum(_serve._outputs(r.volume) for r in requests)
  group = server._take()
  assert group == requests
  need = _batch_bytes(group) + outputs
  reserved = server.budget - server.free
  assert need <= reserved == sum(r.footprint for r in group) == server.peak_reserved
  # a budget that holds all but a page of it leaves the last request for the next batch
  tight = _serve.LabelServer(hbm_budget=reserved - 4096, workers=0)
  requests = [tight.submit(_volume(s), c) for s, c in work]
  assert tight._take() == requests[:-1]
  # the workspace is given back whole
  server._swap_for_stats(group, [1] * len(group))
  assert server.budget - server.free == outputs + 2 * _serve._STAT_BYTES_PER_LABEL * len(group)
