"""A prompt through the quantised mode's kernel: a caller's own update() of the prefill cache is called, put on the instance
or on the class, and the scales that it gives are attended with.  (No launch: the attention call is looked at.)"""

import pytest
import torch

from jetstream_pt_amd import cache_manager as cm
from jetstream_pt_amd import layers
from jetstream_pt_amd.environment import JetEngineEnvironment, JetEngineEnvironmentData


@pytest.mark.parametrize("where", ["nowhere", "instance", "class"])
def test_update_of_the_callers_own(where, monkeypatch):
  kernel = layers.Int8KVAttentionKernel(JetEngineEnvironment(JetEngineEnvironmentData(batch_size=1, num_layers=1)), 0)
  attended, called = [], []

  def attend(xq, keys, values, k_scaler, v_scaler, *rest):
    attended.append((keys, values, k_scaler, v_scaler))
    return xq, (None, None)

  kernel._attend = attend
  cache = cm.KVCachePrefill(kv_quantize=True)
  update = cm.KVCachePrefill.update
  if where == "instance":
    cache.update = lambda *a, **k: called.append(1) or update(cache, *a, **k)
  elif where == "class":
    monkeypatch.setattr(cm.KVCachePrefill, "update", lambda self, *a, **k: called.append(1) or update(self, *a, **k))
  xq, xk, xv = (torch.randn((1, h, 5, 64)) for h in (4, 2, 2))
  assert kernel(xq, xk, xv, None, cache) is xq
  assert cache.state()[0] is xk and cache.state()[1] is xv
  (keys, values, k_scaler, v_scaler), = attended
  assert keys is xk and values is xv and len(called) == (where != "nowhere")
  assert (k_scaler is None) == (v_scaler is None) == (where == "nowhere")
