"""The planner's deal over more bins than a wave has lanes, in steps and, where a
step places few entries, one by one in between: the same places as the host
model of the one-by-one deal, and every property the streaming kernel relies on."""
import numpy as np
import pytest

from test_gpu_attention_plan import check_plan

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv_heads", [1, 2, 4, 8, 32])  # 512, 256, 128, 64 and 16 bins
@pytest.mark.parametrize("kind", ["ragged", "few", "pairs", "uneven", "long"])
def test_plan_matches_the_model(kv_heads, kind):
  rng = np.random.default_rng(kv_heads)
  bins = 512 // kv_heads
  lengths = {
      "ragged": lambda: rng.integers(16, 2048, size=max(bins // 4, 5)).tolist(),
      "few": lambda: rng.integers(1, 2048, size=9).tolist(),  # too few for a step
      "pairs": lambda: rng.integers(900, 1500, size=max(bins // 3, 3)).tolist() + [40, 900, 17],
      # short entries on uneven bins, more than are dealt one by one between two steps
      "uneven": lambda: [16] * (3 * bins) + rng.integers(1000, 2048, size=max(bins // 8, 2)).tolist() + [100] * 90,
      "long": lambda: rng.integers(1, 8192, size=5).tolist(),  # slots of many chunks
  }[kind]()
  check_plan(lengths, kv_heads, 8192 if kind == "long" else 2048)
