"""How many chunks the planner cuts a slot in: as many as the batch's mean chunk asks for and no fewer, whatever a merge costs
- a consumer's largest softmax weight is exact, and a slot in fewer chunks has fewer of them.  Every plan has the properties
the streaming kernel relies on and the host model's deal."""
import numpy as np
import pytest
import torch

from test_gpu_attention_plan import check_plan, read_plan, workers

pytestmark = pytest.mark.gpu


def chunks_of(lengths, kv_heads, seq):
  from jetstream_pt_amd import attention_kernel as ak
  plan = ak.DecodePlan(torch.tensor(lengths, dtype=torch.int32, device="cuda:0"), len(lengths), kv_heads * 4, kv_heads, seq=seq)
  places, _ = read_plan(plan)
  return [int(next(e for e in places if e[0] == slot)[4]) for slot in range(len(lengths))]


def rule(lengths, kv_heads, seq):
  mean = -(-sum(lengths) * kv_heads // (workers() * 5 // 4))
  chunk = max(-(-max(mean, -(-seq // 256)) // 128) * 128, 128)
  return [max(-(-n // chunk), 1) for n in lengths]


@pytest.mark.parametrize("kv_heads", [1, 3, 8, 32])
@pytest.mark.parametrize("n", [1, 128, 129, 256, 257, 384, 385, 512, 513, 640, 780, 781, 1200, 2047, 4000, 8191, 65536])
def test_one_slot(n, kv_heads):
  check_plan([n], kv_heads, 65536)
  check_plan([n], kv_heads, 8192)
  for seq in (65536, 8192):  # the shorter one: chunks of 128
    assert chunks_of([min(n, seq)], kv_heads, seq) == rule([min(n, seq)], kv_heads, seq)


@pytest.mark.parametrize("kv_heads,count", [(8, 32), (8, 3), (16, 24), (1, 160), (4, 118)])
def test_batches(kv_heads, count):
  rng = np.random.default_rng(count)
  lengths = rng.integers(1, 4096, size=count).tolist() + [700] * 5
  check_plan(lengths, kv_heads, 4096)
  assert chunks_of(lengths, kv_heads, 4096) == rule(lengths, kv_heads, 4096)


def test_a_mean_just_above_a_whole_number():
  """One position more than 26240 an item, of more positions than float32 counts: chunks of 26368, and a slot between the two
  is not cut."""
  target = workers() * 5 // 4
  lengths = [26300] + [24000] * 690
  rest = target * 26240 + 1 - sum(lengths)
  lengths += [20000] * (rest // 20000) + [rest % 20000]
  assert rest > 0 and chunks_of(lengths, 1, 65536) == [1] * len(lengths)


def test_the_largest_batch():
  """Every slot's words and every record's are in LDS: 4096 slots with one KV head ask for the most."""
  lengths = [(7 * i) % 300 for i in range(4096)]
  assert chunks_of(lengths, 1, 512) == rule(lengths, 1, 512)
