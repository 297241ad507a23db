"""GPU parity of prompts with enough workgroups of 128 rows to take every place (heads of 64 and 128, no scales), against the
float64 closed form: values whose units differ between tiles and within them, and rows whose small weights meet many
positions, or large values, so that they matter as much as the largest one does.

Bound: half an ulp of the bf16 output, and in units of 2^-24 of the output with every value's magnitude in its place: a
sum's roundings, one a position at most, and 32 for the score (below 8: its product, scale and difference to the maximum),
exp2, the weight and the division.  Where weights are small by construction the units are the same for all sizes, 4096: 2^-12
of the output, an eighth of half its ulp, and as many roundings as a row of 6000 positions has (3000 in a lane's sum of weights,
1125 in the products' sums)."""

import math

import pytest
import torch

from conftest import float32_bound
from oracle import attention as OA

pytestmark = pytest.mark.gpu
DEV = "cuda"


def values(kind, g, b, hkv, s, d):
  v = torch.randn((b, hkv, s, d), generator=g)
  tile = torch.arange(s) // 64
  if kind == "steps":  # every tile in other units, up and down by more and by less than goes into a weight
    v *= torch.tensor([1.0, 2.0 ** 9, 2.0 ** -9, 2.0, 0.5, 2.0 ** 20])[tile % 6][None, None, :, None]
  elif kind == "zeros":  # tiles of zeros, the first and a later one; a head of zeros
    v[:, :, :64] = 0.0
    v[:, :, 128:192] = 0.0
    v[:, 0] = 0.0
  elif kind == "spread":  # numbers that float16 has at the smaller end of its range only, and one that it has not
    v *= 2.0 ** -(torch.randint(0, 28, v.shape, generator=g).float())
    v[0, -1, 5, 3] = 2.0 ** -60
  elif kind == "far":  # units too far apart; too large for any
    v[:, :, :64] *= 2.0 ** 50
    v[:, -1] *= 2.0 ** 60
  return v.to(torch.bfloat16)


CASES = [  # b, hq, hkv, d, t, s, mask
    (6, 64, 8, 64, 130, 450, "causal"),
    (37, 8, 4, 128, 130, 257, "causal"),
    (37, 8, 4, 128, 129, 320, None),
    (6, 64, 8, 64, 130, 256, None),
    (10, 8, 8, 128, 900, 900, "float32"),
]


@pytest.mark.parametrize("kind", ["plain", "steps", "zeros", "spread", "far"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_float16_values(case, kind):
  from jetstream_pt_amd import attention_kernel as ak
  b, hq, hkv, d, t, s, mask_kind = case
  g = torch.Generator().manual_seed(970 + s)
  q, k = (torch.randn((b, h, n, d), generator=g).to(torch.bfloat16) for h, n in ((hq, t), (hkv, s)))
  v = values(kind, g, b, hkv, s, d)
  mask = None
  if mask_kind:
    mask = torch.full((1, 1, t, s), -math.inf, dtype=torch.float32 if mask_kind == "float32" else torch.bfloat16).triu(1 + s - t)
  got, (m, l) = ak.flash_attention(q.to(DEV), k.to(DEV), v.to(DEV), 0, None, None, None if mask is None else mask.to(DEV))
  got, m, l = got.double().cpu(), m.double().cpu(), l.double().cpu()
  for slot in {0, b - 1}:  # (of the batch: the closed form is slow)
    part = slice(slot, slot + 1)
    rows = None if mask is None else mask.expand(1, hq, t, s).reshape(1, hkv, hq // hkv * t, s)
    want, wm, wl = OA.closed_form(q[part], k[part], v[part], mask=rows)
    total, _, _ = OA.closed_form(q[part], k[part], v[part].abs(), mask=rows)
    over = (got[part] - want).abs() / float32_bound(want, total, s + 32)
    assert torch.all(over <= 1.0), float(over.max())
    assert torch.allclose(m[part], wm, rtol=1e-3, atol=1e-4) and torch.allclose(l[part], wl, rtol=1e-3)


def test_float16_values_of_slots_of_their_own_lengths():
  """What lies past a slot's end does not count, whatever it is, nor do its units."""
  from jetstream_pt_amd import attention_kernel as ak
  b, hq, hkv, d, t, s = 37, 8, 4, 128, 130, 320
  g = torch.Generator().manual_seed(980)
  q, k, v = (torch.randn((b, h, n, d), generator=g).to(torch.bfloat16) for h, n in ((hq, t), (hkv, s), (hkv, s)))
  end = torch.randint(0, s + 1, (b,), generator=g).to(torch.int32)
  end[:5] = torch.tensor([0, 1, 64, 65, s])
  want, _, _ = OA.closed_form(q, k, v, lengths=end)
  total, _, _ = OA.closed_form(q, k, v.abs(), lengths=end)
  for slot, n in enumerate(end.tolist()):
    k[slot, :, n:] = math.nan
    v[slot, :, n:] = math.nan if slot % 2 else 2.0 ** 100
  got, _ = ak.ragged_mha(q.to(DEV), k.to(DEV), v.to(DEV), 0, None, end.to(DEV))
  over = (got.double().cpu().reshape(want.shape) - want).abs() / float32_bound(want, total, s + 32)
  assert torch.all(over <= 1.0), float(over.max())


def check(q, k, v, causal, units=4096):
  from jetstream_pt_amd import attention_kernel as ak
  t, s = q.shape[2], k.shape[2]
  mask = torch.full((1, 1, t, s), -math.inf).triu(1 + s - t).to(torch.bfloat16) if causal else None
  got, _ = ak.flash_attention(q.to(DEV), k.to(DEV), v.to(DEV), 0, None, None, None if mask is None else mask.to(DEV), normalize_var=False)
  hkv, rep = k.shape[1], q.shape[1] // k.shape[1]
  # (a slot and a query head of each KV head: the closed form is slow)
  q1, rows = q[:1, ::rep], None if mask is None else mask.expand(1, hkv, t, s)
  want, _, _ = OA.closed_form(q1, k[:1], v[:1], mask=rows, sm_scale=1.0)
  total, _, _ = OA.closed_form(q1, k[:1], v[:1].abs(), mask=rows, sm_scale=1.0)
  over = (got[:1, ::rep].double().cpu() - want).abs() / float32_bound(want, total, units)
  assert torch.all(over <= 1.0), float(over.max())


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("gap", [8.0, 11.0, 14.0, 18.0])
@pytest.mark.parametrize("b,hq,hkv,d,s", [(8, 64, 8, 64, 6000), (40, 8, 4, 128, 3500)])
def test_a_sink_and_a_flat_rest(b, hq, hkv, d, s, gap, causal):
  """One position has all but the whole weight and no value in half of the outputs, which are then the others' alone."""
  g = torch.Generator().manual_seed(int(gap))
  q, k = torch.zeros((b, hq, 130, d)), torch.zeros((b, hkv, s, d))
  q[..., 0] = 8.0
  k[:, :, 0, 0] = gap / 8
  v = torch.rand((b, hkv, s, d), generator=g) + 0.5
  v[:, :, 0, : d // 2] = 0.0
  check(q.to(torch.bfloat16), k.to(torch.bfloat16), v.to(torch.bfloat16), causal)


@pytest.mark.parametrize("one_tile", [False, True])
@pytest.mark.parametrize("x", [1.5625, 1.75, 2.125, 2.4375, 3.0])  # e^-8x: 2^-18, 2^-20.2, 2^-24.5, 2^-28.1, 2^-34.6
def test_small_weights_of_large_values(x, one_tile):
  b, hq, hkv, d, s = 8, 64, 8, 64, 320
  g = torch.Generator().manual_seed(11)
  q, k = torch.zeros((b, hq, 130, d)), torch.zeros((b, hkv, s, d))
  at = torch.arange(s)
  large = at % 2 == 0 if one_tile else at // 64 % 2 == 0
  q[..., 0] = 8.0
  k[:, :, ~large, 0] = x
  v = 1.0 + torch.rand((b, hkv, s, d), generator=g)
  v[:, :, large] *= 2.0 ** round(8 * x / math.log(2))
  check(q.to(torch.bfloat16), k.to(torch.bfloat16), v.to(torch.bfloat16), False)
