"""GPU parity: decode attention over head dims of 64 and 256 and over cache lengths and masks the
streaming kernel does not take, against the float64 closed form, where shares and tiles end: slots
of 0, 1, 31..33 positions, fewer tiles than groups, sequences over many groups, more slots than a
workgroup has threads.  Below 2, where the output's rounding is at most 2^-8, the error stays under
6e-3."""

import math

import pytest
import torch

from conftest import attention_bound, float32_bound
from oracle import attention as OA

pytestmark = pytest.mark.gpu
DEV = "cuda"


def make(g, kind, b, hkv, s, d, hs):
  if kind == "bf16":
    return [torch.randn((b, hkv, s, d), generator=g).to(torch.bfloat16) for _ in range(2)] + [None, None]
  sdt = torch.float32 if kind == "int8_f32" else torch.bfloat16
  kv = [torch.randint(-127, 128, (b, hkv, s, d), generator=g, dtype=torch.int8) for _ in range(2)]
  return kv + [(torch.rand((b, hs, s, 1), generator=g) * 0.015 + 0.005).to(sdt) for _ in range(2)]


def check(got, want, m, l, wm, wl):
  err = (got.double().cpu().reshape(want.shape) - want).abs()
  assert torch.all(err <= torch.where(want.abs() < 2.0, torch.full_like(err, 6e-3), attention_bound(want))), float(err.max())
  m, l, live = m.double().cpu().reshape(wm.shape), l.double().cpu().reshape(wl.shape), wl > 0
  assert torch.allclose(m[live], wm[live], rtol=1e-3, atol=1e-4) and torch.allclose(l[live], wl[live], rtol=1e-3)
  assert torch.all(torch.isneginf(m[~live])) and torch.all(l[~live] == 0)


@pytest.mark.parametrize("kind", ["bf16", "int8_f32", "int8_bf16"])
@pytest.mark.parametrize("d,hq,hkv,s,lens", [
    (64, 4, 4, 96, [0, 1, 31, 32, 33, 96]),
    (256, 16, 2, 64, [64, 0, 63]),
    (256, 8, 8, 4096, [4096, 3000, 17, 2049]),
    (128, 32, 2, 333, [333, 5, 100, 0, 64]),
    (64, 28, 4, 2048, [2047]),
    (256, 2, 1, 40, [(7 * i) % 41 for i in range(300)]),
    (64, 1, 1, 4, [i % 5 for i in range(4200)]),
    (256, 32, 2, 700, [700, 33, 0, 31]),
    (64, 16, 1, 3000, [3000, 1, 2999]),
])
@pytest.mark.parametrize("token", [False, True])
def test_lengths(token, d, hq, hkv, s, lens, kind):
  from jetstream_pt_amd import attention_kernel as ak
  g = torch.Generator().manual_seed(1000 + d + s)
  b = len(lens)
  end = torch.tensor(lens, dtype=torch.int32)
  q = torch.randn((b, hq, 1, d), generator=g).to(torch.bfloat16)
  k, v, ks, vs = make(g, kind, b, hkv, s, d, hkv if kind == "int8_bf16" else 1)
  new = {}
  fk, fv, fks, fvs = k, v, ks, vs
  if token:  # one more position, number `len` of a longer cache
    nk, nv, nks, nvs = make(g, kind, b, hkv, 1, d, hkv if kind == "int8_bf16" else 1)
    new = dict(new_key=nk.to(DEV), new_value=nv.to(DEV))
    if nks is not None:
      new.update(new_k_scaler=nks.to(DEV), new_v_scaler=nvs.to(DEV))
    def longer(x, n):
      if x is None:
        return None
      y = torch.cat([x, torch.zeros_like(x[:, :, :1])], 2)
      for i, at in enumerate(lens):
        y[i, :, at] = n[i, :, 0]
      return y
    fk, fv, fks, fvs = longer(k, nk), longer(v, nv), longer(ks, nks), longer(vs, nvs)
  want, wm, wl = OA.closed_form(q, fk, fv, lengths=end + (1 if token else 0), k_scale=fks, v_scale=fvs)
  dev = [None if x is None else x.to(DEV) for x in (q, k, v, end, ks, vs)]
  o, (m, l) = ak.ragged_mha(*dev[:3], 0, None, dev[3], None, None, dev[4], dev[5], **new)
  check(o, want, m, l, wm, wl)
  o2, _ = ak.ragged_mha(*dev[:3], 0, None, dev[3], None, None, dev[4], dev[5], **new)
  assert torch.equal(o, o2), "the counters are not back at zero, or the order of a sum changed"


@pytest.mark.parametrize("kind", ["bf16", "int8_f32", "int8_bf16"])
@pytest.mark.parametrize("d,hq,hkv,s", [(64, 4, 4, 96), (256, 16, 2, 64), (128, 8, 4, 77)])
@pytest.mark.parametrize("token", [False, True])
def test_what_lies_past_a_slots_end_does_not_count(token, d, hq, hkv, s, kind):
  """Rows from a slot's end on, and their scales, may hold anything: an empty slot, one whose first token
  this is, and slots that end inside a tile and on its edge."""
  from jetstream_pt_amd import attention_kernel as ak
  g = torch.Generator().manual_seed(1050 + d)
  lens = [0, 1, 31, 32, 33, 0, s]
  b, hs = len(lens), hkv if kind == "int8_bf16" else 1
  end = torch.tensor(lens, dtype=torch.int32)
  q = torch.randn((b, hq, 1, d), generator=g).to(torch.bfloat16)
  clean = make(g, kind, b, hkv, s, d, hs)
  new = {}
  if token:
    rows = make(g, kind, b, hkv, 1, d, hs)
    new = {n: x.to(DEV) for n, x in zip(("new_key", "new_value", "new_k_scaler", "new_v_scaler"), rows) if x is not None}
  outs = []
  for poison in (False, True):
    dev = [None if x is None else x.to(DEV) for x in clean]
    for x in dev if poison else ():
      if x is not None and x.is_floating_point():
        for slot, n in enumerate(lens):
          x[slot, :, n:] = math.nan if slot % 2 == 0 else math.inf
    o, (m, l) = ak.ragged_mha(q.to(DEV), dev[0], dev[1], 0, None, end.to(DEV), None, None, dev[2], dev[3], **new)
    outs.append((o, m, l))
  for clean_out, out in zip(*outs):
    assert torch.equal(clean_out, out)
  if not token:
    assert torch.all(outs[0][0][0] == 0) and torch.all(outs[0][2][0] == 0)


@pytest.mark.parametrize("kind", ["bf16", "int8_bf16"])
@pytest.mark.parametrize("d,hq,hkv,t,s,per_head", [(64, 8, 2, 1, 160, False), (256, 4, 4, 3, 90, True), (128, 8, 4, 2, 77, True), (256, 16, 16, 1, 1024, False)])
def test_masks(d, hq, hkv, t, s, per_head, kind):
  from jetstream_pt_amd import attention_kernel as ak
  g = torch.Generator().manual_seed(1100 + d)
  b = 3
  q = torch.randn((b, hq, t, d), generator=g).to(torch.bfloat16)
  k, v, ks, vs = make(g, kind, b, hkv, s, d, 1)
  mask = torch.where(torch.rand((b, hq if per_head else 1, t, s), generator=g) < 0.5, 0.0, -math.inf)
  mask += torch.randn(mask.shape, generator=g)
  mask[1, :, :, : s // 2] = -math.inf
  mask[2] = -math.inf
  mask = mask.to(torch.bfloat16 if per_head else torch.float32)
  rows = mask.expand(b, hq, t, s).reshape(b, hkv, hq // hkv * t, s)
  want, wm, wl = OA.closed_form(q, k, v, mask=rows, k_scale=ks, v_scale=vs)
  dev = [None if x is None else x.to(DEV) for x in (q, k, v, ks, vs, mask)]
  o, (m, l) = ak.flash_attention(*dev[:3], 0, dev[3], dev[4], dev[5])
  check(o, want, m, l, wm, wl)


def cancelling(d, kind, scale, top):
  """Slots of two positions whose values, up to `top`, nearly cancel in some column of every row: anything
  computed in fewer bits than float32's stands out there."""
  b, hq, hkv, s = 130, 4, 2, 40
  q, k, v = torch.zeros((b, hq, 1, d)), torch.zeros((b, hkv, s, d)), torch.zeros((b, hkv, s, d))
  q[..., 0] = (torch.arange(b).reshape(b, 1, 1) + 1) / 64.0
  k[:, :, 1, 0] = -8.0 - torch.arange(hkv)
  v[:, :, 0], v[:, :, 1] = -(torch.arange(d) % (top + 1)), top
  if kind == "bf16":
    return [x.to(torch.bfloat16) for x in (q, k, v)] + [None, None]
  sdt = torch.float32 if kind == "int8_f32" else torch.bfloat16
  return [q.to(torch.bfloat16), k.to(torch.int8), v.to(torch.int8), torch.full((b, 1, s, 1), 0.9).to(sdt),
          torch.full((b, 1, s, 1), scale).to(sdt)]


def check_cancelling(d, kind, scale, top):
  from jetstream_pt_amd import attention_kernel as ak
  q, k, v, ks, vs = cancelling(d, kind, scale, top)
  end = torch.full((q.shape[0],), 2, dtype=torch.int32)
  want, _, _ = OA.closed_form(q, k, v, lengths=end, k_scale=ks, v_scale=vs)
  total, _, _ = OA.closed_form(q, k, v.abs(), lengths=end, k_scale=ks, v_scale=vs)
  dev = [None if x is None else x.to(DEV) for x in (q, k, v, end, ks, vs)]
  got, _ = ak.ragged_mha(*dev[:3], 0, None, dev[3], None, None, dev[4], dev[5])
  over = (got.double().cpu().reshape(want.shape) - want).abs() / float32_bound(want, total)
  assert torch.all(over <= 1.0), float(over.max())


@pytest.mark.parametrize("d", [64, 128, 256])
def test_weights_are_float32(d):
  check_cancelling(d, "bf16", 1.0, min(d - 1, 127))


@pytest.mark.parametrize("kind", ["int8_f32", "int8_bf16"])
@pytest.mark.parametrize("d,top", [(64, 3), (128, 127), (256, 3)])
def test_sums_of_small_codes_are_float32(d, top, kind):
  check_cancelling(d, kind, 1.0, top)


@pytest.mark.parametrize("kind", ["int8_f32", "int8_bf16"])
@pytest.mark.parametrize("d,scale", [(64, 8e-8), (64, 1e3), (128, 1e-5), (256, 1e-6), (256, 1e-3), (256, 1e30)])
def test_value_scales_of_any_size(d, scale, kind):
  check_cancelling(d, kind, scale, min(d - 1, 127))


@pytest.mark.parametrize("d", [64, 128, 256])
def test_value_scales_far_apart(d):
  """Scales of a slot's positions over twelve orders of magnitude, growing, falling and mixed, the large ones
  on positions whose weights are small too: errors stay float32's beside the sum of the magnitudes."""
  from jetstream_pt_amd import attention_kernel as ak
  g = torch.Generator().manual_seed(1200 + d)
  b, hq, hkv, s = 6, 8, 4, 300
  q = (torch.randn((b, hq, 1, d), generator=g) * 0.1).to(torch.bfloat16)
  k, v = (torch.randint(-127, 128, (b, hkv, s, d), generator=g, dtype=torch.int8) for _ in range(2))
  ks = torch.full((b, 1, s, 1), 0.02)
  spread = 10.0 ** (torch.rand((b, 1, s, 1), generator=g) * 12 - 7)
  spread[0], spread[1] = spread[0].sort(1)[0], spread[1].sort(1, descending=True)[0]
  q[2] *= 40.0  # sharp weights
  end = torch.tensor([s, s, s, 33, 299, 64], dtype=torch.int32)
  want, _, _ = OA.closed_form(q, k, v, lengths=end, k_scale=ks, v_scale=spread)
  total, _, _ = OA.closed_form(q, k, v.abs(), lengths=end, k_scale=ks, v_scale=spread)
  got, _ = ak.ragged_mha(q.to(DEV), k.to(DEV), v.to(DEV), 0, None, end.to(DEV), None, None, ks.to(DEV), spread.to(DEV))
  # scores up to 8 (slot 2: 320): a unit of a weight for every 2^-24 of its score, sums of up to 300 terms
  units = torch.tensor([64, 64, 1024, 64, 64, 64]).reshape(b, 1, 1, 1)
  over = (got.double().cpu().reshape(want.shape) - want).abs() / float32_bound(want, total, units)
  assert torch.all(over <= 1.0), over.amax((1, 2, 3))


@pytest.mark.parametrize("kind", ["bf16", "int8_f32"])
@pytest.mark.parametrize("low", [torch.finfo(torch.float32).min, OA.DEFAULT_MASK_VALUE])
@pytest.mark.parametrize("d,s", [(64, 160), (128, 77), (256, 2048)])
def test_masks_of_the_lowest_finite_value(d, s, low, kind):
  from jetstream_pt_amd import attention_kernel as ak
  g = torch.Generator().manual_seed(1300 + d)
  b, hq, hkv = 3, 4, 2
  q = torch.randn((b, hq, 1, d), generator=g).to(torch.bfloat16)
  k, v, ks, vs = make(g, kind, b, hkv, s, d, 1)
  mask = torch.full((b, 1, 1, s), low)      # slot 0: masked throughout
  mask[1, ..., : s // 2] = 0.0              # slot 1: a live half
  mask[2, ..., 5:] = -math.inf              # slot 2: five positions at the lowest value, nothing else
  rows = mask.expand(b, hq, 1, s).reshape(b, hkv, hq // hkv, s)
  want, wm, wl = OA.closed_form(q, k, v, mask=rows, k_scale=ks, v_scale=vs)
  dev = [None if x is None else x.to(DEV) for x in (q, k, v, ks, vs, mask)]
  o, (m, l) = ak.flash_attention(*dev[:3], 0, dev[3], dev[4], dev[5])
  check(o, want, m, l, wm, wl)


@pytest.mark.parametrize("kind", ["bf16", "int8_f32"])
@pytest.mark.parametrize("d,s", [(64, 4096), (128, 4090)])
def test_captured_calls_have_a_workspace_of_their_own(d, s, kind):
  """A captured call replayed after larger calls have come and gone on the stream it was captured on, beside
  another graph's replay on another stream, and with tensors in the memory that was given back: every replay
  gives the eager bits."""
  from jetstream_pt_amd import attention_kernel as ak
  g = torch.Generator().manual_seed(1400)
  hq, hkv = 8, 8
  lens = [s, 17, 0, 2500]
  inputs = []
  for i in range(2):
    k, v, ks, vs = make(g, kind, len(lens), hkv, s, d, 1)
    q = torch.randn((len(lens), hq, 1, d), generator=g).to(torch.bfloat16)
    inputs.append([None if x is None else x.to(DEV) for x in (q, k, v, torch.tensor(lens, dtype=torch.int32), ks, vs)])
  call = lambda x: ak.ragged_mha(*x[:3], 0, None, x[3], None, None, x[4], x[5])[0]
  want = [call(x) for x in inputs]
  stream = torch.cuda.Stream()
  graphs, outs = [], []
  for x in inputs:
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
      outs.append(call(x))
    graphs.append(graph)
  big = torch.randn((8, 16, 1, 256), generator=g).to(torch.bfloat16).to(DEV)
  cache = torch.randn((8, 1, 512, 256), generator=g).to(torch.bfloat16).to(DEV)
  with torch.cuda.stream(stream):  # a larger workspace in the place of the stream's
    ak.dense_attention(big, cache, cache)
  torch.cuda.synchronize()
  others = [torch.full((1 << 20,), 7, dtype=torch.int32, device=DEV) for _ in range(8)]
  side = [torch.cuda.Stream(), torch.cuda.Stream()]
  for _ in range(5):
    for o in outs:
      o.zero_()
    torch.cuda.synchronize()
    for graph, at in zip(graphs, side):
      with torch.cuda.stream(at):
        graph.replay()
    assert torch.equal(call(inputs[0]), want[0])
    torch.cuda.synchronize()
    for o, w in zip(outs, want):
      assert torch.equal(o, w)
  assert all(bool((x == 7).all()) for x in others)
