"""GPU parity: attention of many query rows (prefill) on the matrix cores, against
the float64 closed form, at the edges of its tiles: 128 query rows and 32 a wave,
64 positions a tile, mask blocks of 32 rows x 64 positions, heads folded below 128
rows.  Below 2, where the output's rounding is at most 2^-8, the error stays under
6e-3: half an ulp, 2^-8, plus a score's float32 sums and exp2, far below it."""

import math

import pytest
import torch

from conftest import attention_bound, float32_bound
from oracle import attention as OA

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rnd(g, shape, dtype=torch.bfloat16):
  return torch.randn(shape, generator=g).to(dtype)


def make_mask(kind, g, b, hq, t, s):
  if kind is None:
    return None
  if kind == "causal":  # the last rows of a causal mask over s positions
    return torch.full((t, s), -math.inf).triu(1 + s - t).reshape(1, 1, t, s).to(torch.bfloat16)
  m = torch.randn((b, hq, t, s), generator=g)
  m[:, :, :, : s // 2] = 0.0                              # blocks of zeros
  m[:, :, t // 3:, s // 3: 2 * s // 3] = -math.inf        # dead blocks with ragged edges
  m[0, 0, 0] = -math.inf                                  # a row with nothing to attend
  m[-1, -1, t // 2:] = -math.inf
  return m


CASES = [  # b, hq, hkv, d, t, s, mask, scale heads (None: no scales), scale dtype
    (1, 4, 4, 128, 17, 17, "causal", None, None),
    (2, 8, 2, 128, 31, 65, "causal", None, None),
    (1, 8, 2, 128, 127, 127, "causal", 1, torch.bfloat16),
    (1, 4, 2, 128, 128, 256, "causal", None, None),
    (1, 4, 2, 128, 129, 257, "causal", 1, torch.float32),
    (2, 4, 2, 64, 300, 300, "causal", None, None),
    (1, 2, 1, 256, 321, 321, "causal", 1, torch.bfloat16),
    (1, 28, 4, 128, 259, 259, "causal", None, None),
    (2, 4, 2, 128, 200, 330, "any", 2, torch.float32),
    (2, 2, 2, 256, 130, 384, "any", None, None),
    (2, 4, 1, 64, 33, 400, "any", 1, torch.float32),
    (1, 8, 2, 128, 64, 63, None, 2, torch.bfloat16),
    (1, 2, 2, 64, 1, 77, None, None, None),
    (3, 4, 2, 256, 5, 1, None, None, None),
    (1, 4, 2, 128, 130, 257, "any", None, None),            # mask rows that no wide load fits
    (1, 2, 1, 256, 190, 320, "causal", 1, torch.float32),
    (5, 64, 8, 64, 130, 130, "causal", None, None),         # enough rows for workgroups of 128: no mask pass ...
    (5, 64, 8, 64, 130, 258, "causal", 1, torch.bfloat16),  # ... with one
    (40, 8, 1, 128, 129, 192, None, None, None),
    (11, 32, 4, 256, 129, 257, "causal", None, None),
    (6, 64, 8, 64, 130, 130, "causal", None, None),         # either side of the limits between the two kinds of workgroups
    (6, 64, 8, 64, 130, 258, "causal", 1, torch.bfloat16),
    (28, 8, 4, 128, 130, 258, "causal", None, None),
    (34, 8, 4, 128, 130, 130, None, 1, torch.float32),
    (32, 8, 8, 128, 130, 200, None, None, None),
    (12, 8, 8, 256, 130, 200, None, None, None),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(x).replace("torch.", "") for x in c))
def test_many_query_rows(case):
  from jetstream_pt_amd import attention_kernel as ak
  b, hq, hkv, d, t, s, kind, hs, sdt = case
  g = torch.Generator().manual_seed(900 + t)
  q, k, v = rnd(g, (b, hq, t, d)), rnd(g, (b, hkv, s, d)), rnd(g, (b, hkv, s, d))
  mask = make_mask(kind, g, b, hq, t, s)
  ks = vs = None
  if hs:
    ks, vs = ((torch.rand((b, hs, s, 1), generator=g) + 0.5).to(sdt) for _ in range(2))
  rows = None if mask is None else mask.expand(b, hq, t, s).reshape(b, hkv, hq // hkv * t, s)
  want, wm, wl = OA.closed_form(q, k, v, mask=rows, k_scale=ks, v_scale=vs)
  dev = [None if x is None else x.to(DEV) for x in (q, k, v, ks, vs, mask)]
  got, (m, l) = ak.flash_attention(*dev[:3], 0, dev[3], dev[4], dev[5])
  err = (got.double().cpu() - want).abs()
  assert torch.all(err <= torch.where(want.abs() < 2.0, torch.full_like(err, 6e-3), attention_bound(want))), float(err.max())
  live = wl > 0
  assert torch.allclose(m.double().cpu()[live], wm[live], rtol=1e-3, atol=1e-4)
  assert torch.allclose(l.double().cpu()[live], wl[live], rtol=1e-3)
  assert torch.all(torch.isneginf(m.cpu()[~live])) and torch.all(l.cpu()[~live] == 0) and torch.all(got.cpu()[(~live).expand_as(got)] == 0)


def test_many_query_rows_with_lengths():
  """Left-aligned slots of their own lengths, empty and full ones among them."""
  from jetstream_pt_amd import attention_kernel as ak
  g = torch.Generator().manual_seed(940)
  b, hq, hkv, d, t, s = 5, 8, 4, 128, 20, 192
  q, k, v = rnd(g, (b, hq, t, d)), rnd(g, (b, hkv, s, d)), rnd(g, (b, hkv, s, d))
  end = torch.tensor([0, 1, 64, 65, 192], dtype=torch.int32)
  want, _, _ = OA.closed_form(q, k, v, lengths=end)
  for slot, n in enumerate(end.tolist()):  # what lies past a slot's end does not count, whatever it is
    k[slot, :, n:] = math.nan
    v[slot, :, n:] = math.nan
  got, _ = ak.ragged_mha(q.to(DEV), k.to(DEV), v.to(DEV), 0, None, end.to(DEV))
  err = (got.double().cpu().reshape(want.shape) - want).abs()
  assert torch.all(err <= 6e-3), float(err.max())


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("sdt", [None, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("masked", [False, True])
def test_weights_are_float32(masked, sdt, d):
  """Two positions whose values nearly cancel in some column of every row: weights of fewer bits than
  float32's stand out there."""
  from jetstream_pt_amd import attention_kernel as ak
  b, hq, hkv, t = 2, 4, 2, 130
  s = t if masked else 2
  q, k, v = torch.zeros((b, hq, t, d)), torch.zeros((b, hkv, s, d)), torch.zeros((b, hkv, s, d))
  q[..., 0] = (torch.arange(t) + 1) / 64.0
  k[:, :, 1, 0] = -8.0 - torch.arange(b * hkv).reshape(b, hkv)
  v[:, :, 0], v[:, :, 1] = -torch.arange(d) / d, 1.0
  q, k, v = (x.to(torch.bfloat16) for x in (q, k, v))
  mask = ks = vs = rows = None
  if masked:
    mask = torch.full((1, 1, t, s), -math.inf)
    mask[..., :2] = 0.0
    rows = mask.expand(b, hq, t, s).reshape(b, hkv, hq // hkv * t, s)
  if sdt is not None:
    ks, vs = torch.full((b, 1, s, 1), 0.9).to(sdt), torch.full((b, 1, s, 1), 0.7).to(sdt)
  want, _, _ = OA.closed_form(q, k, v, mask=rows, k_scale=ks, v_scale=vs)
  total, _, _ = OA.closed_form(q, k, v.abs(), mask=rows, k_scale=ks, v_scale=vs)
  dev = [None if x is None else x.to(DEV) for x in (q, k, v, ks, vs, mask)]
  got = ak.dense_attention(*dev).double().cpu()
  over = (got - want).abs() / float32_bound(want, total)
  assert torch.all(over <= 1.0), float(over.max())


@pytest.mark.parametrize("heads", [2, 336])
@pytest.mark.parametrize("jump", [2.0, 7.0, 40.0])
def test_maxima_that_rise(jump, heads):
  """Scores that climb from tile to tile, by less and by more than what sums are carried over without being
  rescaled; both ways of dividing a workgroup's waves."""
  from jetstream_pt_amd import attention_kernel as ak
  d, t, s = 64, 130, 512
  g = torch.Generator().manual_seed(945)
  q, k = torch.zeros((1, heads, t, d)), 0.05 * torch.randn((1, heads, s, d), generator=g)
  q[..., 0] = math.sqrt(d) * (torch.arange(t) % 3 - 1)  # rows whose scores fall, stay and climb
  k[..., 0] = (torch.arange(s) // 64) * jump
  q, k, v = q.to(torch.bfloat16), k.to(torch.bfloat16), rnd(g, (1, heads, s, d))
  mask = torch.zeros((1, 1, t, s))
  mask[..., 300:310] = -math.inf
  for m in (None, mask):
    want, wm, wl = OA.closed_form(q, k, v, mask=None if m is None else m.expand(1, heads, t, s))
    got, (gm, gl) = ak.flash_attention(q.to(DEV), k.to(DEV), v.to(DEV), 0, None, None, None if m is None else m.to(DEV))
    err = (got.double().cpu() - want).abs()
    assert torch.all(err <= torch.where(want.abs() < 2.0, torch.full_like(err, 6e-3), attention_bound(want))), float(err.max())
    assert torch.allclose(gm.double().cpu(), wm, rtol=1e-3, atol=1e-4) and torch.allclose(gl.double().cpu(), wl, rtol=1e-3)


@pytest.mark.parametrize("heads", [2, 336])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("up", [3.0, 5.0, 7.5])
def test_large_values_under_a_maximum_that_rises(up, d, heads):
  """A value near bfloat16's largest whose score comes late and is 2^up times the weight of the others: its weight is at
  most 1 in the sums, which so stay finite.  One bfloat16 rounding of the result."""
  from jetstream_pt_amd import attention_kernel as ak
  t, s, late = 130, 320, 200
  q, k, v = torch.zeros((1, heads, t, d)), torch.zeros((1, heads, s, d)), torch.ones((1, heads, s, d))
  q[..., 0] = 1.0
  k[..., late, 0] = up * math.log(2) * math.sqrt(d)
  v[..., late, ::3] = 2.0 ** 127
  q, k, v = (x.to(torch.bfloat16) for x in (q, k, v))
  mask = torch.zeros((1, 1, t, s))
  mask[..., 300:310] = -math.inf
  for m in (None, mask):
    want, _, _ = OA.closed_form(q[:, :1], k[:, :1], v[:, :1], mask=None if m is None else m.expand(1, 1, t, s))
    got = ak.dense_attention(q.to(DEV), k.to(DEV), v.to(DEV), mask=None if m is None else m.to(DEV)).double().cpu()
    assert torch.all((got - want).abs() <= 2.0 ** -8 * want.abs())


@pytest.mark.parametrize("scale", [-0.25, 0.0])
@pytest.mark.parametrize("kind", [None, "causal"])
def test_scales_that_are_not_positive(kind, scale):
  from jetstream_pt_amd import attention_kernel as ak
  b, hq, hkv, d, t, s = 1, 4, 2, 128, 200, 333
  g = torch.Generator().manual_seed(947)
  q, k, v = rnd(g, (b, hq, t, d)), rnd(g, (b, hkv, s, d)), rnd(g, (b, hkv, s, d))
  mask = make_mask(kind, g, b, hq, t, s)
  rows = None if mask is None else mask.expand(b, hq, t, s).reshape(b, hkv, hq // hkv * t, s)
  want, wm, wl = OA.closed_form(q, k, v, mask=rows, sm_scale=scale)
  got, m, l = ak._attend("dense", q.to(DEV), k.to(DEV), v.to(DEV), mask=None if mask is None else mask.to(DEV), sm_scale=scale, want_stats=True)
  err = (got.double().cpu() - want.reshape(got.shape)).abs()
  assert torch.all(err <= torch.where(want.reshape(got.shape).abs() < 2.0, torch.full_like(err, 6e-3), attention_bound(want.reshape(got.shape)))), float(err.max())
  assert torch.allclose(m.double().cpu().reshape(wm.shape), wm, rtol=1e-3, atol=1e-4)
  assert torch.allclose(l.double().cpu().reshape(wl.shape), wl, rtol=1e-3)


LOWEST = [torch.finfo(torch.float32).min, OA.DEFAULT_MASK_VALUE, -2.0 ** 127]


@pytest.mark.parametrize("low", LOWEST)
@pytest.mark.parametrize("d,t,s,dtype", [(64, 20, 100, torch.float32), (128, 200, 300, torch.float32), (256, 20, 64, torch.float32),
                                         (128, 150, 320, torch.bfloat16)])
def test_masks_of_the_lowest_finite_value(d, t, s, dtype, low):
  """A row masked throughout with a finite value attends every position alike; a row with a live position
  attends only those that are live; beyond them -inf still counts for nothing."""
  from jetstream_pt_amd import attention_kernel as ak
  g = torch.Generator().manual_seed(950 + d + t)
  b, hq, hkv = 2, 4, 2
  low = max(low, torch.finfo(dtype).min)
  q, k, v = rnd(g, (b, hq, t, d)), rnd(g, (b, hkv, s, d)), rnd(g, (b, hkv, s, d))
  mask = torch.full((b, 1, t, s), low).to(dtype)
  mask[:, :, t // 2:, : s // 3] = 0.0
  mask[1, :, 0] = -math.inf
  mask[1, :, :, s - 1] = -math.inf
  rows = mask.expand(b, hq, t, s).reshape(b, hkv, hq // hkv * t, s)
  want, wm, wl = OA.closed_form(q, k, v, mask=rows)
  got, (m, l) = ak.flash_attention(*(x.to(DEV) for x in (q, k, v)), 0, None, None, mask.to(DEV))
  err = (got.double().cpu() - want).abs()
  assert torch.all(err <= torch.where(want.abs() < 2.0, torch.full_like(err, 6e-3), attention_bound(want))), float(err.max())
  live = wl > 0
  assert torch.allclose(m.double().cpu()[live], wm[live], rtol=1e-3, atol=1e-4)
  assert torch.allclose(l.double().cpu()[live], wl[live], rtol=1e-3)


def test_prompts_of_two_threads_on_one_stream():
  """A call is two launches, the mask's pass and the attention: calls that other threads enqueue between
  them, prompts and decode steps, change nothing."""
  import threading
  from jetstream_pt_amd import attention_kernel as ak
  g = torch.Generator().manual_seed(960)
  hq, hkv, d, t = 8, 2, 64, 512
  work = []
  for i in range(2):
    q, k, v = rnd(g, (1, hq, t, d)).to(DEV), rnd(g, (1, hkv, t, d)).to(DEV), rnd(g, (1, hkv, t, d)).to(DEV)
    mask = torch.full((1, 1, t, t), -math.inf, device=DEV).triu(1)
    if i:  # a mask that leaves in what the other leaves out
      mask = mask.flip(2, 3).contiguous()
    work.append((q, k, v, mask))
  step = [x[:, :, :1].contiguous() if i == 0 else x for i, x in enumerate(work[0][:3])]
  want = [ak.dense_attention(q, k, v, mask=m) for q, k, v, m in work]
  torch.cuda.synchronize()
  outs, errors = [[], []], []

  def prompts(i):
    try:
      q, k, v, m = work[i]
      for _ in range(100):
        outs[i].append(ak.dense_attention(q, k, v, mask=m))
        ak.dense_attention(*step, mask=m[:, :, :1].contiguous())
    except Exception as e:  # pylint: disable=broad-except
      errors.append(e)

  threads = [threading.Thread(target=prompts, args=(i,)) for i in range(2)]
  for x in threads:
    x.start()
  for x in threads:
    x.join()
  torch.cuda.synchronize()
  assert not errors
  for i in range(2):
    assert all(torch.equal(o, want[i]) for o in outs[i])


def test_a_prompt_uses_no_memory_that_outlives_its_call(monkeypatch):
  from jetstream_pt_amd import attention_kernel as ak
  g = torch.Generator().manual_seed(961)
  t = 700
  q, k, v = (rnd(g, (1, h, t, 128)).to(DEV) for h in (4, 2, 2))
  mask = torch.full((1, 1, t, t), -math.inf, device=DEV).triu(1)
  monkeypatch.setattr(ak, "_workspaces", {})
  ak.dense_attention(q, k, v, mask=mask)
  ak.dense_attention(q, k, v, mask=mask.transpose(2, 3))  # the general way: not contiguous
  assert not ak._workspaces


@pytest.mark.parametrize("t,d,masked", [(40, 64, False), (300, 128, True), (130, 256, False)])
def test_outputs_that_lie_on_8_bytes(t, d, masked):
  """The same bits as on 16, and nothing before or behind them."""
  from jetstream_pt_amd import _ffi
  g = torch.Generator().manual_seed(t)
  q, k, v = (torch.randn((2, h, t, d), generator=g).to(torch.bfloat16).to(DEV) for h in (4, 2, 2))
  mask = torch.full((t, t), -math.inf, device=DEV).triu(1) if masked else None
  a = _ffi.AttnArgs(q=_ffi.ptr(q), k=_ffi.ptr(k), v=_ffi.ptr(v), batch=2, q_heads=4, kv_heads=2, q_rows=t, seq=t, dim=d,
                    q_dtype=_ffi.BF16, kv_dtype=_ffi.BF16, sm_scale=d ** -0.5)
  if masked:
    a.mask, a.mask_dtype, a.mask_stride_t = _ffi.ptr(mask), _ffi.F32, t
  outs = []
  for shift in (8, 4):  # elements: 16 bytes, 8 bytes
    room = torch.full((q.numel() + 16,), 7.0, dtype=torch.bfloat16, device=DEV)
    a.out = room.data_ptr() + 2 * shift
    assert a.out % 16 == 2 * shift % 16 and _ffi.lib.jpt_attn_kernel(a, 1) == _ffi.ATTN_PREFILL
    _ffi.check(_ffi.lib.jpt_attn_dense(a, _ffi.stream()))
    torch.cuda.synchronize()
    assert torch.all(room[:shift] == 7.0) and torch.all(room[shift + q.numel():] == 7.0)
    outs.append(room[shift:shift + q.numel()].clone())
  assert torch.equal(outs[0], outs[1]) and torch.isfinite(outs[0]).all()
