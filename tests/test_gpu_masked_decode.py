"""GPU parity: decode attention under a float32 row mask, whose dead tiles the streaming kernel leaves out, and
the step's line written by the launch that attends.  Tiles are 32 positions, a map's bytes 8 tiles, its words 32; a
worker's first 10 items have a map if they are no longer than 256 tiles."""

import math

import pytest
import torch

from conftest import attention_bound
from oracle import attention as OA

pytestmark = pytest.mark.gpu
DEV = "cuda"
INF = math.inf


def caches(g, b, hkv, s, kind, hs=1):
  if kind == "bf16":
    return [torch.randn((b, hkv, s, 128), generator=g).to(torch.bfloat16) for _ in range(2)] + [None, None]
  dtype = torch.float32 if kind == "int8_f32" else torch.bfloat16
  codes = [torch.randint(-127, 128, (b, hkv, s, 128), generator=g).to(torch.int8) for _ in range(2)]
  return codes + [((torch.rand((b, hs, s, 1), generator=g) + 0.5) * 0.02).to(dtype) for _ in range(2)]


def masks(g, kind, b, s):
  m = torch.full((b, s), -INF)
  if kind == "window":  # a ring buffer's: the last n positions before one of the buffer
    now = int(torch.randint(0, s, (1,), generator=g))
    age = (now - torch.arange(s)) % s
    n = torch.randint(0, s + 1, (b,), generator=g)
    n[0], n[-1] = 0, s
    m[age[None] < n[:, None]] = 0.0
  elif kind == "single":  # one position a slot, somewhere
    m[torch.arange(b), torch.randint(0, s, (b,), generator=g)] = -0.5
  elif kind == "edges":  # the first and last positions of tiles, bytes and words of the map
    for at in (0, 31, 32, 255, 256, 1023, 1024, s - 1):
      if at < s:
        m[at % b, at] = 0.25
  elif kind == "sparse":
    m[torch.rand((b, s), generator=g) < 0.01] = 1.0
  else:  # nothing is dead
    m = torch.randn((b, s), generator=g)
  return m


@pytest.mark.parametrize("mask", ["window", "single", "edges", "sparse", "full"])
@pytest.mark.parametrize("b,hq,hkv,s,kind", [
    (2, 8, 8, 32, "bf16"), (3, 8, 2, 96, "int8_f32"), (8, 32, 32, 1024, "bf16"), (5, 32, 4, 2080, "int8_bf16"), (2, 28, 4, 4096, "bf16"),
    (33, 64, 8, 512, "int8_f32"), (3, 16, 1, 1056, "int8_bf16"), (200, 32, 32, 64, "bf16"), (3, 8, 8, 9216, "int8_f32"), (96, 8, 8, 8448, "int8_bf16")])
def test_what_a_mask_leaves_out_is_left_out(b, hq, hkv, s, kind, mask):
  from jetstream_pt_amd import attention_kernel as ak
  g = torch.Generator().manual_seed(b * s + hkv)
  big = b * hkv * s > 1 << 20
  if big:  # too much for the closed form: some slots of it, the rest copies of them
    k, v, ks, vs = (None if x is None else x.repeat((b // 4 + 1, 1, 1, 1))[:b] for x in caches(g, 4, hkv, s, kind))
  else:
    k, v, ks, vs = caches(g, b, hkv, s, kind)
  q = torch.randn((b, hq, 1, 128), generator=g).to(torch.bfloat16)
  m = masks(g, mask, b, s)
  got, (gm, gl) = ak.flash_attention(*(x.to(DEV) for x in (q, k, v)), 0, *(None if x is None else x.to(DEV) for x in (ks, vs)), m.reshape(b, 1, 1, s).to(DEV))
  few = torch.arange(b) if not big else torch.tensor([0, 1, 2, b - 2, b - 1])
  rows = m[few].reshape(-1, 1, 1, s).expand(len(few), hkv, hq // hkv, s)
  want, wm, wl = OA.closed_form(q[few], k[few], v[few], mask=rows, **({} if ks is None else dict(k_scale=ks[few], v_scale=vs[few])))
  err = (got.double().cpu()[few] - want).abs()
  assert torch.all(err <= attention_bound(want)), float(err.max())
  live = wl > 0
  assert torch.allclose(gm.double().cpu()[few][live], wm[live], rtol=1e-3, atol=1e-3) and torch.allclose(gl.double().cpu()[few][live], wl[live], rtol=1e-3)
  assert torch.all(got.cpu()[few][(~live).expand_as(want)] == 0) and torch.all(gl.cpu()[few][~live] == 0) and torch.all(torch.isneginf(gm.cpu()[few][~live]))


@pytest.mark.parametrize("mask", ["window", "single", "edges", "sparse"])
@pytest.mark.parametrize("b,hq,hkv,s,kind", [
    (8, 32, 32, 1024, "bf16"), (64, 32, 8, 2048, "int8_f32"), (5, 32, 4, 2080, "int8_bf16"), (40, 20, 5, 512, "bf16"), (200, 12, 12, 256, "int8_bf16"),
    (3, 8, 8, 9216, "int8_f32"), (200, 32, 32, 96, "bf16")])
def test_leaving_tiles_out_changes_no_bit(b, hq, hkv, s, kind, mask):
  """float32's lowest value at one position of a tile makes it a tile that is read, whose weights are all 0: the same
  outputs and statistics as where nothing of it is left and it is not read."""
  from jetstream_pt_amd import attention_kernel as ak
  g = torch.Generator().manual_seed(b * s + hkv)
  k, v, ks, vs = (None if x is None else x.repeat((b // 4 + 1, 1, 1, 1))[:b].to(DEV) for x in caches(g, min(b, 4), hkv, s, kind))
  q = torch.randn((b, hq, 1, 128), generator=g).to(torch.bfloat16).to(DEV)
  left_out = masks(g, mask, b, s)
  read = left_out.clone()
  tiles = read.view(b, s // 32, 32)
  tiles[..., 7][torch.isneginf(tiles).all(-1)] = torch.finfo(torch.float32).min
  assert not torch.equal(left_out, read)
  got, want = (ak.flash_attention(q, k, v, 0, ks, vs, m.reshape(b, 1, 1, s).to(DEV)) for m in (left_out, read))
  assert torch.equal(got[0].view(torch.int16), want[0].view(torch.int16))
  assert torch.equal(got[1][0], want[1][0]) and torch.equal(got[1][1], want[1][1])


@pytest.mark.parametrize("b,hq,hkv,s", [(90, 5, 5, 1120), (200, 12, 12, 256), (64, 32, 8, 2048)])
def test_a_mask_of_zeros_changes_no_bit(b, hq, hkv, s):
  """... nor does the order of the heads under a mask."""
  from jetstream_pt_amd import attention_kernel as ak
  g = torch.Generator().manual_seed(b + s)
  k, v = (x.repeat((b // 4 + 1, 1, 1, 1))[:b].to(DEV) for x in caches(g, 4, hkv, s, "bf16")[:2])
  q = torch.randn((b, hq, 1, 128), generator=g).to(torch.bfloat16).to(DEV)
  got, want = (ak.flash_attention(q, k, v, 0, None, None, m) for m in (torch.zeros((b, 1, 1, s), device=DEV), None))
  assert torch.equal(got[0], want[0]) and torch.equal(got[1][1], want[1][1])


def test_a_tile_with_a_nan_is_not_left_out():
  from jetstream_pt_amd import attention_kernel as ak
  g = torch.Generator().manual_seed(5)
  k, v, _, _ = caches(g, 2, 8, 512, "bf16")
  q = torch.randn((2, 8, 1, 128), generator=g).to(torch.bfloat16)
  m = masks(g, "window", 2, 512)
  m[1, 300] = math.nan
  got = ak.dense_attention(*(x.to(DEV) for x in (q, k, v)), mask=m.reshape(2, 1, 1, 512).to(DEV))
  assert torch.isnan(got[1]).all() and not torch.isnan(got[0]).any()


@pytest.mark.parametrize("count", ["one", "each"])
@pytest.mark.parametrize("b,hq,hkv,s,kind,hs,rounding,rope", [
    (8, 32, 32, 1024, "bf16", 1, None, False), (3, 8, 2, 96, "bf16", 1, None, False), (200, 32, 32, 64, "bf16", 1, None, False),
    (64, 32, 32, 64, "bf16", 1, None, False), (65, 32, 32, 64, "bf16", 1, None, False), (128, 16, 16, 64, "int8_bf16", 1, "rne", False),
    (129, 16, 16, 64, "int8_f32", 1, "trunc", False), (128, 8, 8, 96, "int8_f32", 1, "trunc", True), (129, 8, 8, 96, "int8_bf16", 1, "rne", True),
    (5, 32, 8, 2048, "int8_f32", 1, "trunc", False), (5, 32, 8, 2048, "int8_bf16", 1, "rne", True), (3, 28, 4, 4096, "int8_bf16", 4, "trunc", True),
    (33, 64, 8, 512, "int8_f32", 8, "rne", False), (40, 32, 32, 64, "int8_bf16", 1, "trunc", True), (1, 8, 8, 32, "int8_bf16", 1, "rne", False)])
def test_the_launch_that_attends_writes_the_line(b, hq, hkv, s, kind, hs, rounding, rope, count):
  """Cache, scales and output are those of the line's own launch followed by attention, bit for bit - at every place of a
  tile and of a chunk, and outside the cache, where nothing is written.  One launch up to 2048 bf16 items, to 32768
  batch * kv_heads^2 int8, to 8192 with the key rotated; with 2048 items a worker has four records."""
  from jetstream_pt_amd import _ffi
  from jetstream_pt_amd import attention_kernel as ak
  g = torch.Generator().manual_seed(b * s + hq)
  base = [None if x is None else x.to(DEV) for x in caches(g, b, hkv, s, kind, hs)]
  q = torch.randn((b, hq, 1, 128), generator=g).to(torch.bfloat16).to(DEV)
  xk, xv = (torch.randn((b, hkv, 1, 128), generator=g).to(torch.bfloat16).to(DEV) for _ in range(2))
  angle = torch.rand((b, 64), generator=g) * 6
  freqs = torch.stack([angle.cos(), angle.sin()], -1).to(DEV) if rope else None
  mask = masks(g, "window", b, s)
  places = sorted({0, 1, 31, 32, s // 2 - 1, s // 2, s - 1}) + [-1, s]
  for i, at in enumerate(places):
    pos = torch.tensor([at], dtype=torch.int32) if count == "one" else torch.tensor([places[(i + j) % len(places)] for j in range(b)], dtype=torch.int32)
    m = mask.clone()
    for slot in range(b):  # the line's position is live, but where there are slots enough to leave it out in one
      p = int(pos[0 if count == "one" else slot])
      if 0 <= p < s and (slot != 1 or b < 3):
        m[slot, p] = 0.0
    m, pos = m.reshape(b, 1, 1, s).to(DEV), pos.to(DEV)
    one, two = ([None if x is None else x.clone() for x in base] for _ in range(2))

    def args(c):
      a = _ffi.AttnArgs(q=_ffi.ptr(q), k=_ffi.ptr(c[0]), v=_ffi.ptr(c[1]), mask=_ffi.ptr(m), batch=b, q_heads=hq, kv_heads=hkv, q_rows=1, dim=128,
                        seq=s, q_dtype=_ffi.BF16, kv_dtype=_ffi.dtype_code(c[0].dtype), mask_dtype=_ffi.F32, mask_stride_b=s, sm_scale=128 ** -0.5)
      if c[2] is not None:
        a.k_scale, a.v_scale, a.scale_dtype, a.scale_heads = _ffi.ptr(c[2]), _ffi.ptr(c[3]), _ffi.dtype_code(c[2].dtype), hs
      return a

    outs = []
    for c, fused in ((one, True), (two, False)):
      a = args(c)
      ws, planned = ak._dense_workspace(0, b, hq, hkv, 1, s)
      a.workspace, a.workspace_bytes, a.reuse_plan = _ffi.ptr(ws.buf), ws.nbytes, int(planned)
      outs.append(torch.empty_like(q))
      a.out = _ffi.ptr(outs[-1])
      if kind == "bf16":
        if fused:
          _ffi.check(_ffi.lib.jpt_attn_dense_line(a, _ffi.ptr(xk), _ffi.ptr(xv), _ffi.ptr(pos), pos.numel(), _ffi.stream()))
        else:
          t = (_ffi.LineTensor * 2)()
          for j, (dst, src) in enumerate(((c[0], xk), (c[1], xv))):
            t[j].dst, t[j].src, t[j].heads, t[j].row_bytes = dst.data_ptr(), src.data_ptr(), hkv, 256
          _ffi.check(_ffi.lib.jpt_kv_scatter_lines(t, 2, _ffi.ptr(pos), pos.numel(), 1, b, s, _ffi.stream()))
      else:
        w = _ffi.QuantAppendArgs(new_k=_ffi.ptr(xk), new_v=_ffi.ptr(xv), cache_k=_ffi.ptr(c[0]), cache_v=_ffi.ptr(c[1]), k_scale=_ffi.ptr(c[2]),
                                 v_scale=_ffi.ptr(c[3]), pos=_ffi.ptr(pos), pos_count=pos.numel(), batch=b, heads=hkv, seq=s, dim=128, in_dtype=_ffi.BF16,
                                 scale_dtype=_ffi.dtype_code(c[2].dtype), scale_heads=hs, rounding=0 if rounding == "trunc" else 1,
                                 rope=_ffi.ptr(freqs))
        _ffi.check(_ffi.lib.jpt_attn_dense_append(a, w, _ffi.stream()) if fused else _ffi.lib.jpt_kv_append_quant_i8(w, _ffi.stream()))
      if not fused:
        _ffi.check(_ffi.lib.jpt_attn_dense(a, _ffi.stream()))
    assert torch.equal(outs[0].view(torch.int16), outs[1].view(torch.int16)), at
    for x, y in zip(one, two):
      assert x is None or torch.equal(x.view(torch.uint8), y.view(torch.uint8)), at


def test_a_line_without_a_mask_or_beside_its_neighbours():
  """Calls that the launch does not take as one: no mask, a cache that begins inside a cache line, heads of 64."""
  from jetstream_pt_amd import attention_kernel as ak, cache_manager as cm, layers
  from jetstream_pt_amd.environment import JetEngineEnvironment, JetEngineEnvironmentData
  g = torch.Generator().manual_seed(11)
  b, h, s = 2, 4, 64
  env = JetEngineEnvironment(JetEngineEnvironmentData(batch_size=b, num_layers=1, cache_sequence_length=s, ring_buffer=True))
  for d, shift, masked in ((128, 0, False), (128, 16, True), (64, 0, True)):
    n = b * h * s * d
    k, v = (torch.randn(n + 64, generator=g).to(torch.bfloat16).to(DEV)[shift // 2: shift // 2 + n].view(b, h, s, d) for _ in range(2))
    q, xk, xv = (torch.randn((b, h, 1, d), generator=g).to(torch.bfloat16).to(DEV) for _ in range(3))
    mask = masks(g, "window", b, s)
    mask[:, 40] = 0.0
    mask = mask.reshape(b, 1, 1, s).to(DEV) if masked else None
    want_k, want_v = k.clone(), v.clone()
    want_k[:, :, 40], want_v[:, :, 40] = xk[:, :, 0], xv[:, :, 0]
    want = ak.dense_attention(q, want_k, want_v, mask=mask)
    cache = cm.KVCacheGenerate(k, v, torch.tensor([40], dtype=torch.int32, device=DEV), None, env=env)
    got = layers.AttentionKernel(env, 0)(q, xk, xv, mask, cache)
    assert torch.equal(cache.cache_k, want_k) and torch.equal(cache.cache_v, want_v)
    assert torch.equal(got, want)
