"""Rotary embedding of the step's keys folded into the KV append (and the
stand-alone rotary launch) against oracle.rope; everything exact: the kernels
follow the oracle's op order (one rounding per op, no fused multiply-add)."""
import numpy as np
import pytest
import torch

from oracle import quant as oq
from oracle import rope as orope

pytestmark = pytest.mark.gpu
DEV = "cuda"


def step_inputs(b, hq, hkv, d, seed, dtype=torch.bfloat16):
  g = torch.Generator().manual_seed(seed)
  xq = (torch.randn((b, 1, hq, d), generator=g) * 2).to(dtype)
  xk = (torch.randn((b, 1, hkv, d), generator=g) * 2).to(dtype)
  xv = (torch.randn((b, 1, hkv, d), generator=g) * 2).to(dtype)
  pos = torch.randint(0, 8192, (b, 1), generator=g)
  freqs = orope.precompute_freqs_cis(d, 8192)[pos]  # (b, 1, d/2) complex64
  return xq, xk, xv, freqs


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(3, 1, 32, 128), (2, 5, 8, 128), (4, 3, 2, 6)])
def test_apply_rotary_emb(shape, dtype):
  from jetstream_pt_amd.layers import apply_rotary_emb
  g = torch.Generator().manual_seed(7)
  b, t, h, d = shape
  xq = torch.randn(shape, generator=g).to(dtype)
  xk = torch.randn((b, t, max(h // 2, 1), d), generator=g).to(dtype)
  pos = torch.randint(0, 4096, (b, t), generator=g)
  freqs = orope.precompute_freqs_cis(d, 4096)[pos]
  gq, gk = apply_rotary_emb(xq.to(DEV), xk.to(DEV), freqs.to(DEV))
  assert gq.dtype == dtype and torch.equal(gq.cpu(), orope.rotate(xq, freqs))
  assert torch.equal(gk.cpu(), orope.rotate(xk, freqs))
  only_q, none = apply_rotary_emb(xq.to(DEV), None, torch.view_as_real(freqs).to(DEV))
  assert none is None and torch.equal(only_q, gq)


@pytest.mark.parametrize("heads,in_dtype", [(8, torch.bfloat16), (32, torch.bfloat16), (5, torch.bfloat16), (8, torch.float32)])
@pytest.mark.parametrize("rounding", ["trunc", "rne"])
@pytest.mark.parametrize("per_head", [False, True])
def test_quantiser_rotates_the_key_first(per_head, rounding, heads, in_dtype):
  from jetstream_pt_amd.quantize import quantize_kv
  b, d = 33, 128
  _, xk, xv, freqs = step_inputs(b, 32, heads, d, 11, in_dtype)
  hs = heads if per_head else 1
  want_k = orope.rotate(xk, freqs).transpose(1, 2)  # (b, heads, 1, d), rotated on the CPU
  ofn = oq.quantize_decode if rounding == "trunc" else oq.quantize_insert
  wc, ws = ofn(want_k, hs, None)
  wvc, wvs = ofn(xv.transpose(1, 2), hs, None)
  kq, vq, ks, vs = quantize_kv(xk.transpose(1, 2).contiguous().to(DEV), xv.transpose(1, 2).contiguous().to(DEV),
                               rounding=rounding, scale_heads=hs, freqs_cis=freqs.to(DEV))
  assert torch.equal(kq.cpu(), wc) and torch.equal(ks.cpu().reshape(-1), ws.reshape(-1)), "rotated key"
  assert torch.equal(vq.cpu(), wvc) and torch.equal(vs.cpu().reshape(-1), wvs.reshape(-1)), "value untouched by the rotation"


@pytest.mark.parametrize("hq,hkv,d", [(32, 8, 128), (16, 4, 128), (8, 1, 128), (16, 16, 128), (32, 32, 128), (4, 2, 64)])
@pytest.mark.parametrize("sdt,per_head", [(torch.float32, False), (torch.bfloat16, True)])
def test_attention_launch_rotates_and_quantises_the_new_token(sdt, per_head, hq, hkv, d):
  """new_key_rope on ragged_mha == the same call on a key rotated beforehand."""
  from jetstream_pt_amd import attention_kernel as ak
  b, s = 7, 256
  g = torch.Generator().manual_seed(13)
  xq, xk, xv, freqs = step_inputs(b, hq, hkv, d, 13)
  end = torch.tensor([0, 5, 128, 200, 256, 33, 31], dtype=torch.int32)
  hs = hkv if per_head else 1
  k = torch.randint(-127, 128, (b, hkv, s, d), generator=g, dtype=torch.int8)
  v = torch.randint(-127, 128, (b, hkv, s, d), generator=g, dtype=torch.int8)
  ks = (torch.rand((b, hs, s, 1), generator=g) * 0.045 + 0.005).to(sdt)
  vs = (torch.rand((b, hs, s, 1), generator=g) * 0.045 + 0.005).to(sdt)
  gq = xq.transpose(1, 2).contiguous().to(DEV)
  raw_k, raw_v = xk.transpose(1, 2).contiguous().to(DEV), xv.transpose(1, 2).contiguous().to(DEV)
  rot_k = orope.rotate(xk, freqs).transpose(1, 2).contiguous().to(DEV)
  gk, gv, gks, gvs, gend = k.to(DEV), v.to(DEV), ks.to(DEV), vs.to(DEV), end.to(DEV)

  def run(key_raw, rope):
    nk, nv = torch.zeros_like(raw_k, dtype=torch.int8), torch.zeros_like(raw_k, dtype=torch.int8)
    nks = torch.zeros((b, hs, 1, 1), dtype=sdt, device=DEV)
    nvs = torch.zeros_like(nks)
    out, (m, l) = ak.ragged_mha(gq, gk, gv, 0, None, gend, None, None, gks, gvs, new_key=nk, new_value=nv,
                                new_k_scaler=nks, new_v_scaler=nvs, new_key_raw=key_raw, new_value_raw=raw_v,
                                new_key_rope=rope)
    return out, m, l, nk, nv, nks, nvs

  want = run(rot_k, None)
  got = run(raw_k, freqs.to(DEV))
  for a, w, name in zip(got, want, "out max denom codes_k codes_v scale_k scale_v".split()):
    assert torch.equal(a, w), name
  wc, ws = oq.quantize_decode(rot_k.cpu(), hs, None if sdt == torch.bfloat16 else sdt)
  assert torch.equal(got[3].cpu(), wc) and torch.equal(got[5].cpu().reshape(-1), ws.to(sdt).reshape(-1))


@pytest.mark.parametrize("b,hq,hkv", [(8, 32, 32), (33, 16, 16), (128, 32, 8)])
@pytest.mark.parametrize("sdt,per_head", [(torch.float32, False), (torch.bfloat16, False), (torch.bfloat16, True)])
def test_many_rotated_tokens_are_quantised_ahead_of_the_launch(sdt, per_head, b, hq, hkv):
  """From batch * kv_heads^2 = 8192 on the token is rotated and quantised by a launch of its own: codes and
  scales are the quantiser's, the outputs those of the call that is given them on the same plan, bit for bit
  (two plans of the same lengths may deal equally long slots out in another order, and with it the order of
  a row's float32 sums)."""
  from jetstream_pt_amd import attention_kernel as ak
  from jetstream_pt_amd.quantize import quantize_kv
  s, d = 96, 128
  g = torch.Generator().manual_seed(5)
  xq, xk, xv, freqs = step_inputs(b, hq, hkv, d, 5)
  end = torch.randint(0, s + 1, (b,), generator=g, dtype=torch.int32).to(DEV)
  hs = hkv if per_head else 1
  k, v = (torch.randint(-127, 128, (b, hkv, s, d), generator=g, dtype=torch.int8).to(DEV) for _ in range(2))
  ks, vs = ((torch.rand((b, hs, s, 1), generator=g) * 0.045 + 0.005).to(sdt).to(DEV) for _ in range(2))
  gq, raw_k, raw_v = (x.transpose(1, 2).contiguous().to(DEV) for x in (xq, xk, xv))
  want = quantize_kv(raw_k, raw_v, rounding="trunc", scale_heads=hs, scale_dtype=sdt, freqs_cis=freqs.to(DEV))
  got = [torch.zeros_like(raw_k, dtype=torch.int8) for _ in range(2)] + [torch.zeros((b, hs, 1, 1), dtype=sdt, device=DEV) for _ in range(2)]
  names = ("new_key", "new_value", "new_k_scaler", "new_v_scaler")
  plan, _ = ak.precompute_ragged_block_indices(end, b, hq, hkv, s)
  end = plan.lengths
  out, stats = ak.ragged_mha(gq, k, v, 0, None, end, plan, None, ks, vs, **dict(zip(names, got)), new_key_raw=raw_k,
                             new_value_raw=raw_v, new_key_rope=freqs.to(DEV))
  for a, w, name in zip(got, want, names):
    assert torch.equal(a.reshape(-1), w.reshape(-1)), name
  given, given_stats = ak.ragged_mha(gq, k, v, 0, None, end, plan, None, ks, vs, **dict(zip(names, got)))
  assert torch.equal(out, given) and all(torch.equal(a, w) for a, w in zip(stats, given_stats))


@pytest.mark.parametrize("b,hq,hkv", [(8, 32, 32), (33, 16, 16), (128, 32, 8)])
@pytest.mark.parametrize("sdt,per_head", [(torch.float32, False), (torch.bfloat16, True)])
def test_many_rotated_tokens_go_to_their_pages(sdt, per_head, b, hq, hkv):
  """The same over pages, from the same number of rows on: codes and scales lie in the token's page and
  nothing else changes (an inactive slot and one without a page among them); outputs as with given codes."""
  from jetstream_pt_amd import attention_kernel as ak
  from jetstream_pt_amd.quantize import quantize_kv
  ps, mp, d = 32, 4, 128
  total, hs = b * mp, hkv if per_head else 1
  g = torch.Generator().manual_seed(6)
  xq, xk, xv, freqs = step_inputs(b, hq, hkv, d, 6)
  lens = torch.randint(1, ps * mp - 1, (b,), generator=g, dtype=torch.int32)
  lens[0], lens[1], lens[2] = 0, ps, 2 * ps - 1
  table = torch.randperm(total, generator=g).reshape(b, mp).to(torch.int32)
  table[3, int(lens[3]) // ps] = -1
  q, raw_k, raw_v = (x.transpose(1, 2).contiguous().to(DEV) for x in (xq, xk, xv))
  pool = [torch.randint(-127, 128, (hkv, total, ps, d), generator=g, dtype=torch.int8) for _ in range(2)]
  pool += [(torch.rand((hs, total, ps), generator=g) * 0.045 + 0.005).to(sdt) for _ in range(2)]
  codes = quantize_kv(raw_k, raw_v, rounding="trunc", scale_heads=hs, scale_dtype=sdt, freqs_cis=freqs.to(DEV))
  codes = [c.contiguous() for c in codes]
  dlens, dtable = lens.to(DEV), table.to(DEV)
  plan = ak.DecodePlan(dlens, b, hq, hkv, page_size=ps, max_pages=mp)
  names = ("new_key", "new_value", "new_k_scaler", "new_v_scaler")

  def run(new):
    pages = [x.to(DEV) for x in pool]
    out = ak.call_paged_attention(None, q.squeeze(2), *pages[:2], dlens, dtable, sm_scale=0.1, k_scaler=pages[2], v_scaler=pages[3],
                                  plan=plan, append=new)
    return [out] + pages

  outputs = [torch.zeros_like(raw_k, dtype=torch.int8) for _ in range(2)] + [torch.zeros((b, hs), dtype=sdt, device=DEV) for _ in range(2)]
  got = run(dict(zip(names, outputs), new_key_raw=raw_k, new_value_raw=raw_v, new_key_rope=freqs.to(DEV)))
  want = run(dict(zip(names, codes)))
  assert all(torch.equal(a.reshape(-1), w.reshape(-1)) for a, w in zip(outputs, codes))
  for a, w in zip(got, want):
    assert torch.equal(a, w)
  written = pool  # what the pages hold with every live slot's token in its place
  for slot, n in enumerate(lens.tolist()):
    page = int(table[slot, n // ps])
    if n > 0 and page >= 0:
      for x, c in zip(written[:2], codes[:2]):
        x[:, page, n % ps] = c[slot, :, 0].cpu()
      for x, c in zip(written[2:], codes[2:]):
        x[:, page, n % ps] = c.reshape(b, hs)[slot].cpu()
  for a, w in zip(got[1:], written):
    assert torch.equal(a.cpu(), w)


def test_orchestration_with_unrotated_keys():
  """Int8KVAttentionKernel(freqs_cis=...) on raw keys == the same kernel on keys
  rotated beforehand, in lazy ragged (fused), eager dense and paged int8 modes;
  caches end up identical."""
  from jetstream_pt_amd import cache_manager as cm
  from jetstream_pt_amd import layers
  from jetstream_pt_amd.environment import JetEngineEnvironment, JetEngineEnvironmentData
  from jetstream_pt_amd.page_attention_manager import PageAttentionManager
  b, hq, hkv, d, s = 4, 16, 8, 128, 128
  xq, xk, xv, freqs = step_inputs(b, hq, hkv, d, 17)
  gq = xq.transpose(1, 2).contiguous().to(DEV)
  raw_k, gv = xk.transpose(1, 2).contiguous().to(DEV), xv.transpose(1, 2).contiguous().to(DEV)
  rot_k = orope.rotate(xk, freqs).transpose(1, 2).contiguous().to(DEV)
  pos = torch.tensor([5, 64, 100, 1], dtype=torch.int32, device=DEV)
  for mode in ("lazy_ragged", "eager_dense", "paged"):
    outs, states = [], []
    for key, fc in ((rot_k, None), (raw_k, freqs.to(DEV))):
      kw = {} if fc is None else {"freqs_cis": fc}
      if mode == "paged":
        env = JetEngineEnvironment(JetEngineEnvironmentData(batch_size=b, paged_attention_total_num_pages=32,
                                                            paged_attention_page_size=32))
        pam = PageAttentionManager(b, 32, 32, 6)
        lens = np.array([5, 64, 100, 1], dtype=np.int32)
        for slot, n in enumerate(lens):
          pam.reserve_pages_insert(slot, int(n))
        pam.fill_new_pages(lens)
        cache = cm.Int8PageKVCacheGenerate.empty((hkv, 32, 32, d), DEV, env)
        cache.page_attention_manager = pam
        cache.page_token_indices = pam.get_page_token_indices(lens)
        cache.cache_k.copy_(torch.randint(-127, 128, cache.cache_k.shape, generator=torch.Generator().manual_seed(3), dtype=torch.int8))
        out = layers.Int8KVAttentionKernel(env, 0)(gq, key, gv, None, cache, **kw)
        st = (cache.cache_k, cache.cache_v, cache.k_scaler, cache.v_scaler)
      else:
        lazy = mode == "lazy_ragged"
        env = JetEngineEnvironment(JetEngineEnvironmentData(
            batch_size=b, num_layers=1, ring_buffer=False, testing=True, lazy_cache_update=lazy, ragged_mha=lazy,
            generate_cache_stacked=lazy, new_cache_stacked=lazy, flash_attention=lazy))
        shape = (1, b, hkv, s, d) if lazy else (b, hkv, s, d)
        cache = cm.Int8KVCacheGenerate.empty(shape, DEV, env)
        cache.cache_k.copy_(torch.randint(-127, 128, shape, generator=torch.Generator().manual_seed(3), dtype=torch.int8))
        cache.input_pos = pos
        mask = torch.full((b, s), float("-inf"), device=DEV)
        for i, p in enumerate(pos.tolist()):
          mask[i, :p + 1] = 0
        out = layers.Int8KVAttentionKernel(env, 0)(gq, key, gv, mask[:, None, None, :], cache, start=None, end=pos, **kw)
        cache.finalize()
        st = (cache.cache_k, cache.cache_v, cache.k_scaler, cache.v_scaler)
      outs.append(out)
      states.append([t.clone() for t in st])
    assert torch.equal(outs[0], outs[1]), mode
    for a, w in zip(states[1], states[0]):
      assert torch.equal(a, w), mode
