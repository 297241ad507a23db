"""The native host side (jetstream_pt_amd._host) against the general Python way: the same call with
inputs it does not take (which go the general way) and with inputs it does gives the same bits; and
the small launches it uses, at their edges."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _step(int8, ring, strided, dim):
  """One layer of a decode step; `strided`: the token's rows are not contiguous."""
  from jetstream_pt_amd import attention_kernel as ak
  from jetstream_pt_amd import cache_manager as cm
  from jetstream_pt_amd import layers
  from jetstream_pt_amd.environment import JetEngineEnvironment, JetEngineEnvironmentData
  g = torch.Generator().manual_seed(31)
  b, hq, hkv, s, nl = 3, 8, 2, 96, 2
  env = JetEngineEnvironment(JetEngineEnvironmentData(batch_size=b, num_layers=nl, ring_buffer=ring))
  kind = cm.Int8KVCacheGenerate if int8 else cm.KVCacheGenerate
  cache = kind.empty((b, hkv, s, dim) if ring else (nl, b, hkv, s, dim), DEV, env)
  for t in (cache.cache_k, cache.cache_v):
    t.copy_(torch.randint(-100, 100, t.shape, generator=g) if int8 else torch.randn(t.shape, generator=g))
  rows = lambda h: torch.randn((b, h, dim, 2), generator=g).to(torch.bfloat16).to(DEV)[..., 0].unsqueeze(2)
  xq, xk, xv = rows(hq).contiguous(), rows(hkv), rows(hkv)
  if not strided:
    xk, xv = xk.contiguous(), xv.contiguous()
  kern = (layers.Int8KVAttentionKernel if int8 else layers.AttentionKernel)(env, 1)
  if ring:
    cache.input_pos = torch.tensor([40], dtype=torch.int32, device=DEV)
    mask = torch.zeros((b, 1, 1, s), device=DEV)
    mask[:, :, :, 41:] = float("-inf")
    out = kern(xq, xk, xv, mask, cache)
  else:
    pos = torch.tensor([0, 33, 95], dtype=torch.int32, device=DEV)
    cache.input_pos = pos
    plan, _ = ak.precompute_ragged_block_indices(pos, b, hq, hkv, s)
    out = kern(xq, xk, xv, None, cache, start=None, end=plan.lengths, ragged_batch_index=plan)
    cache.finalize()
  return [out, cache.cache_k, cache.cache_v] + ([cache.k_scaler, cache.v_scaler] if int8 else [])


@pytest.mark.parametrize("dim", [128, 64])
@pytest.mark.parametrize("ring", [False, True])
@pytest.mark.parametrize("int8", [False, True])
def test_a_step_is_the_same_bits_whichever_way_it_goes(int8, ring, dim):
  for a, b in zip(_step(int8, ring, False, dim), _step(int8, ring, True, dim)):
    assert torch.equal(a, b)


@pytest.mark.parametrize("n,skip", [(1, 0), (15, 1), (16, 0), (4096, 0), (4100, 0), (65552, 16), (1000, 3)])
def test_stash_lines(n, skip):
  from jetstream_pt_amd import _ffi
  src = torch.arange(2 * (n + skip), device=DEV).to(torch.uint8)
  dst = torch.full((2, n + skip + 64), 77, dtype=torch.uint8, device=DEV)
  _ffi.check(_ffi.lib.jpt_kv_stash_lines(dst[0, skip:].data_ptr(), src[skip:].data_ptr(), dst[1, skip:].data_ptr(),
                                         src[n + skip:].data_ptr(), n, _ffi.stream()))
  assert torch.equal(dst[0, skip:skip + n], src[skip:skip + n]) and torch.equal(dst[1, skip:skip + n], src[n + skip:][:n])
  assert bool((dst[:, :skip] == 77).all() and (dst[:, skip + n:] == 77).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("seq,lo,hi,wrap", [(1, 0, 1, False), (300, 0, 300, False), (300, 17, 256, False), (300, 290, 5, True), (512, 100, 100, True)])
def test_insert_state(seq, lo, hi, wrap, dtype):
  from jetstream_pt_amd import _host
  mask = torch.ones((3, seq), dtype=dtype, device=DEV)
  rows = [torch.full((3,), -5, dtype=torch.int32, device=DEV) for _ in range(3)]
  assert _host.insert_state(mask, *rows, 1, 7, 9, lo, hi, wrap)
  x = torch.arange(seq)
  live = ((x >= lo) | (x < hi)) if wrap else ((x >= lo) & (x < hi))
  assert torch.equal(mask[1].cpu(), torch.where(live, 0.0, float("-inf")).to(dtype))
  assert bool((mask[0] == 1).all() and (mask[2] == 1).all())
  assert [r.tolist() for r in rows] == [[-5, 7, -5], [-5, 9, -5], [-5, 1, -5]]


@pytest.mark.parametrize("dim,seq", [(128, 256), (128, 250), (64, 256)])
def test_a_fresh_plan_needs_no_cleared_workspace(dim, seq):
  """torch hands out used memory: a plan on a workspace full of other data gives the same outputs
  and no status bit (seq 250 and dim 64 run on the kernel whose counters lie in the state block)."""
  from jetstream_pt_amd import attention_kernel as ak
  g = torch.Generator().manual_seed(7)
  b, hq, hkv = 5, 8, 4
  q = torch.randn((b, hq, 1, dim), generator=g).to(torch.bfloat16).to(DEV)
  k, v = (torch.randn((b, hkv, seq, dim), generator=g).to(torch.bfloat16).to(DEV) for _ in range(2))
  end = torch.tensor([seq - 1, 0, 31, 100, 129], dtype=torch.int32, device=DEV)
  outs = []
  for fill in (0, 255, 1):
    torch.cuda.synchronize()
    junk = torch.full((64 << 20,), fill, dtype=torch.uint8, device=DEV)
    del junk  # the next allocation is cut from it
    plan, _ = ak.precompute_ragged_block_indices(end, b, hq, hkv, seq)
    outs.append(ak.ragged_mha(q, k, v, 0, None, plan.lengths, plan)[0])
    assert ak.check_status(plan) == 0
  assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


@pytest.mark.parametrize("b,hq,hkv,d,s", [(1, 32, 8, 128, 2048), (5, 8, 8, 128, 512), (3, 8, 1, 128, 4096), (300, 16, 1, 128, 64),
                                          (4, 8, 4, 64, 256), (3, 4, 2, 128, 333)])
def test_lazy_bf16_step_leaves_the_token_in_the_stash(b, hq, hkv, d, s):
  """The attention launch leaves the rows it was given in the layer's stash and nowhere else: empty, full and
  cut slots, and shapes of the kernels beside the streaming one; outputs as without it, on the same plan."""
  from jetstream_pt_amd import attention_kernel as ak, cache_manager as cm, layers
  from jetstream_pt_amd.environment import JetEngineEnvironment, JetEngineEnvironmentData
  g = torch.Generator().manual_seed(70 + b)
  env = JetEngineEnvironment(JetEngineEnvironmentData(batch_size=b, num_layers=3, cache_sequence_length=s, ring_buffer=False))
  cache = cm.KVCacheGenerate.empty((3, b, hkv, s, d), DEV, env)
  for t in (cache.cache_k, cache.cache_v):
    t.copy_(torch.randn(t.shape, generator=g).to(torch.bfloat16))
  q, k, v = (torch.randn((b, h, 1, d), generator=g).to(torch.bfloat16).to(DEV) for h in (hq, hkv, hkv))
  lens = torch.randint(0, s + 1, (b,), generator=g, dtype=torch.int32)
  lens[0] = s
  if b > 1:
    lens[1] = 0
  cache.input_pos = lens.to(DEV)
  for t in (cache.new_ks, cache.new_vs):
    t.fill_(7.0)
  plan, _ = ak.precompute_ragged_block_indices(cache.input_pos, b, hq, hkv, s)
  want, _ = ak.ragged_mha(q, cache.cache_k, cache.cache_v, 1, None, plan.lengths, plan, None, new_key=k, new_value=v)
  got = layers.AttentionKernel(env, 1)(q, k, v, None, cache, start=None, end=plan.lengths, ragged_batch_index=plan)
  assert torch.equal(got.reshape(-1), want.reshape(-1))
  for stash, row in ((cache.new_ks, k), (cache.new_vs, v)):
    assert torch.equal(stash[1], row)
    assert torch.all(stash[0] == 7.0) and torch.all(stash[2] == 7.0)


def test_stacks_of_layers_are_taken_only_where_a_layer_is_named():
  """Five-dimensional keys without a layer, and stacks beside tensors of one layer, are refused; a named
  layer of a stack gives that layer's bits."""
  from jetstream_pt_amd import attention_kernel as ak
  g = torch.Generator().manual_seed(12)
  b, hq, hkv, s, d = 2, 8, 2, 64, 128
  q = torch.randn((b, hq, 1, d), generator=g).to(torch.bfloat16).to(DEV)
  k, v = (torch.randn((3, b, hkv, s, d), generator=g).to(torch.bfloat16).to(DEV) for _ in range(2))
  codes = torch.randint(-127, 128, (3, b, hkv, s, d), generator=g, dtype=torch.int8).to(DEV)
  scales = torch.rand((3, b, 1, s, 1), generator=g).to(DEV)
  lens = torch.tensor([64, 5], dtype=torch.int32, device=DEV)
  refused = [lambda: ak.dense_attention(q, k, v), lambda: ak.dense_attention(q, codes, codes, scales, scales),
             lambda: ak.flash_attention(q, codes[1], codes[1], 1, scales, scales),
             lambda: ak.flash_attention(q, codes, codes, 1, scales[1], scales),
             lambda: ak.ragged_mha(q, k[1], v, 1, None, lens),
             lambda: ak.call_paged_attention(None, q.squeeze(2), k.reshape(3, hkv, b * 2, s // 2, d), v.reshape(3, hkv, b * 2, s // 2, d), lens,
                                             torch.zeros((b, 2), dtype=torch.int32, device=DEV))]
  for call in refused:
    with pytest.raises(ValueError):
      call()
  for a, w in zip(ak.flash_attention(q, codes, codes, 1, scales, scales)[1], ak.flash_attention(q, codes[1], codes[1], 0, scales[1], scales[1])[1]):
    assert torch.equal(a, w)
  assert torch.equal(ak.ragged_mha(q, k, v, 2, None, lens)[0], ak.ragged_mha(q, k[2], v[2], 0, None, lens)[0])


@pytest.mark.parametrize("int8_kernel", [False, True])
@pytest.mark.parametrize("mode", ["ring", "lazy", "paged"])
def test_kernels_and_caches_that_do_not_belong_together_are_refused(mode, int8_kernel):
  """The bf16 kernel on an int8 cache and the int8 kernel on a bf16 one raise, as they do launch by launch."""
  from jetstream_pt_amd import attention_kernel as ak, cache_manager as cm, layers
  from jetstream_pt_amd.environment import JetEngineEnvironment, JetEngineEnvironmentData
  from jetstream_pt_amd.page_attention_manager import DevicePageAttentionManager
  b, hq, hkv, s, d, nl = 2, 8, 2, 64, 128, 2
  env = JetEngineEnvironment(JetEngineEnvironmentData(batch_size=b, num_layers=nl, ring_buffer=mode == "ring",
                                                      paged_attention_total_num_pages=8 if mode == "paged" else 0, paged_attention_page_size=32))
  kern = (layers.Int8KVAttentionKernel if int8_kernel else layers.AttentionKernel)(env, 0)
  lens = torch.tensor([3, 40], dtype=torch.int32, device=DEV)
  kw = {}
  if mode == "paged":
    pam = DevicePageAttentionManager(b, 8, 32, 4, device=DEV)
    pam.reserve_pages_insert_many(torch.arange(b, dtype=torch.int32), lens.cpu())
    pages = [torch.zeros((hkv, 8, 32, d), dtype=torch.bfloat16 if int8_kernel else torch.int8, device=DEV) for _ in range(2)]
    scales = [torch.ones((1, 8, 32), device=DEV) for _ in range(2)]
    cache = cm.PageKVCacheGenerate(*pages, pam, None, env=env) if int8_kernel else cm.Int8PageKVCacheGenerate(*pages, *scales, pam, None, env=env)
    cache.page_token_indices = pam.decode_step(lens)
  else:
    kind = cm.KVCacheGenerate if int8_kernel else cm.Int8KVCacheGenerate
    cache = kind.empty((b, hkv, s, d) if mode == "ring" else (nl, b, hkv, s, d), DEV, env)
    cache.input_pos = torch.tensor([40], dtype=torch.int32, device=DEV) if mode == "ring" else lens
    if mode == "lazy":
      plan, _ = ak.precompute_ragged_block_indices(lens, b, hq, hkv, s)
      kw = dict(start=None, end=plan.lengths, ragged_batch_index=plan)
  q, k, v = (torch.ones((b, h, 1, d), dtype=torch.bfloat16, device=DEV) for h in (hq, hkv, hkv))
  with pytest.raises(ValueError, match="unpack"):
    kern(q, k, v, torch.zeros((b, 1, 1, s), device=DEV) if mode == "ring" else None, cache, **kw)


@pytest.mark.parametrize("int8", [False, True])
def test_how_a_cache_is_updated_is_the_caches_to_say(int8):
  """A cache that stashes its lines, under a kernel whose environment writes at once: the cache stashes."""
  from jetstream_pt_amd import cache_manager as cm, layers
  from jetstream_pt_amd.environment import JetEngineEnvironment, JetEngineEnvironmentData
  b, hq, hkv, s, d = 2, 8, 2, 64, 128
  eager, lazy = (JetEngineEnvironment(JetEngineEnvironmentData(batch_size=b, num_layers=1, testing=True, lazy_cache_update=x)) for x in (False, True))
  cache = (cm.Int8KVCacheGenerate if int8 else cm.KVCacheGenerate).empty((b, hkv, s, d), DEV, lazy)
  cache.input_pos = torch.tensor([40], dtype=torch.int32, device=DEV)
  q, k, v = (torch.ones((b, h, 1, d), dtype=torch.bfloat16, device=DEV) for h in (hq, hkv, hkv))
  (layers.Int8KVAttentionKernel if int8 else layers.AttentionKernel)(eager, 0)(q, k, v, torch.zeros((b, 1, 1, s), device=DEV), cache)
  assert torch.all(cache.cache_k == 0) and torch.all(cache.new_ks != 0)


@pytest.mark.parametrize("mode", ["ring", "lazy", "paged"])
def test_an_attention_put_in_the_kernels_place_is_the_one_that_runs(mode):
  from jetstream_pt_amd import attention_kernel as ak, cache_manager as cm, layers
  from jetstream_pt_amd.environment import JetEngineEnvironment, JetEngineEnvironmentData
  from jetstream_pt_amd.page_attention_manager import DevicePageAttentionManager
  b, hq, hkv, s, d, nl = 2, 8, 2, 64, 128, 2
  env = JetEngineEnvironment(JetEngineEnvironmentData(batch_size=b, num_layers=nl, ring_buffer=mode == "ring",
                                                      paged_attention_total_num_pages=8 if mode == "paged" else 0, paged_attention_page_size=32))
  kern = layers.AttentionKernel(env, 0)
  lens = torch.tensor([3, 40], dtype=torch.int32, device=DEV)
  kw, name = {}, {"ring": "dense_attention", "lazy": "ragged_attention_new", "paged": "page_attention"}[mode]
  ran = []
  own = getattr(kern, name)
  setattr(kern, name, lambda *a, **k: ran.append(name) or own(*a, **k))
  if mode == "paged":
    pam = DevicePageAttentionManager(b, 8, 32, 4, device=DEV)
    pam.reserve_pages_insert_many(torch.arange(b, dtype=torch.int32), lens.cpu())
    cache = cm.PageKVCacheGenerate(*(torch.zeros((hkv, 8, 32, d), dtype=torch.bfloat16, device=DEV) for _ in range(2)), pam, None, env=env)
    cache.page_token_indices = pam.decode_step(lens)
  else:
    cache = cm.KVCacheGenerate.empty((b, hkv, s, d) if mode == "ring" else (nl, b, hkv, s, d), DEV, env)
    cache.input_pos = torch.tensor([40], dtype=torch.int32, device=DEV) if mode == "ring" else lens
    if mode == "lazy":
      plan, _ = ak.precompute_ragged_block_indices(lens, b, hq, hkv, s)
      kw = dict(start=None, end=plan.lengths, ragged_batch_index=plan)
  q, k, v = (torch.ones((b, h, 1, d), dtype=torch.bfloat16, device=DEV) for h in (hq, hkv, hkv))
  kern(q, k, v, torch.zeros((b, 1, 1, s), device=DEV) if mode == "ring" else None, cache, **kw)
  assert ran == [name]


def test_other_threads_run_while_the_library_does():
  """Every call into the library is made without the interpreter's lock: in the library's place stands the
  interpreter's own question whether this thread holds it, whose "no" is the library's OK."""
  import ctypes
  from jetstream_pt_amd import _ffi, _host, attention_kernel as ak
  held = ctypes.cast(ctypes.pythonapi.PyGILState_Check, ctypes.c_void_p).value
  asked = {name: at if name in ("jpt_attn_workspace_bytes", "jpt_attn_kernel") else held for name, at in _ffi.addresses().items()}

  def status(code):
    raise AssertionError("the interpreter's lock was held")

  b, hq, hkv, s, d, nl, t = 2, 8, 2, 64, 128, 2, 16
  bf16 = lambda *shape: torch.zeros(shape, dtype=torch.bfloat16, device=DEV)
  i8 = lambda *shape: torch.zeros(shape, dtype=torch.int8, device=DEV)
  lens, table = (torch.ones(shape, dtype=torch.int32, device=DEV) for shape in ((b,), (b, 2)))
  q, row, mask = bf16(b, hq, 1, d), bf16(b, hkv, 1, d), torch.zeros((b, s), device=DEV)
  stack, lines, one = bf16(nl, b, hkv, s, d), bf16(nl, b, hkv, 1, d), bf16(b, hkv, s, d)
  scale, new_scale, layer_scale = (torch.ones(shape, device=DEV) for shape in ((nl, b, 1, s, 1), (nl, b, 1, 1, 1), (b, 1, s, 1)))
  pages, prompt = bf16(hkv, 8, 32, d), [(bf16(1, hkv, t, d), bf16(1, hkv, t, d))] * nl
  torch.cuda.synchronize()
  _host.bind(asked, status, ak._shared_workspace_buf, ak._split_workspace_buf, ak._dense_workspace_buf)
  try:
    done = [
        _host.attend(0, q, one, one, -1, lens, None, None, None, None, None, None, None, None, None, None, None, 0, None, False, False, None),
        _host.lazy_step(q, row, row, stack, stack, None, None, lines, lines, None, None, 0, lens, None, 0, None),
        _host.lazy_step(q, row, row, stack.char(), stack.char(), scale, scale, lines.char(), lines.char(), new_scale, new_scale, 0, lens, None, 0, None),
        _host.eager_step(q, row, row, mask[:, None, None], i8(b, hkv, s, d), i8(b, hkv, s, d), layer_scale, layer_scale, lens, False, 0, None),
        _host.eager_step(q, row, row, mask[:, None, None], one, one, None, None, lens, False, 0, None),
        _host.paged_step(q, row, row, pages, pages, None, None, lens, table, None, 1.0, 0, None),
        _host.scatter_lines((stack,), (lines,), lens, b, nl, b, s),
        _host.insert_layers(prompt, [(stack, stack)], None, None, 0, 0, 1),
        _host.plan(lens, b, hq, hkv, 1, s, 0, 0, None),
        _host.insert_state(mask, lens, lens, lens, 0, 0, 1, 0, 1, False),
    ]
  finally:
    _host.bind(_ffi.addresses(), _ffi.check, ak._shared_workspace_buf, ak._split_workspace_buf, ak._dense_workspace_buf)
  assert all(x is not None for x in done)


def test_two_threads_on_streams_of_their_own():
  """Steps through the native host side from two threads at once, each on its own stream: the bits of the
  same steps one after the other."""
  import threading
  from jetstream_pt_amd import attention_kernel as ak
  g = torch.Generator().manual_seed(77)
  b, hq, hkv, s, d = 4, 8, 2, 512, 128
  work = []
  for dim in (d, 64):
    q = torch.randn((b, hq, 1, dim), generator=g).to(torch.bfloat16).to(DEV)
    k, v = (torch.randn((b, hkv, s, dim), generator=g).to(torch.bfloat16).to(DEV) for _ in range(2))
    work.append((q, k, v, torch.zeros((b, 1, 1, s), device=DEV)))
  run = lambda q, k, v, mask: ak.dense_attention(q, k, v, mask=mask)
  want = [run(*w) for w in work]
  torch.cuda.synchronize()
  outs, errors = [[], []], []

  def steps(i):
    try:
      with torch.cuda.stream(torch.cuda.Stream()):
        for n in range(50):
          outs[i].append(run(*work[(i + n) % 2]))
        torch.cuda.current_stream().synchronize()
    except Exception as e:  # pylint: disable=broad-except
      errors.append(e)

  threads = [threading.Thread(target=steps, args=(i,)) for i in range(2)]
  for t in threads:
    t.start()
  for t in threads:
    t.join()
  assert not errors
  for i in range(2):
    for n, o in enumerate(outs[i]):
      assert torch.equal(o, want[(i + n) % 2])


def test_inserts_refuse_what_they_refused():
  """Prompts without their batch dimension into pages, stacks of pages, and masks of another length."""
  from jetstream_pt_amd import insert as pi
  from jetstream_pt_amd.environment import JetEngineEnvironment, JetEngineEnvironmentData
  from jetstream_pt_amd.page_attention_manager import PageAttentionManager
  hkv, t, d, ps, nl = 2, 40, 128, 32, 2
  bf16 = lambda *shape: torch.ones(shape, dtype=torch.bfloat16, device=DEV)
  ids = torch.tensor([3, 5], dtype=torch.int32, device=DEV)
  pages = [(bf16(hkv, 8, ps, d), bf16(hkv, 8, ps, d)) for _ in range(nl)]
  flat = [(bf16(hkv, t, d) * 2, bf16(hkv, t, d) * 2) for _ in range(nl)]
  whole = [(k[None], v[None]) for k, v in flat]
  pam = PageAttentionManager(2, 8, ps, 4)
  with pytest.raises((ValueError, IndexError)):
    pam.insert_prefill_cache(flat, pages, ids)
  with pytest.raises(ValueError):
    pi.insert_prefix_pages_copy(whole, [(bf16(nl, hkv, 8, ps, d), bf16(nl, hkv, 8, ps, d))], ids)
  assert all(bool((x == 1).all()) for pair in pages for x in pair)
  assert pi.insert_prefix_pages_copy(whole, pages, ids) and all(bool((x[:, 3] == 2).all()) for pair in pages for x in pair)
  env = JetEngineEnvironment(JetEngineEnvironmentData(batch_size=2, num_layers=nl, cache_sequence_length=64, ring_buffer=False))
  mask = torch.zeros((2, 96), device=DEV)
  with pytest.raises(RuntimeError):
    pi.insert(env, whole, t, [(bf16(nl, 2, hkv, 64, d), bf16(nl, 2, hkv, 64, d))], None, 1, mask=mask)
  assert bool((mask == 0).all())


def test_a_scale_that_is_not_a_number_is_not_the_default():
  from jetstream_pt_amd import attention_kernel as ak
  g = torch.Generator().manual_seed(3)
  q = torch.randn((1, 4, 128), generator=g).to(torch.bfloat16).to(DEV)
  pages = torch.randn((2, 4, 32, 128), generator=g).to(torch.bfloat16).to(DEV)
  lens, table = torch.tensor([20], dtype=torch.int32, device=DEV), torch.tensor([[1, 2]], dtype=torch.int32, device=DEV)
  assert bool(ak.call_paged_attention(None, q, pages, pages, lens, table, sm_scale=float("nan")).isnan().all())
  assert bool(ak.call_paged_attention(None, q, pages, pages, lens, table, sm_scale=0.1).isfinite().all())


@pytest.mark.parametrize("b,fill", [(5, 255), (5, 1), (4200, 255)])
def test_a_fresh_plans_workspace_serves_the_kernel_whose_counters_it_holds(b, fill):
  """At the library's entries: a workspace full of other data, planned as a fresh one, then a call whose
  kernel counts in the state block (batches beyond the planner's have no plan: the block is cleared)."""
  from jetstream_pt_amd import _ffi, attention_kernel as ak
  g = torch.Generator().manual_seed(8)
  hq, hkv, s, d = 8, 4, 250, 128
  q = torch.randn((b, hq, 1, d), generator=g).to(torch.bfloat16).to(DEV)
  k, v = (torch.randn((b, hkv, s, d), generator=g).to(torch.bfloat16).to(DEV) for _ in range(2))
  end = torch.randint(0, s + 1, (b,), generator=g, dtype=torch.int32).to(DEV)
  want = ak.ragged_mha(q, k, v, 0, None, end)[0]
  out = torch.empty_like(q)
  a = _ffi.AttnArgs(q=_ffi.ptr(q), k=_ffi.ptr(k), v=_ffi.ptr(v), lengths=_ffi.ptr(end), out=_ffi.ptr(out), batch=b, q_heads=hq, kv_heads=hkv,
                    q_rows=1, dim=d, seq=s, q_dtype=_ffi.BF16, kv_dtype=_ffi.BF16, sm_scale=1.0 / d ** 0.5)
  assert _ffi.lib.jpt_attn_kernel(a, 0) == _ffi.ATTN_SPLIT
  ws = torch.full((_ffi.lib.jpt_attn_workspace_bytes(a),), fill, dtype=torch.uint8, device=DEV)
  a.workspace, a.workspace_bytes = _ffi.ptr(ws), ws.numel()
  _ffi.check(_ffi.lib.jpt_attn_plan_fresh(a, 0, _ffi.stream()))
  for _ in range(3):
    out.zero_()
    _ffi.check(_ffi.lib.jpt_attn_ragged(a, _ffi.stream()))
    assert torch.equal(out.reshape(want.shape), want)


def test_rows_that_do_not_belong_together_are_refused():
  """What a kernel walks side by side, or by another tensor's shape, agrees with it: everything else is
  refused before a launch (a bf16 value read as the float32 its key is ends past its rows)."""
  from jetstream_pt_amd import attention_kernel as ak, cache_manager as cm, insert as pi, layers
  from jetstream_pt_amd.environment import JetEngineEnvironment, JetEngineEnvironmentData
  from jetstream_pt_amd.page_attention_manager import PageAttentionManager
  from jetstream_pt_amd.quantize import quantize_kv
  b, hq, hkv, s, d, ps, total, nl, t = 2, 4, 2, 64, 128, 32, 8, 2, 40
  z = lambda *shape, dt=torch.bfloat16: torch.zeros(shape, dtype=dt, device=DEV)
  i8, f32 = torch.int8, torch.float32
  row, q, wide = z(b, hkv, 1, d), z(b, hq, 1, d), z(b, hkv, 1, d, dt=f32)
  few = z(b, 1, 1, d)  # a head short
  ring = JetEngineEnvironment(JetEngineEnvironmentData(batch_size=b, num_layers=nl))
  lazy = JetEngineEnvironment(JetEngineEnvironmentData(batch_size=b, num_layers=nl, ring_buffer=False))
  pos, lens, idx = (torch.tensor(x, dtype=torch.int32, device=DEV) for x in ([3], [3, 40], [[1, 2], [3, 8], [0, 1]]))
  mask = z(b, 1, 1, s, dt=f32)

  def step(env, kind, k, v, **kw):
    cache = kind.empty((b, hkv, s, d) if env is ring else (nl, b, hkv, s, d), DEV, env, **kw)
    cache.input_pos = pos if env is ring else lens
    kern = (layers.Int8KVAttentionKernel if kind is cm.Int8KVCacheGenerate else layers.AttentionKernel)(env, 0)
    kern(q, k, v, mask if env is ring else None, cache, start=None, end=lens)

  def paged(k, v, int8, scale_shape=(1, total, ps), pages_v=(hkv, total, ps, d)):
    pam = PageAttentionManager(b, total, ps, 4)
    dt = i8 if int8 else torch.bfloat16
    pages = [z(hkv, total, ps, d, dt=dt), z(*pages_v, dt=dt)]
    scales = [z(*scale_shape, dt=f32), z(*scale_shape, dt=f32)]
    cache = cm.Int8PageKVCacheGenerate(*pages, *scales, pam, idx) if int8 else cm.PageKVCacheGenerate(*pages, pam, idx)
    cache.update(k, v)

  prompt, wide_prompt = z(1, hkv, t, d), z(1, hkv, t, d, dt=f32)
  dense8, dense_scale = lambda: z(b, hkv, s, d, dt=i8), z(b, 1, s, 1, dt=f32)
  pages8, scale_pages = z(hkv, total, ps, d, dt=i8), z(1, total, ps, dt=f32)
  stack8, stack_scale, prompts = z(nl, hkv, total, ps, d, dt=i8), z(nl, 1, total, ps, dt=f32), z(nl, hkv, t, d)
  ids = torch.tensor([1, 2], dtype=torch.int32, device=DEV)
  codes, scale = z(b, hkv, s, d, dt=i8), z(b, 1, s, 1, dt=f32)
  refused = [
      lambda: quantize_kv(row, wide), lambda: quantize_kv(wide, row),
      lambda: step(ring, cm.Int8KVCacheGenerate, wide, row, scale_dtype=f32), lambda: step(ring, cm.Int8KVCacheGenerate, row, few),
      lambda: step(ring, cm.Int8KVCacheGenerate, few, few), lambda: step(ring, cm.KVCacheGenerate, row, few),
      lambda: step(ring, cm.KVCacheGenerate, few, few), lambda: step(lazy, cm.Int8KVCacheGenerate, wide, row, scale_dtype=f32),
      lambda: step(lazy, cm.Int8KVCacheGenerate, few, few),
      lambda: paged(wide, row, True), lambda: paged(row, wide, True), lambda: paged(few, few, True), lambda: paged(row, few, True),
      lambda: paged(row, row, True, scale_shape=(1, total, 1)), lambda: paged(row, row, True, pages_v=(hkv, 2, ps, d)),
      lambda: paged(row, few, False), lambda: paged(few, few, False), lambda: paged(row, row, False, pages_v=(hkv, 2, ps, d)),
      lambda: pi.insert_prefix_caches([(wide_prompt, prompt)], [(dense8(), dense8())], [(dense_scale, dense_scale)], 0, 0),
      lambda: pi.insert_prefix_caches([(prompt, prompt[:, :, :8])], [(dense8(), dense8())], [(dense_scale, dense_scale)], 0, 0),
      lambda: pi.insert_prefix_caches([(prompt, prompt)], [(dense8(), dense8()[:1])], [(dense_scale, dense_scale)], 0, 0),
      lambda: pi.insert_prefix_caches([(prompt, prompt)], [(dense8(), dense8())], [(dense_scale[:, :, :8].contiguous(), dense_scale[:, :, :8].contiguous())], 0, 0),
      lambda: pi.insert_prefix_pages_int8([(wide_prompt, prompt)], [(pages8, pages8)], [(scale_pages, scale_pages)], ids),
      lambda: pi.insert_prefix_pages_int8([(prompt, prompt)], [(pages8, pages8[:1])], [(scale_pages, scale_pages)], ids),
      lambda: pi.insert_prefix_pages_int8([(prompt, prompt)], [(pages8, pages8)], [(scale_pages, scale_pages[:, :2])], ids),
      lambda: pi.insert_prefix_pages_int8_stacked(prompts.float(), prompts, stack8, stack8, stack_scale, stack_scale, ids),
      lambda: pi.insert_prompts_pages_int8_stacked([(prompts, prompts[:, :, :8])], stack8, stack8, stack_scale, stack_scale, [ids]),
      lambda: pi.insert_prefix_pages_copy([(prompt, prompt[:, :, :8])] * 2, [(z(hkv, total, ps, d), z(hkv, total, ps, d))] * 2, ids),
      lambda: PageAttentionManager(b, total, ps, 4).insert_prefill_cache([(prompt, prompt[:, :, :8])], [(z(hkv, total, ps, d), z(hkv, total, ps, d))], ids),
      lambda: ak.dense_attention(q, codes, codes, scale[:1], scale[:1]), lambda: ak.dense_attention(q, codes, codes, scale[:, :, :8].contiguous(), scale[:, :, :8].contiguous()),
      lambda: ak.ragged_mha(q, codes, codes, 0, None, lens, None, None, scale, scale, new_key=row.char(), new_value=few.char(),
                            new_k_scaler=scale[:, :, :1].contiguous(), new_v_scaler=scale[:, :, :1].contiguous()),
      lambda: ak.ragged_mha(q, codes, codes, 0, None, lens, None, None, scale, scale, new_key=row.char(), new_value=row.char(),
                            new_k_scaler=scale[:1, :, :1].contiguous(), new_v_scaler=scale[:1, :, :1].contiguous()),
  ]
  for call in refused:
    with pytest.raises(ValueError):
      call()
