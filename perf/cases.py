"""The work that is timed: what a serving loop has this framework do.

Five kinds of pass, each through the package's own entry points:

  step     one decode step of a few layers over a dense cache: the step's split plan, every
           layer's cache update and attention, finalize (left-aligned mode, ring=False), or the
           mask update, every layer's eager line write and masked attention (ring buffer)
  paged    one decode step over paged caches with the device-resident allocator: requests
           replaced (churn), page allocation, every layer's append and attention
  insert   one prompt's keys and values of all layers into its slot of a dense cache
  pages    one prompt's keys and values of all layers into pages handed out by the host allocator
  prefill  the prompt's own attention, causal, before its keys and values are inserted

A pass leaves its state as it found it but for the values it writes, so it can be repeated: a
step does not advance the positions, and paged slots that stay do not sit on a page boundary
(one that does would take a page more at every pass).  Layers are fewer than a model's where the
cache would not leave room for several states; the step's plan and its finalize are shared by
them as they are by a model's.
"""

import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "jetstream-pytorch_amd")  # the package's folder in the working tree
if _PACKAGE not in sys.path:
  sys.path.insert(0, _PACKAGE)

from jetstream_pt_amd import attention_kernel as ak  # noqa: E402
from jetstream_pt_amd import cache_manager as cm  # noqa: E402
from jetstream_pt_amd import decode_state  # noqa: E402
from jetstream_pt_amd import insert as prompt_insert  # noqa: E402
from jetstream_pt_amd import layers as attn_layers  # noqa: E402
from jetstream_pt_amd.environment import JetEngineEnvironment, JetEngineEnvironmentData  # noqa: E402
from jetstream_pt_amd.page_attention_manager import DevicePageAttentionManager, PageAttentionManager  # noqa: E402

DEV = "cuda"
BF16 = torch.bfloat16


def _step(name, batch, heads, kv_heads, dim, seq, layers, int8, ring, rope, scale32, lens, mid):
  return dict(name=name, kind="step", batch=batch, heads=heads, kv_heads=kv_heads, dim=dim, seq=seq, layers=layers,
              int8=int8, ring=ring, rope=rope, scale32=scale32, lens=lens, mid=mid)


def _paged(name, batch, heads, kv_heads, page, pages, max_pages, layers, int8, churn, lens, mid, prompt):
  return dict(name=name, kind="paged", batch=batch, heads=heads, kv_heads=kv_heads, dim=128, page=page, pages=pages,
              max_pages=max_pages, layers=layers, int8=int8, churn=churn, lens=lens, mid=mid, prompt=prompt)


def listed():
  return [
      # One interactive user: a short conversation, one slot; launches and host work count.
      _step("step_one_user", 1, 32, 8, 128, 2048, 8, False, False, False, False, "lognormal", 300),
      # The headline workload: a Llama-3-8B server, int8 cache, 128 slots of very different lengths.
      _step("step_int8_gqa", 128, 32, 8, 128, 8192, 8, True, False, False, True, "lognormal", 400),
      # The same mode with as many KV heads as query heads (Llama-2-7B), the reference's bf16 scales,
      # the rotary embedding left to the launch that quantises the key.
      _step("step_int8_mha", 96, 32, 32, 128, 2048, 4, True, False, True, False, "uniform", 1024),
      # Ring buffer, bf16, the reference's default mode: line write, attention under a mask.
      _step("step_ring_bf16", 8, 32, 32, 128, 1024, 8, False, True, False, False, "uniform", 512),
      # Ring buffer with the quantised cache.
      _step("step_ring_int8", 64, 32, 8, 128, 2048, 8, True, True, False, False, "uniform", 1024),
      # Heads of 256 elements (Gemma-7B's shape), int8 cache, left-aligned.
      _step("step_dim256", 48, 16, 16, 256, 1024, 4, True, False, False, False, "uniform", 512),
      # Llama-2-70B on one GPU: bf16 pages, every slot's token appended by the attention launch.
      _paged("paged_bf16", 256, 64, 8, 64, 32768, 128, 2, False, 0, "uniform", 1024, 0),
      # Continuous batching over int8 pages: sixteen requests replaced in the step.
      _paged("paged_int8_churn", 256, 32, 8, 64, 16384, 64, 4, True, 16, "lognormal", 600, 1024),
      # A prompt's insert: quantised into a dense slot; copied into pages.
      dict(name="insert_int8", kind="insert", batch=8, kv_heads=8, dim=128, seq=2048, layers=32, int8=True,
           scale32=False, tokens=1000, ring=False),
      dict(name="insert_pages", kind="pages", kv_heads=8, dim=128, page=64, pages=512, layers=16, tokens=1500),
      # Prefill: an ordinary prompt; a long one through the quantised mode's kernel.
      dict(name="prefill", kind="prefill", batch=1, heads=32, kv_heads=8, dim=128, tokens=1024, int8=False, mask32=False),
      dict(name="prefill_long", kind="prefill", batch=1, heads=32, kv_heads=8, dim=128, tokens=3500, int8=True, mask32=False),
  ]


_HEADS = [(32, 8), (32, 32), (64, 8), (16, 16), (8, 1), (28, 4), (8, 8)]


def _spread(rng, lo, hi):
  """An integer of [lo, hi], spread over its logarithm."""
  return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
  kind = rng.choice(["step", "step", "step", "paged", "paged", "insert", "pages", "prefill", "prefill"])
  heads, kv_heads = rng.choice(_HEADS)
  if kind == "step":
    dim = rng.choice([128, 128, 128, 64, 256])
    int8, ring = rng.random() < 0.6, rng.random() < 0.3
    batch, seq = _spread(rng, 1, 160), 128 * _spread(rng, 4, 64)
    layers = rng.randint(2, 8)
    per_slot = layers * kv_heads * seq * dim * (2 if int8 else 4)
    batch = max(1, min(batch, int(16e9 // per_slot)))  # what a state may hold
    c = _step("", batch, heads, kv_heads, dim, seq, layers, int8, ring, int8 and not ring and rng.random() < 0.5,
              rng.random() < 0.5, rng.choice(["uniform", "lognormal"]), rng.randint(60, max(100, seq // 4)))
    if dim != 128:  # no more work than the listed cases
      c["batch"] = max(1, min(c["batch"], int(c["batch"] * 1.5e10 // work(c)["flops"]), int(4e10 // (layers * seq * heads * dim * 4))))
  elif kind == "paged":
    int8, page, batch = rng.random() < 0.5, rng.choice([32, 64, 64, 128]), _spread(rng, 2, 256)
    layers = rng.randint(2, 4)
    most = rng.choice([1024, 2048, 4096])  # positions a slot may hold
    per_slot = layers * kv_heads * most * 128 * (2 if int8 else 4)
    batch = max(2, min(batch, int(16e9 // per_slot)))
    churn = min(batch // 2, rng.randint(1, 16)) if int8 else 0
    c = _paged("", batch, heads, kv_heads, page, (batch + 4) * most // page, most // page, layers, int8, churn,
               rng.choice(["uniform", "lognormal"]), rng.randint(60, most // 4), rng.randint(64, most // 2))
  elif kind == "insert":
    seq = 128 * _spread(rng, 4, 32)
    c = dict(kind="insert", batch=rng.randint(2, 8), kv_heads=kv_heads, dim=rng.choice([128, 128, 64, 256]), seq=seq,
             layers=rng.randint(4, 32), int8=rng.random() < 0.7, scale32=rng.random() < 0.5,
             tokens=_spread(rng, 16, seq - 1), ring=rng.random() < 0.3)
    c["layers"] = max(2, min(c["layers"], int(6e9 // (c["batch"] * kv_heads * seq * c["dim"] * 4))))
  elif kind == "pages":
    page = rng.choice([32, 64, 128])
    tokens = _spread(rng, 16, 4096)
    c = dict(kind="pages", kv_heads=kv_heads, dim=rng.choice([128, 128, 64, 256]), page=page,
             pages=4 * (tokens // page + 1), layers=rng.randint(4, 24), tokens=tokens)
    c["layers"] = max(2, min(c["layers"], int(3e9 // (c["pages"] * page * kv_heads * c["dim"] * 4))))
  else:
    tokens = _spread(rng, 16, 3500)
    if rng.random() < 0.4:
      tokens = 1 << int(math.log2(tokens))  # prompts padded to a power of two, as the reference's engine pads them
    dim = rng.choice([128, 128, 64, 256])
    heads, kv_heads = (heads, kv_heads) if heads * dim <= 4096 else (4096 // dim, min(kv_heads, 4096 // dim // 2))
    c = dict(kind="prefill", batch=1 if tokens > 1000 else rng.randint(1, 3), heads=heads, kv_heads=kv_heads, dim=dim,
             tokens=tokens, int8=rng.random() < 0.4, mask32=rng.random() < 0.5)
  c.pop("name", None)
  return c


# ---- inputs ------------------------------------------------------------------------------------


def _lengths(case, seed, lo, hi):
  g = torch.Generator().manual_seed(seed)
  if case["lens"] == "uniform":
    return torch.randint(lo, min(hi, 2 * case["mid"]) + 1, (case["batch"],), generator=g, dtype=torch.int32)
  z = torch.randn(case["batch"], generator=g, dtype=torch.float64)
  return torch.clamp(torch.round(torch.exp(math.log(case["mid"]) + z)), lo, hi).to(torch.int32)


def _normal(g, *shape):
  return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32).to(BF16)


def _fill_normal(t, g):
  """Unit normal values (codes: what quantising them gives), one outer index at a time."""
  for row in t:
    if t.dtype == torch.int8:
      row.copy_(torch.empty(row.shape, dtype=BF16, device=DEV).normal_(0, 36, generator=g).clamp_(-127, 127))
    else:
      row.normal_(generator=g)


def _fill_scales(t, g):
  t.uniform_(0.02, 0.036, generator=g)


def _tokens(case, g):
  """A layer's new query, key and value rows, for every layer."""
  b, d = case["batch"], case["dim"]
  return [(_normal(g, b, case["heads"], 1, d), _normal(g, b, case["kv_heads"], 1, d), _normal(g, b, case["kv_heads"], 1, d))
          for _ in range(case["layers"])]


def _rotary(lengths, dim):
  freqs = 1.0 / (10000.0 ** (torch.arange(0, dim, 2, dtype=torch.float64) / dim))
  angle = lengths.to(torch.float64)[:, None] * freqs
  return torch.polar(torch.ones_like(angle), angle).to(torch.complex64).reshape(-1, 1, dim // 2).to(DEV)


def _prepare_step(case, seed):
  b, hkv, s, d, nl = case["batch"], case["kv_heads"], case["seq"], case["dim"], case["layers"]
  g = torch.Generator(device=DEV).manual_seed(seed)
  lengths = _lengths(case, seed, 16, s - 1)
  env = JetEngineEnvironment(JetEngineEnvironmentData(batch_size=b, num_layers=nl, cache_sequence_length=s,
                                                      ring_buffer=case["ring"]))
  scale_dtype = torch.float32 if case["scale32"] else BF16
  shapes = [(b, hkv, s, d)] * nl if case["ring"] else [(nl, b, hkv, s, d)]
  caches = []
  for shape in shapes:
    if case["int8"]:
      c = cm.Int8KVCacheGenerate.empty(shape, DEV, env, scale_dtype=scale_dtype)
      _fill_scales(c.k_scaler, g)
      _fill_scales(c.v_scaler, g)
    else:
      c = cm.KVCacheGenerate.empty(shape, DEV, env)
    _fill_normal(c.cache_k, g)
    _fill_normal(c.cache_v, g)
    caches.append(c)
  kernel = attn_layers.Int8KVAttentionKernel if case["int8"] else attn_layers.AttentionKernel
  st = dict(case=case, caches=caches, kernels=[kernel(env, l) for l in range(nl)], tokens=_tokens(case, g))
  if case["ring"]:
    # every slot's live positions end at the buffer's current position
    now = seed % s
    age = (now - torch.arange(s)) % s
    st["mask"] = torch.where((age[None] >= 1) & (age[None] <= lengths[:, None]), 0.0, float("-inf")).to(DEV)
    st["now"] = now
    st["input_pos"] = lengths.to(DEV)
    position = torch.tensor([now], dtype=torch.int32, device=DEV)
    for c in caches:
      c.input_pos = position
  else:
    st["positions"] = lengths.to(DEV)
    caches[0].input_pos = st["positions"]
    st["rope"] = dict(freqs_cis=_rotary(lengths, d)) if case["rope"] else {}
  return st


def _run_step(st):
  case = st["case"]
  if case["ring"]:
    mask = decode_state.update_mask(st["mask"], st["input_pos"], ring_buffer=True, current_position=st["now"])
    mask = mask.reshape(case["batch"], 1, 1, case["seq"])
    outs = [k(xq, xk, xv, mask, c) for k, c, (xq, xk, xv) in zip(st["kernels"], st["caches"], st["tokens"])]
  else:
    cache = st["caches"][0]
    plan, _ = ak.precompute_ragged_block_indices(st["positions"], case["batch"], case["heads"], case["kv_heads"], case["seq"])
    outs = [k(xq, xk, xv, None, cache, start=None, end=plan.lengths, ragged_batch_index=plan, **st["rope"])
            for k, (xq, xk, xv) in zip(st["kernels"], st["tokens"])]
    cache.finalize()
  state = [t for c in st["caches"] for t in (c.cache_k, c.cache_v) + ((c.k_scaler, c.v_scaler) if case["int8"] else ())]
  return dict(outs=outs, state=state)


def _prepare_paged(case, seed):
  b, hkv, ps, d, nl, total = (case[k] for k in ("batch", "kv_heads", "page", "dim", "layers", "pages"))
  g = torch.Generator(device=DEV).manual_seed(seed)
  cg = torch.Generator().manual_seed(seed + 1)
  lengths = _lengths(case, seed, 16, ps * case["max_pages"] - 2)
  lengths += (lengths % ps == 0).to(torch.int32)  # not on a page boundary (see the head of the file)
  st = dict(case=case)
  if case["churn"]:
    slots = torch.randperm(b, generator=cg)[:case["churn"]].to(torch.int32)
    new = torch.randint(16, case["prompt"] + 1, (case["churn"],), generator=cg, dtype=torch.int32)
    lengths[slots.long()] = new
    st["slots"], st["new_lens"] = slots.to(DEV), new.to(DEV)
    st["requests"] = list(zip(slots.tolist(), new.tolist()))
  env = JetEngineEnvironment(JetEngineEnvironmentData(
      batch_size=b, num_layers=nl, paged_attention_total_num_pages=total, paged_attention_page_size=ps))
  order = torch.randperm(total, generator=cg).to(torch.int32).numpy()
  pam = DevicePageAttentionManager(b, total, ps, case["max_pages"], device=DEV, free_list_order=order)
  pam.reserve_pages_insert_many(torch.arange(b, dtype=torch.int32), lengths)
  pool = (nl, hkv, total, ps, d)
  if case["int8"]:
    st["pools"] = [torch.empty(pool, dtype=torch.int8, device=DEV) for _ in range(2)]
    st["pools"] += [torch.empty((nl, 1, total, ps), device=DEV) for _ in range(2)]
    for t in st["pools"][2:]:
      _fill_scales(t, g)
    caches = [cm.Int8PageKVCacheGenerate(*(t[l] for t in st["pools"]), pam, None, env=env) for l in range(nl)]
    st["kernels"] = [attn_layers.Int8KVAttentionKernel(env, l) for l in range(nl)]
  else:
    st["pools"] = [torch.empty(pool, dtype=BF16, device=DEV) for _ in range(2)]
    caches = [cm.PageKVCacheGenerate(*(t[l] for t in st["pools"]), pam, None, env=env) for l in range(nl)]
    st["kernels"] = [attn_layers.AttentionKernel(env, l) for l in range(nl)]
  for t in st["pools"][:2]:
    _fill_normal(t, g)
  if case["churn"]:
    st["prompts"] = [(_normal(g, nl, hkv, n, d), _normal(g, nl, hkv, n, d)) for _, n in st["requests"]]
  st.update(pam=pam, caches=caches, lens=lengths.to(DEV), tokens=_tokens(case, g))
  return st


def _run_paged(st):
  case, pam = st["case"], st["pam"]
  if case["churn"]:
    pam.free_pages_resource_many(st["slots"])
    pam.reserve_pages_insert_many(st["slots"], st["new_lens"])
    ps = case["page"]
    prompt_insert.insert_prompts_pages_int8_stacked(
        st["prompts"], *st["pools"], [pam.page_indices[slot, : (n + ps - 1) // ps] for slot, n in st["requests"]])
  indices = pam.decode_step(st["lens"])
  outs = []
  for k, c, (xq, xk, xv) in zip(st["kernels"], st["caches"], st["tokens"]):
    c.page_token_indices = indices
    outs.append(k(xq, xk, xv, None, c))
  return dict(outs=outs, pools=st["pools"], table=pam.page_indices, lengths=pam.lengths)


def _prepare_insert(case, seed):
  b, hkv, s, d, nl = case["batch"], case["kv_heads"], case["seq"], case["dim"], case["layers"]
  g = torch.Generator(device=DEV).manual_seed(seed)
  env = JetEngineEnvironment(JetEngineEnvironmentData(batch_size=b, num_layers=nl, cache_sequence_length=s,
                                                      ring_buffer=case["ring"]))
  prompt = [(_normal(g, 1, hkv, case["tokens"], d), _normal(g, 1, hkv, case["tokens"], d)) for _ in range(nl)]
  shape = (nl, b, hkv, s, d)
  dtype = torch.int8 if case["int8"] else BF16
  k, v = (torch.zeros(shape, dtype=dtype, device=DEV) for _ in range(2))
  scales = None
  if case["int8"]:
    scales = [tuple(torch.ones((nl, b, 1, s, 1), dtype=torch.float32 if case["scale32"] else BF16, device=DEV) for _ in range(2))]
  mask = torch.full((b, s), float("-inf"), device=DEV)
  rows = [torch.zeros(b, dtype=torch.int32, device=DEV) for _ in range(3)]
  return dict(case=case, env=env, prompt=prompt, caches=[(k, v)], scales=scales, mask=mask, rows=rows, slot=seed % b,
              now=(seed * 7919) % s)


def _run_insert(st):
  case = st["case"]
  start, input_pos, lens = st["rows"]
  first = prompt_insert.insert(st["env"], st["prompt"], case["tokens"], st["caches"], st["scales"], st["slot"],
                               current_position=st["now"], mask=st["mask"], start=start, input_pos=input_pos, lens=lens)
  return dict(first=first, caches=st["caches"], scales=st["scales"], mask=st["mask"], rows=st["rows"])


def _prepare_pages(case, seed):
  hkv, ps, d, nl, total = case["kv_heads"], case["page"], case["dim"], case["layers"], case["pages"]
  g = torch.Generator(device=DEV).manual_seed(seed)
  order = torch.randperm(total, generator=torch.Generator().manual_seed(seed)).to(torch.int32).numpy()
  pam = PageAttentionManager(4, total, ps, total, free_list_order=order)
  prompt = [(_normal(g, 1, hkv, case["tokens"], d), _normal(g, 1, hkv, case["tokens"], d)) for _ in range(nl)]
  caches = [tuple(torch.zeros((hkv, total, ps, d), dtype=BF16, device=DEV) for _ in range(2)) for _ in range(nl)]
  return dict(case=case, pam=pam, prompt=prompt, caches=caches)


def _run_pages(st):
  pam = st["pam"]
  _, pages = pam.reserve_pages_insert(1, st["case"]["tokens"])
  pam.insert_prefill_cache(st["prompt"], st["caches"], pages)
  pam.free_pages_resource(1)  # the request is over: its pages go to the end of the free list
  return st["caches"]


def _prepare_prefill(case, seed):
  b, t, d = case["batch"], case["tokens"], case["dim"]
  g = torch.Generator(device=DEV).manual_seed(seed)
  env = JetEngineEnvironment(JetEngineEnvironmentData(batch_size=b, num_layers=1))
  mask = torch.full((1, 1, t, t), float("-inf"), dtype=torch.float32 if case["mask32"] else BF16, device=DEV).triu(1)
  kernel = attn_layers.Int8KVAttentionKernel if case["int8"] else attn_layers.AttentionKernel
  xq, xk, xv = _normal(g, b, case["heads"], t, d), _normal(g, b, case["kv_heads"], t, d), _normal(g, b, case["kv_heads"], t, d)
  return dict(case=case, kernel=kernel(env, 0), mask=mask, rows=(xq, xk, xv))


def _run_prefill(st):
  cache = cm.KVCachePrefill(kv_quantize=st["case"]["int8"])
  out = st["kernel"](*st["rows"], st["mask"], cache)
  return dict(out=out, cache=cache.state())


def prepare(case, seed):
  return {"step": _prepare_step, "paged": _prepare_paged, "insert": _prepare_insert, "pages": _prepare_pages,
          "prefill": _prepare_prefill}[case["kind"]](case, seed)


def run(state):
  return {"step": _run_step, "paged": _run_paged, "insert": _run_insert, "pages": _run_pages,
          "prefill": _run_prefill}[state["case"]["kind"]](state)


# ---- what a pass cannot do without, and how exact it is ------------------------------------------


def _mean_length(case, lo, hi):
  lengths = [_lengths(case, seed, lo, hi) for seed in range(8)]
  return float(torch.stack(lengths).to(torch.float64).mean())


def work(case):
  kind, hkv, d = case["kind"], case["kv_heads"], case["dim"]
  if kind in ("step", "paged"):
    b, hq, nl = case["batch"], case["heads"], case["layers"]
    paged = kind == "paged"
    top = case["page"] * case["max_pages"] - 2 if paged else case["seq"] - 1
    live = _mean_length(case, 16, top) + 1  # attended positions of a slot
    if paged and case["churn"]:
      live += (case["prompt"] / 2 - live) * case["churn"] / b
    e = 1 if case["int8"] else 2
    es = 0 if not case["int8"] else 4 if paged or case["scale32"] else 2
    keys = b * live * (2 * hkv * d * e + 2 * es)
    token = b * (2 * hkv * d * (2 + e) + 2 * es)          # the step's rows in, the cache's lines out
    rows = b * hq * d * 2 * 2                             # query in, output out
    mask = b * case["seq"] * 4 if not paged and case["ring"] else 0
    total = nl * (keys + token + rows + mask)
    if paged and case["churn"]:
      total += nl * case["churn"] * case["prompt"] / 2 * 2 * (hkv * d * 3 + es)
    return {"bytes": total, "flops": nl * b * live * hq * d * 4}
  t = case["tokens"]
  if kind == "prefill":
    b, hq = case["batch"], case["heads"]
    return {"bytes": b * t * d * 2 * (2 * hq + 2 * hkv) + t * t * (4 if case["mask32"] else 2),
            "flops": 4.0 * b * hq * d * t * (t + 1) / 2}
  out = 1 if kind == "insert" and case["int8"] else 2
  scales = 2 * t * (4 if case["scale32"] else 2) if kind == "insert" and case["int8"] else 0
  return {"bytes": case["layers"] * (2 * hkv * d * t * (2 + out) + scales), "flops": 0}


def tolerance(case):
  # Cache lines, codes, scales and page tables are the same bits whichever way they are written.
  # Attention outputs are bf16: against softmax attention in 64 bits over the same rows the path
  # differs by 1.6e-3 (the output's own rounding) to 2.1e-3 (bf16 softmax weights as well, bf16
  # caches), by at most 0.009 of the larger of the value and the root mean square; four times that.
  if case["kind"] in ("insert", "pages"):
    return "exact"
  return {"rel": 8e-3, "max": 0.036}
