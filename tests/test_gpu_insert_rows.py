"""GPU parity of the insert's wide kernels at the edges of their shapes: rows of
bf16 quantised by threads that keep a few heads of one token, and rows copied as
16-byte pieces, into slots (with ring wrap) and pages, bit for bit against the
CPU oracle."""
import pytest
import torch

from oracle import quant as oquant
from test_gpu_insert import DEV, run_both

pytestmark = pytest.mark.gpu


# one head; heads that do not fill a pass; three passes; a row of one piece, of 64 and, of one head, of 128; the most heads a token may have,
# one more than that, and rows that are no power of two (both: the general kernel)
@pytest.mark.parametrize("heads,dim", [(1, 128), (3, 64), (5, 256), (24, 128), (40, 128), (64, 128), (65, 128), (16, 512),
                                       (7, 8), (60, 8), (4, 96), (16, 64), (4, 256), (1, 1024), (3, 1024), (8, 1024), (9, 1024), (1, 2048)])
@pytest.mark.parametrize("ring,position,prompt,scale_dtype", [(False, 0, 17, torch.bfloat16), (True, 5, 40, torch.float32)])
def test_quantised_rows(heads, dim, ring, position, prompt, scale_dtype):
  run_both(ring, True, (2, heads, 64, dim, 2), prompt=prompt, seq_len=prompt - 3, slot=1, current_position=position,
           scale_dtype=scale_dtype)


# rows of one 16-byte piece, of an odd number, of half a piece more (the ordinary kernel); several workgroups a head
@pytest.mark.parametrize("heads,dim,dtype", [(2, 8, torch.bfloat16), (3, 24, torch.bfloat16), (3, 12, torch.bfloat16),
                                             (8, 128, torch.bfloat16), (1, 256, torch.bfloat16)])
@pytest.mark.parametrize("ring,position,prompt", [(False, 0, 24), (True, 7, 40), (True, 199, 200)])
def test_copied_rows(heads, dim, dtype, ring, position, prompt):
  run_both(ring, False, (2, heads, 256, dim, 2), prompt=prompt, seq_len=prompt - 1, slot=1, current_position=position,
           prefix_dtype=dtype)


@pytest.mark.parametrize("heads,dim,ps,tokens", [(1, 8, 16, 1), (3, 24, 10, 37), (8, 128, 64, 65), (2, 64, 128, 128), (4, 12, 16, 30)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shift", [0, 4])
def test_copied_pages(heads, dim, ps, tokens, dtype, shift):
  """shift: the prompt lies that many elements into its memory, so that bf16 rows
  are not aligned for 16-byte loads."""
  from jetstream_pt_amd import insert as gins
  layers, n_pages = 2, -(-tokens // ps)
  total = n_pages + 3
  g = torch.Generator().manual_seed(heads + tokens)
  ids = torch.randperm(total, generator=g)[:n_pages].to(torch.int32)
  pools = [tuple(torch.randn((heads, total, ps, dim), generator=g).to(dtype) for _ in range(2)) for _ in range(layers)]
  prefix = [tuple(torch.randn((1, heads, tokens, dim), generator=g).to(dtype) for _ in range(2)) for _ in range(layers)]

  def shifted(t):
    flat = torch.zeros(t.numel() + shift, dtype=dtype, device=DEV)
    flat[shift:] = t.to(DEV).reshape(-1)
    return flat[shift:].reshape(t.shape)
  dpools = [tuple(t.to(DEV) for t in pair) for pair in pools]
  assert gins.insert_prefix_pages_copy([tuple(shifted(t) for t in pair) for pair in prefix], dpools, ids.to(DEV))
  torch.cuda.synchronize()
  for layer in range(layers):
    for which in (0, 1):
      want = pools[layer][which].clone()
      padded = torch.zeros((heads, n_pages * ps, dim), dtype=dtype)
      padded[:, :tokens] = prefix[layer][which][0]
      want[:, ids.long()] = padded.reshape(heads, n_pages, ps, dim)
      assert torch.equal(dpools[layer][which].cpu(), want)


@pytest.mark.parametrize("heads,dim,scale_heads", [(3, 64, 3), (24, 128, 1), (64, 128, 64), (2, 512, 2), (4, 96, 1), (1, 1024, 1), (4, 1024, 1), (2, 1024, 2)])
def test_quantised_pages(heads, dim, scale_heads):
  """One scale a token and one a (token, head), several prompts in one launch
  and one by one: the same pool, and the codes the oracle's quantiser gives.
  (4, 96): the library's prompt-by-prompt route."""
  from jetstream_pt_amd import insert as gins
  layers, total, ps = 2, 12, 16
  g = torch.Generator().manual_seed(heads)
  lens, ids, at = [1, 33, 50], [], 0
  perm = torch.randperm(total, generator=g).to(torch.int32)
  buf = [torch.randn((layers, heads, 60, dim), generator=g).to(torch.bfloat16) for _ in range(2)]
  pools = [torch.randint(-127, 128, (layers, heads, total, ps, dim), generator=g, dtype=torch.int8) for _ in range(2)]
  scales = [torch.rand((layers, scale_heads, total, ps), generator=g) for _ in range(2)]
  many, one = [t.to(DEV) for t in pools + scales], [t.to(DEV) for t in pools + scales]
  dbuf = [t.to(DEV) for t in buf]
  for n in lens:
    ids.append(perm[at:at + -(-n // ps)])
    at += -(-n // ps)
  gins.insert_prompts_pages_int8_stacked([(dbuf[0][:, :, :n], dbuf[1][:, :, :n]) for n in lens], *many, [i.to(DEV) for i in ids])
  for n, i in zip(lens, ids):
    gins.insert_prefix_pages_int8_stacked(dbuf[0][:, :, :n], dbuf[1][:, :, :n], *one, i.to(DEV))
  torch.cuda.synchronize()
  for a, b in zip(many, one):
    assert torch.equal(a, b)
  for which in (0, 1):
    want, want_s = pools[which].clone(), scales[which].clone()
    for n, i in zip(lens, ids):
      x = buf[which][:, :, :n].float()
      if scale_heads == 1:
        codes, s = oquant.quantize_insert(x)
      else:  # a head at a time: the scale of a token with that head alone
        per = [oquant.quantize_insert(x[:, h:h + 1]) for h in range(heads)]
        codes, s = torch.cat([c for c, _ in per], 1), torch.cat([c for _, c in per], 1)
      padded = torch.zeros((layers, heads, len(i) * ps, dim), dtype=torch.int8)
      padded[:, :, :n] = codes
      want[:, :, i.long()] = padded.reshape(layers, heads, len(i), ps, dim)
      flat = want_s[:, :, i.long()].reshape(layers, scale_heads, -1)
      flat[:, :, :n] = s.reshape(layers, scale_heads, n)
      want_s[:, :, i.long()] = flat.reshape(layers, scale_heads, len(i), ps)
    assert torch.equal(many[which].cpu(), want)
    assert torch.equal(many[2 + which].cpu(), want_s)
