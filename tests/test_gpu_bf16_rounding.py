"""GPU parity of the rounding to bfloat16: every float32, NaNs among them, against
the format's definition; and of the quantisers', one operation at a time: every
finite bfloat16 as a token's largest number, so that scale, quotient and
reciprocal take ties, subnormal numbers and overflow, bit for bit against the
same steps in PyTorch on the CPU (whole numbers and stored bits: no tolerance)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def by_steps(x, rounding):
  amax = x.abs().amax(-1, keepdim=True)
  if rounding == "rne":
    amax = amax.clamp_min(torch.tensor(1e-5, dtype=torch.bfloat16))
    s = amax / 127
    return (x * (1 / s)).float().round().clamp(-128, 127).to(torch.int8), s
  s = amax / 127
  return (x / s).float().nan_to_num(0.).trunc().to(torch.int8), s


@pytest.mark.parametrize("dim", [8, 12])  # the rows kernel; the general one
def test_every_largest_number(dim):
  from jetstream_pt_amd import insert as gins
  tokens = 0x7f80
  top = torch.arange(tokens, dtype=torch.int16).view(torch.bfloat16)
  g = torch.Generator().manual_seed(dim)
  x = (top[:, None].float() * (2 * torch.rand((tokens, dim), generator=g) - 1)).to(torch.bfloat16)
  x[:, 3] = top
  want, scale = by_steps(x, "rne")
  k, v = (torch.zeros((1, 1, tokens, dim), dtype=torch.int8, device=DEV) for _ in range(2))
  ks, vs = (torch.zeros((1, 1, tokens, 1), dtype=torch.bfloat16, device=DEV) for _ in range(2))
  p = x.reshape(1, 1, tokens, dim).to(DEV)
  gins.insert_prefix_caches([(p, -p)], [(k, v)], [(ks, vs)], 0, 0)
  torch.cuda.synchronize()
  for s in (ks, vs):
    assert torch.equal(s.cpu().reshape(-1).view(torch.int16), scale.reshape(-1).view(torch.int16))
  assert torch.equal(k.cpu().reshape(tokens, dim), want)
  assert torch.equal(v.cpu().reshape(tokens, dim), by_steps(-x, "rne")[0])


def test_every_float32():
  """Through the rotation, whose first output is 1 * c - 0 * 0 rounded: to nearest, ties to even, NaN kept and made quiet."""
  from jetstream_pt_amd import _ffi
  rows, half = 1 << 15, 1 << 11
  n = rows * half
  x = torch.tensor([1.0, 0.0], device=DEV).repeat(n).to(torch.bfloat16)
  out, freqs = torch.empty_like(x), torch.zeros((n, 2), device=DEV)
  for first in range(-1 << 31, 1 << 31, n):
    bits = torch.arange(first, first + n, device=DEV)  # int64
    freqs[:, 0] = bits.to(torch.int32).view(torch.float32)
    _ffi.check(_ffi.lib.jpt_rope(_ffi.ptr(out), _ffi.ptr(x), _ffi.ptr(freqs), rows, 1, 2 * half, _ffi.BF16, _ffi.stream()))
    nan = (bits & 0x7fffffff) > 0x7f800000
    want = torch.where(nan, (bits >> 16) | 0x40, (bits + 0x7fff + ((bits >> 16) & 1)) >> 16).to(torch.int16)
    assert torch.equal(out.view(torch.int16)[::2], want), hex(first & 0xffffffff)
