"""The register-resident quantiser (one run of four elements a thread) at the
edges of its shapes, bit for bit against the oracle's quantisers."""
import pytest
import torch

from oracle import quant as oquant

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# one run; a part of a wave; a wave; a wave and a part; an odd number of waves; all of a workgroup; one run too many (the
# generic kernel); rows no power of two of runs (generic with a scale a head)
@pytest.mark.parametrize("heads,dim", [(1, 4), (1, 128), (2, 128), (5, 64), (3, 256), (4, 128), (16, 256), (32, 128), (33, 128),
                                       (1, 4096), (1025, 4), (6, 12)])
@pytest.mark.parametrize("rounding,ofn", [("trunc", oquant.quantize_decode), ("rne", oquant.quantize_insert)])
@pytest.mark.parametrize("scale_dtype", [None, torch.float32])
def test_quantiser_shapes(heads, dim, rounding, ofn, scale_dtype):
  from jetstream_pt_amd.quantize import quantize_kv
  g = torch.Generator().manual_seed(heads * dim)
  x = (torch.randn((37, heads, 1, dim), generator=g) * torch.logspace(-3, 2, 37).reshape(-1, 1, 1, 1)).to(torch.bfloat16)
  x[5] = 0
  y = torch.randn((37, heads, 1, dim), generator=g).to(torch.bfloat16)
  for hs in {1, heads if heads <= 64 else 1}:
    kq, vq, ks, vs = quantize_kv(x.to(DEV), y.to(DEV), rounding=rounding, scale_heads=hs, scale_dtype=scale_dtype)
    for got_c, got_s, src in ((kq, ks, x), (vq, vs, y)):
      want_c, want_s = ofn(src, hs, scale_dtype)
      assert torch.equal(got_s.cpu(), want_s) and torch.equal(got_c.cpu(), want_c)
