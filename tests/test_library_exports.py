"""The C-ABI library loads without a GPU and exports every function the public
header declares; no compute entry point is called here."""

import ctypes
import os
import re

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "jpt_mi355.h")


def declared_functions():
  text = open(HEADER).read()
  text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
  return sorted(set(re.findall(r"\b(jpt_[a-z0-9_]+)\s*\(", text)))


def test_every_declared_symbol_is_exported():
  from jetstream_pt_amd import _ffi
  names = declared_functions()
  assert len(names) >= 20
  lib = ctypes.CDLL(_ffi.LIB_PATH)
  missing = [n for n in names if not hasattr(lib, n)]
  assert not missing, f"declared in the header but not exported: {missing}"
  assert sorted(_ffi.EXPORTS) == names


def test_version_and_error_channel():
  from jetstream_pt_amd import _ffi
  assert _ffi.lib.jpt_version() == 1
  # argument validation happens before any device work
  assert _ffi.lib.jpt_attn_ragged(None, None) == _ffi.E_BADARG
  assert b"NULL" in _ffi.lib.jpt_last_error()
  with pytest.raises(ValueError):
    _ffi.check(_ffi.lib.jpt_kv_append_quant_i8(None, None))


def test_ops_refuse_cpu_tensors():
  import torch
  from jetstream_pt_amd import attention_kernel as ak
  q = torch.zeros((1, 2, 1, 8))
  with pytest.raises(RuntimeError, match="ROCm device only"):
    ak.dense_attention(q, q, q)


@pytest.mark.parametrize("change,mode,want", [
    ({}, 0, "STREAMING"), ({}, 1, "STREAMING"), (dict(seq=96), 1, "STREAMING"), (dict(seq=90), 1, "SPLIT"), (dict(dim=64), 0, "SPLIT"),
    (dict(dim=256), 1, "SPLIT"), (dict(dim=80), 1, "GENERIC"), (dict(mask=64, mask_stride_h=4), 1, "SPLIT"),
    (dict(mask=64, mask_dtype=1), 1, "STREAMING"), (dict(mask=64, mask_dtype=0), 1, "SPLIT"), (dict(q_rows=5), 1, "PREFILL"),
    (dict(q_rows=4), 1, "STREAMING"), (dict(q_rows=500, kv_dtype=2, k_scale=64, v_scale=64, scale_heads=1), 1, "GENERIC"),
    (dict(kv_dtype=2), 0, "GENERIC"), (dict(kv_dtype=2, k_scale=64, v_scale=64, scale_heads=1), 0, "STREAMING"), (dict(q=8), 0, "GENERIC"),
    (dict(seq=0, page_size=32), 2, "STREAMING"), (dict(seq=0, page_size=16), 2, "GENERIC"), (dict(seq=0, page_size=32, dim=64), 2, "GENERIC"),
    (dict(force_generic=1), 0, "GENERIC"), (dict(batch=5000), 1, "SPLIT"), (dict(kv_heads=0), 0, "GENERIC"),
])
def test_which_kernel_takes_a_call(change, mode, want):
  """Addresses are looked at, not followed."""
  from jetstream_pt_amd import _ffi
  a = dict(q=64, k=64, v=64, out=64, batch=2, q_heads=8, kv_heads=2, q_rows=1, dim=128, seq=256, q_dtype=_ffi.BF16, kv_dtype=_ffi.BF16)
  assert _ffi.lib.jpt_attn_kernel(_ffi.AttnArgs(**dict(a, **change)), mode) == getattr(_ffi, "ATTN_" + want)


def test_page_ids_on_the_host_are_for_copies():
  """A quantising call is left to the entry that takes its ids on the device: 1, and nothing done."""
  from jetstream_pt_amd import _ffi
  address = 4096  # looked at, not followed
  layer = (_ffi.InsertLayer * 1)(_ffi.InsertLayer(*([address] * 6)))
  ids = (ctypes.c_int32 * 4)(0, 1, 2, 3)
  fn = _ffi.lib.jpt_prefill_insert_layers_host_pages
  fn.restype, fn.argtypes = ctypes.c_int32, [ctypes.c_void_p] * 3 + [ctypes.c_int32, ctypes.c_void_p]
  for scale_dtype in (_ffi.BF16, _ffi.F32):
    a = _ffi.PrefillInsertArgs(tokens=100, heads=8, dim=128, n_pages=4, total_pages=8, page_size=32, in_dtype=_ffi.BF16, dst_dtype=_ffi.I8,
                               scale_dtype=scale_dtype, scale_heads=1)
    assert fn(ctypes.byref(a), ids, layer, 1, None) == 1
