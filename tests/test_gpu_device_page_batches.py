"""Requests of one launch are served side by side: the page table, lengths, free
list and status bits must be what one launch a request leaves (those are pinned
to the oracle), whatever the requests name."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def i32(x):
  return torch.tensor(x, dtype=torch.int32, device=DEV)


def same(a, b):
  assert torch.equal(a.page_indices, b.page_indices)
  assert torch.equal(a.lengths, b.lengths)
  assert a.unused_page_ids().tolist() == b.unused_page_ids().tolist()
  assert a.status() == b.status()


# one request; a share of more than 16 threads each; 16 each; more requests than threads; rows of many pages
@pytest.mark.parametrize("batch,total,mp,n_req", [(8, 64, 6, 1), (8, 64, 6, 3), (40, 300, 9, 16), (70, 500, 40, 17), (400, 900, 5, 300),
                                                  (4, 900, 300, 2)])
@pytest.mark.parametrize("kind", ["distinct", "twice", "refused"])
def test_a_batch_equals_its_requests_one_by_one(batch, total, mp, n_req, kind):
  from jetstream_pt_amd.page_attention_manager import DevicePageAttentionManager
  rng = np.random.default_rng(n_req)
  ps = 4
  order = rng.permutation(total).astype(np.int32)
  many, one = (DevicePageAttentionManager(batch, total, ps, mp, device=DEV, free_list_order=order) for _ in range(2))
  for _ in range(6):
    slots = rng.choice(batch, size=n_req, replace=kind == "twice")
    # on average a little more than the free list holds where requests may be refused
    most = mp * ps if kind == "refused" else max(min(mp * ps, ps * total // (2 * n_req)), 1)
    lens = rng.integers(0, most + 1, size=n_req)
    if kind == "refused" and n_req > 2:
      slots[1], lens[2] = batch + 3, (mp + 1) * ps  # no such slot, too many pages
    many.reserve_pages_insert_many(i32(slots), i32(lens))
    for s, n in zip(slots, lens):
      one.reserve_pages_insert_many(i32([s]), i32([n]))
    same(many, one)
    slots = rng.choice(batch, size=n_req, replace=kind == "twice")
    if kind == "refused" and n_req > 2:
      slots[0] = -1
    many.free_pages_resource_many(i32(slots))
    for s in slots:
      one.free_pages_resource_many(i32([s]))
    same(many, one)


@pytest.mark.parametrize("n", [41, 2 ** 31 - 4, 2 ** 31 - 1])
def test_lengths_that_no_slot_holds_are_refused(n):
  """... up to the largest: the count of their pages does not wrap round."""
  from jetstream_pt_amd import _ffi
  from jetstream_pt_amd.page_attention_manager import DevicePageAttentionManager
  pam = DevicePageAttentionManager(4, 64, 4, 10, device=DEV)
  before = pam.page_indices.clone(), pam.lengths.clone(), pam.unused_page_ids().tolist()
  pam.reserve_pages_insert_many(i32([1]), i32([n]))
  assert torch.equal(pam.page_indices, before[0]) and torch.equal(pam.lengths, before[1]) and pam.unused_page_ids().tolist() == before[2]
  assert pam.status() == _ffi.DPAM_OVERFLOW
