"""How a batch of the transposed event product is divided into groups (bpl_batched_scatter_plan; no device needed)."""
import ctypes

import pytest

from brainpylib_amd import _lib


def _plan(n_row, n_col, nnz, batch, value_bytes):
  entries, pairs = ctypes.c_uint32(), ctypes.c_uint64()
  f = _lib.lib().bpl_batched_scatter_plan
  f.restype, f.argtypes = None, [ctypes.c_uint32] * 5 + [ctypes.c_void_p] * 2
  f(n_row, n_col, nnz, batch, value_bytes, ctypes.byref(entries), ctypes.byref(pairs))
  return entries.value, pairs.value


SHAPES = [(1000, 1000), (1000, 20_000), (20_000, 20_000), (50_000, 50_000), (300_000, 5000), (100_000, 100_000),
          (1_000_000, 300_000), (7, 3_000_000)]


@pytest.mark.parametrize("value_bytes", [4, 8])
@pytest.mark.parametrize("per_row", [1, 30, 400, 2000])
def test_every_pair_of_a_large_group_finds_room(value_bytes, per_row):
  for n_row, n_col in SHAPES:
    nnz = n_row * per_row
    for batch in (1, 2, 7, 8, 9, 16, 20, 33, 64, 500):
      entries, pairs = _plan(n_row, n_col, nnz, batch, value_bytes)
      what = (n_row, n_col, nnz, batch, entries, pairs)
      assert 1 <= entries <= batch, what
      # (more than 8 entries: with every event set all pairs fit, and half as many again)
      assert entries <= 8 or 2 * pairs >= 3 * entries * nnz, what
      assert pairs * (2 * value_bytes) <= 2 ** 31, what
      # never fewer entries to a group than eight, but for outputs of 2^24 columns and more
      if entries * n_col < 2 ** 23:
        assert entries >= min(batch, 8) or -(-batch // entries) == -(-batch // 8), what


def test_no_matrix():
  assert _plan(0, 5, 0, 3, 4) == _plan(5, 0, 0, 3, 4) == _plan(5, 5, 9, 0, 4) == (0, 0)
