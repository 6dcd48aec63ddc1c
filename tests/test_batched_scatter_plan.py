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


@pytest.mark.parametrize("value_bytes", [4, 8])
def test_small_networks_take_little_scratch_memory(value_bytes):
  # 20 entries of a 1,000 x 1,000 network of 50,000 nonzeros: every nonzero of an entry may lie in one of the four windows that
  # an entry spans, which makes five times the 1e6 pairs there are at most
  entries, pairs = _plan(1000, 1000, 50_000, 20, value_bytes)
  assert entries == 20 and 1_000_000 * 4 <= pairs <= 1_000_000 * 6
  for n_row, n_col in SHAPES:
    for per_row in (1, 3, 50):
      nnz = n_row * per_row
      for batch in (2, 8, 20, 500):
        entries, pairs = _plan(n_row, n_col, nnz, batch, value_bytes)
        # never more than every nonzero of every entry in each of at most 128 windows, twice, but for the least the sort
        # works with (1,024 pairs in each of the eight parts of a window's run)
        assert pairs <= max(2 * 128 * entries * nnz, 128 * 8 * 1024), (n_row, n_col, nnz, entries, pairs)


def test_no_matrix():
  assert _plan(0, 5, 0, 3, 4) == _plan(5, 0, 0, 3, 4) == _plan(5, 5, 9, 0, 4) == (0, 0)
