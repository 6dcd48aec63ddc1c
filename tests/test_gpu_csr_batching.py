"""GPU parity of event_csr_matvec_batching against the CPU oracle, through the C ABI."""
import numpy as np
import pytest
import torch

import brainpylib_amd as bpl
import benchdata as synth
from util import assert_close, assert_close_reordered, batched_csr

pytestmark = pytest.mark.gpu


def _check(oracle_mod, values, indices, indptr, events, batch, shape, transpose, what):
  want = oracle_mod.event_csr_matvec_batching(values, indices, indptr, events, batch_size=batch, shape=shape,
                                              transpose=transpose)
  got = bpl.event_csr_matvec_batching(values, indices, indptr, events, batch_size=batch, shape=shape,
                                      transpose=transpose).cpu().numpy()
  assert got.shape == want.shape and got.dtype == want.dtype
  if transpose:
    mag = oracle_mod.event_csr_matvec_batching(np.abs(values), indices, indptr, events, batch_size=batch,
                                               shape=shape, transpose=True)
    assert_close_reordered(got, want, mag, values.dtype.type, what=what)
  else:
    assert_close(got, want, what=what)
  return got, want


@pytest.mark.parametrize("shape", [(100, 200), (200, 100), (10, 1000), (1000, 10), (3000, 2500)])
@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_batching_broadcast_combinations(cuda, oracle_mod, shape, transpose, dtype):
  rng = np.random.default_rng(11)
  n_in = shape[0] if transpose else shape[1]
  for dims, batch in (((1, 1, 1, 5), 5), ((1, 1, 1, 9), 9), ((1, 1, 1, 1), 1), ((1, 1, 1, 3), 20), ((1, 1, 1, 1), 4),
                      ((1, 3, 3, 1), 3), ((4, 1, 1, 4), 4), ((3, 3, 3, 3), 3), ((2, 1, 1, 3), 6)):
    vb, ib, pb, eb = dims
    print("case", shape, transpose, dtype.__name__, dims, batch, flush=True)
    data, indices, indptr = batched_csr(shape, 40 if shape[1] >= 100 else 5, max(vb, ib), seed=shape[0] + batch,
                                        dtype=dtype)
    events = rng.random((eb, n_in)) < 0.15
    _check(oracle_mod, data[:vb], indices[:ib], indptr[:pb], events, batch, shape, transpose, "heter bool")
    fev = (events * rng.uniform(0.5, 2.0, events.shape)).astype(dtype)
    _check(oracle_mod, data[:vb], indices[:ib], indptr[:pb], fev, batch, shape, transpose, "heter float")
    w = rng.standard_normal((vb, 1)).astype(dtype)
    # homogeneous weights are added once per synapse, as the reference adds them: its bits, whatever the order
    got, want = _check(oracle_mod, w, indices[:ib], indptr[:pb], events, batch, shape, transpose, "homo bool")
    assert np.array_equal(got, want)
    one = np.full((1, 1), 0.6, dtype=dtype)
    got, want = _check(oracle_mod, one, indices[:ib], indptr[:pb], events, batch, shape, transpose, "counts")
    assert np.array_equal(got, want)


def test_batching_short_and_long_rows_and_wide_matrices(cuda, oracle_mod):
  # mean row length below / above 32 selects 8 lanes / one wave per row; 200,000 columns do not
  # fit the LDS copy of the event masks (global probes)
  rng = np.random.default_rng(12)
  for n_row, n_col, mean in ((20000, 3000, 6), (2000, 3000, 300), (500, 200_000, 900), (30000, 200_000, 10)):
    counts = np.minimum(rng.poisson(mean, size=n_row), n_col)
    indices, indptr = synth.counted_csr(counts, n_col, seed=n_row)
    data = rng.standard_normal(indices.shape[0]).astype(np.float32)
    shape = (n_row, n_col)
    print("shape", shape, flush=True)
    events = rng.random((11, n_col)) < 0.05
    got, want = _check(oracle_mod, data[None], indices[None], indptr[None], events, 11, shape, False, "heter")
    one = np.full((1, 1), 0.7, dtype=np.float32)
    got, want = _check(oracle_mod, one, indices[None], indptr[None], events, 11, shape, False, "homo")
    assert np.array_equal(got, want), "homogeneous gather is bit-exact"


def test_batching_transposed_through_one_sorted_scatter(cuda, oracle_mod):
  # transpose=True with one matrix for all entries: the active rows of all entries go through one
  # coarse sort over batch * n_col virtual columns.  Many virtual rows (several row tiles per
  # producer), wide virtual outputs (sliced windows above 2^21), events broadcast (3 vectors for 6 entries).
  rng = np.random.default_rng(13)
  for n_row, n_col, mean, batch, eb, rate in ((20_000, 30_000, 30, 8, 8, 0.05), (300_000, 5000, 4, 6, 3, 0.6),
                                              (2000, 1_500_000, 200, 4, 4, 0.3)):
    counts = np.minimum(rng.poisson(mean, size=n_row), n_col)
    indices, indptr = synth.counted_csr(counts, n_col, seed=n_row)
    data = rng.standard_normal(indices.shape[0]).astype(np.float32)
    shape = (n_row, n_col)
    print("shape", shape, "batch", batch, flush=True)
    events = rng.random((eb, n_row)) < rate
    _check(oracle_mod, data[None], indices[None], indptr[None], events, batch, shape, True, "heter")
    one = np.full((1, 1), 0.6, dtype=np.float32)
    got, want = _check(oracle_mod, one, indices[None], indptr[None], events, batch, shape, True, "counts")
    assert np.array_equal(got, want)
    # twice in a row (the list's counter is back at zero), float events
    fev = (events * rng.uniform(0.5, 2.0, events.shape)).astype(np.float32)
    _check(oracle_mod, data[None], indices[None], indptr[None], fev, batch, shape, True, "heter float events")


def test_batching_equals_single_operator(cuda):
  # every row of the batched result is the single operator's result (exactly so for the
  # homogeneous weight, to rounding of one float64 sum otherwise)
  c = synth.config_event_csr_small()
  rng = np.random.default_rng(13)
  shape = c["shape"]
  events = rng.random((10, shape[1])) < 0.02
  got = bpl.event_csr_matvec_batching(np.full((1, 1), 0.6, np.float32), c["indices"][None], c["indptr"][None],
                                      events, batch_size=10, shape=shape)
  for bi in range(10):
    single = bpl.event_csr_matvec(np.float32(0.6), c["indices"], c["indptr"], events[bi], shape=shape)
    assert torch.equal(got[bi], single)


def test_batching_edge_cases(cuda, oracle_mod):
  indptr = np.array([[0, 0, 3, 3, 5]], dtype=np.int32)
  indices = np.array([[0, 2, 4, 1, 4]], dtype=np.int32)
  data = np.array([[1, 2, 3, 4, 5]], dtype=np.float32)
  shape = (4, 5)
  for tr in (False, True):
    n_in = shape[0] if tr else shape[1]
    for ev in (np.zeros((3, n_in), bool), np.ones((3, n_in), bool)):
      got, want = _check(oracle_mod, data, indices, indptr, ev, 3, shape, tr, "edge")
      assert np.array_equal(got, want)
  # empty batch, empty matrix
  out = bpl.event_csr_matvec_batching(data, indices, indptr, np.ones((1, 5), bool), batch_size=0, shape=shape)
  assert tuple(out.shape) == (0, 4)
  e = np.zeros((1, 0), dtype=np.int32)
  out = bpl.event_csr_matvec_batching(np.ones((1, 1), np.float32), e, np.zeros((1, 4), np.int32),
                                      np.ones((5, 7), bool), batch_size=5, shape=(3, 7)).cpu().numpy()
  assert out.shape == (5, 3) and not out.any()
  with pytest.raises(ValueError):
    bpl.event_csr_matvec_batching(data[0], indices, indptr, np.ones((1, 5), bool), batch_size=1, shape=shape)
  with pytest.raises(ValueError):
    bpl.event_csr_matvec_batching(data, indices, indptr, np.ones((1, 4), bool), batch_size=1, shape=shape)


def test_full_size_batching_rows_equal_single_operator(cuda):
  # 100,000 x 100,000, ~1e8 nnz, nine event vectors (two tiles of eight): every row of the batched
  # result against the single operator; the homogeneous weight bit for bit
  c = synth.config_event_csr_large()
  shape = c["shape"]
  dev = cuda
  data = torch.from_numpy(c["data"]).to(dev)
  indices = torch.from_numpy(c["indices"]).to(dev)
  indptr = torch.from_numpy(c["indptr"]).to(dev)
  rng = np.random.default_rng(17)
  events = torch.from_numpy(rng.random((9, shape[1])) < 0.05).to(dev)
  w = torch.full((1, 1), 0.6, dtype=torch.float32, device=dev)
  het = bpl.event_csr_matvec_batching(data[None], indices[None], indptr[None], events, batch_size=9, shape=shape)
  hom = bpl.event_csr_matvec_batching(w, indices[None], indptr[None], events, batch_size=9, shape=shape)
  for bi in range(9):
    single = bpl.event_csr_matvec(data, indices, indptr, events[bi], shape=shape)
    assert_close(het[bi].cpu().numpy(), single.cpu().numpy(), what="heter entry %d" % bi)
    single = bpl.event_csr_matvec(w[0], indices, indptr, events[bi], shape=shape)
    assert torch.equal(hom[bi], single)


# one group of all entries (listed one virtual row per thread, then eight per thread); groups bounded by the width of the
# virtual output (33 entries of 100,000 columns: two groups) and a last group of fewer entries; events shared by entries
@pytest.mark.parametrize("n_row,n_col,mean,batch,eb", [(900, 700, 40, 33, 33), (30_000, 3000, 5, 21, 21),
                                                       (500, 100_000, 60, 33, 11), (40, 9000, 30, 23, 23)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_batching_transposed_in_groups(cuda, oracle_mod, n_row, n_col, mean, batch, eb, dtype):
  rng = np.random.default_rng(n_row)
  counts = np.minimum(rng.poisson(mean, size=n_row), n_col)
  indices, indptr = synth.counted_csr(counts, n_col, seed=n_row)
  data = rng.standard_normal(indices.shape[0]).astype(dtype)
  print("case", n_row, n_col, batch, eb, dtype.__name__, flush=True)
  for rate in (0.02, 0.6):
    events = rng.random((eb, n_row)) < rate
    _check(oracle_mod, data[None], indices[None], indptr[None], events, batch, (n_row, n_col), True, "heter")
    one = np.full((1, 1), 0.7, dtype=dtype)
    got, want = _check(oracle_mod, one, indices[None], indptr[None], events, batch, (n_row, n_col), True, "homo")
    assert np.array_equal(got, want)  # (counts: the reference's bits whatever the order)


def test_batching_transposed_with_every_event_set(cuda):
  # 40 entries of 8e6 nonzeros: one group of them has 3.2e8 pairs, more than the runs of the sort hold; what finds them full
  # goes through atomics on device memory, which is right but takes five times as long.  Integer weights: exact sums.
  n_row, n_col, batch = 20_000, 20_000, 40
  rng = np.random.default_rng(3)
  indptr = np.arange(n_row + 1, dtype=np.int32) * 400
  indices = rng.integers(0, n_col, n_row * 400).astype(np.int32)
  data = rng.integers(-3, 4, indices.shape[0]).astype(np.float32)
  events = np.ones((batch, n_row), bool)
  events[5], events[17, ::2] = False, False
  dev = [torch.from_numpy(a).to(cuda) for a in (data[None], indices[None], indptr[None], events)]
  call = lambda b: bpl.event_csr_matvec_batching(*dev[:3], dev[3][:b], batch_size=b, shape=(n_row, n_col), transpose=True)
  got = call(batch).cpu().numpy()
  want = np.bincount(indices, weights=data, minlength=n_col)
  half = np.repeat(np.arange(n_row) % 2 == 1, 400)
  for b in range(batch):
    if b == 5:
      assert not got[b].any()
    elif b == 17:
      assert np.array_equal(got[b], np.bincount(indices[half], weights=data[half], minlength=n_col))
    else:
      assert np.array_equal(got[b], want)
  times = {}
  for b in (8, batch):  # (eight entries' pairs fit in any case)
    times[b] = []
    for _ in range(4):
      t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
      t0.record()
      call(b)
      t1.record()
      t1.synchronize()
      times[b].append(t0.elapsed_time(t1) / b)
  assert min(times[batch]) < 2.0 * min(times[8]), times


def test_batching_transposed_shares_out_long_rows_of_more_nonzeros_than_32_bits_count(cuda):
  # 600 rows of a million nonzeros: eight entries of them are 4.8e9, seven 4.2e9 (below 2^32).  Two rows are active: they
  # are shared out among the workgroups in either case (a workgroup to a row takes some 200 rounds one after the other).
  n_row, n_col = 600, 1_000_000
  indices = torch.arange(n_col, dtype=torch.int32, device=cuda).repeat(n_row)[None]
  indptr = (torch.arange(n_row + 1, dtype=torch.int64, device=cuda) * n_col).to(torch.int32)[None]
  one = torch.ones((1, 1), device=cuda)
  times = {}
  for batch in (7, 8):
    events = torch.zeros((batch, n_row), dtype=torch.bool, device=cuda)
    events[0, 0], events[batch - 1, n_row - 1] = True, True
    call = lambda: bpl.event_csr_matvec_batching(one, indices, indptr, events, batch_size=batch, shape=(n_row, n_col), transpose=True)
    got = call()
    assert bool((got == events.any(1).float()[:, None]).all())
    times[batch] = []
    for _ in range(5):
      t0, t1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
      t0.record()
      call()
      t1.record()
      t1.synchronize()
      times[batch].append(t0.elapsed_time(t1))
  print(times)
  assert min(times[8]) < 2.0 * min(times[7]), times
