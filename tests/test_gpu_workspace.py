"""The library's scratch memory (one cached allocation per stream): a buffer that was handed out
is never freed when a larger one replaces it, and nothing is allocated while the stream is being
captured into a HIP graph (the call fails instead and enqueues nothing)."""
import ctypes

import numpy as np
import pytest
import torch

import brainpylib_amd as bpl
from brainpylib_amd import _lib, sparse_ops
import benchdata as synth
from util import jitconn_by_lane

pytestmark = pytest.mark.gpu


def _query(stream_handle):
  lib = _lib.lib()
  lib.bpl_stream_workspace_query.restype = ctypes.c_int
  lib.bpl_stream_workspace_query.argtypes = [ctypes.c_void_p, ctypes.POINTER(ctypes.c_void_p),
                                             ctypes.POINTER(ctypes.c_size_t), ctypes.POINTER(ctypes.c_size_t)]
  ptr, size, retired = ctypes.c_void_p(), ctypes.c_size_t(), ctypes.c_size_t()
  has = lib.bpl_stream_workspace_query(ctypes.c_void_p(stream_handle), ctypes.byref(ptr), ctypes.byref(size),
                                       ctypes.byref(retired))
  return bool(has), ptr.value, size.value, retired.value


def _scatter_inputs(cuda, n_row, n_col, seed, dtype=np.float32):
  rng = np.random.default_rng(seed)
  indices, indptr = synth.counted_csr(rng.poisson(30, size=n_row), n_col, seed=seed)
  data = torch.from_numpy(rng.standard_normal(indices.shape[0]).astype(dtype)).to(cuda)
  ev = torch.from_numpy(rng.random(n_row) < 0.1).to(cuda)
  return data, torch.from_numpy(indices).to(cuda), torch.from_numpy(indptr).to(cuda), ev


def test_outgrown_buffer_is_retired_not_freed(cuda):
  s = torch.cuda.Stream()
  small = _scatter_inputs(cuda, 20_000, 20_000, 1)     # sorted scatter: 4,096 pairs per row, 0.6 GB of runs
  large = _scatter_inputs(cuda, 100_000, 100_000, 2)   # 1 GB of runs: a larger buffer
  torch.cuda.synchronize()
  with torch.cuda.stream(s):
    assert not _query(s.cuda_stream)[0]
    a = bpl.event_csr_matvec(*small, shape=(20_000, 20_000), transpose=True)
    has, p1, n1, r1 = _query(s.cuda_stream)
    assert has and p1 and n1 > 0 and r1 == 0
    b = bpl.event_csr_matvec(*large, shape=(100_000, 100_000), transpose=True)
    has, p2, n2, r2 = _query(s.cuda_stream)
    assert has and p2 != p1 and n2 >= 2 * n1
    assert r2 == n1, "the first buffer is kept (retired), not freed"
    # the same sizes again: no further growth
    a2 = bpl.event_csr_matvec(*small, shape=(20_000, 20_000), transpose=True)
    assert _query(s.cuda_stream)[1:] == (p2, n2, r2)
  s.synchronize()
  assert torch.allclose(a, a2, rtol=1e-5, atol=1e-5)
  # the retired buffer is still a valid allocation of its old size
  hip = ctypes.CDLL("libamdhip64.so")
  base, size = ctypes.c_void_p(), ctypes.c_size_t()
  rc = hip.hipMemGetAddressRange(ctypes.byref(base), ctypes.byref(size), ctypes.c_void_p(p1))
  assert rc == 0 and base.value == p1 and size.value == n1
  del b


def test_growth_is_refused_during_capture_and_works_after_a_warm_up(cuda, oracle_mod):
  s = torch.cuda.Stream()
  args = _scatter_inputs(cuda, 30_000, 30_000, 3)
  torch.cuda.synchronize()
  g = torch.cuda.CUDAGraph()
  with torch.cuda.stream(s):
    out = torch.zeros(30_000, dtype=torch.float32, device=cuda)
  s.synchronize()
  # cold stream: the call would have to allocate inside the capture; it must fail loudly instead
  with pytest.raises(RuntimeError, match="being captured"):
    with torch.cuda.graph(g, stream=s):
      bpl.event_csr_matvec(*args, shape=(30_000, 30_000), transpose=True)
  torch.cuda.synchronize()
  assert not _query(s.cuda_stream)[0], "nothing was allocated"
  # warmed on the stream first, the same call is captured and replays onto the same buffer
  with torch.cuda.stream(s):
    want = bpl.event_csr_matvec(*args, shape=(30_000, 30_000), transpose=True).clone()
  s.synchronize()
  # (the stream's first call: its counters and scratch memory were allocated inside it)
  host = [a.cpu().numpy() for a in args]
  ref = oracle_mod.event_csr_matvec(*host, shape=(30_000, 30_000), transpose=True)
  assert np.allclose(want.cpu().numpy(), ref, rtol=1e-5, atol=1e-5)
  before = _query(s.cuda_stream)
  g2 = torch.cuda.CUDAGraph()
  with torch.cuda.graph(g2, stream=s):
    out = bpl.event_csr_matvec(*args, shape=(30_000, 30_000), transpose=True)
  for _ in range(3):
    out.zero_()
    g2.replay()
    torch.cuda.synchronize()
    assert torch.allclose(out, want, rtol=1e-5, atol=1e-6)
  # a larger eager call on that stream afterwards moves on to a new buffer and leaves the graph's alone
  big = _scatter_inputs(cuda, 100_000, 120_000, 4, np.float64)  # (2 GB of float64 pairs)
  with torch.cuda.stream(s):
    bpl.event_csr_matvec(*big, shape=(100_000, 120_000), transpose=True)
  s.synchronize()
  after = _query(s.cuda_stream)
  assert after[1] != before[1] and after[3] >= before[2]
  out.zero_()
  g2.replay()
  torch.cuda.synchronize()
  assert torch.allclose(out, want, rtol=1e-5, atol=1e-6)


def test_calls_that_did_without_scratch_memory_are_captured_on_a_cold_stream(cuda):
  n_row, n_col = 2_000, 60_000
  rng = np.random.default_rng(5)
  indices, indptr = synth.fixed_count_csr(n_row, n_col, 600, seed=5)
  data = torch.from_numpy(rng.integers(-3, 4, size=indices.shape[0]).astype(np.float32)).to(cuda)
  idx, ptr = torch.from_numpy(indices).to(cuda), torch.from_numpy(indptr).to(cuda)
  x = torch.zeros(n_col, dtype=torch.float32, device=cuda)
  v = torch.zeros(n_row, dtype=torch.float32, device=cuda)
  s = torch.cuda.Stream()
  torch.cuda.synchronize()
  g = torch.cuda.CUDAGraph()
  with torch.cuda.graph(g, stream=s):
    y = bpl.csr_matvec(data, idx, ptr, x, shape=(n_row, n_col))
    products, sums = sparse_ops._gradients(data, idx, ptr, v, x, (n_row, n_col), True)
  for i in range(3):  # (eager work between the replays; integers: exact sums)
    x.copy_(torch.from_numpy(rng.integers(-4, 5, size=n_col).astype(np.float32)))
    v.copy_(torch.from_numpy(rng.integers(-4, 5, size=n_row).astype(np.float32)))
    torch.cuda.synchronize()
    g.replay()
    torch.cuda.synchronize()
    want, want_sums = sparse_ops._gradients(data, idx, ptr, v, x, (n_row, n_col), True)
    assert torch.equal(products, want), i
    assert torch.equal(y, want_sums), i
    assert sums is None or torch.equal(sums, want_sums)


def test_batched_scatter_of_a_small_network_is_captured_on_a_cold_stream(cuda):
  n, batch = 1_000, 20
  rng = np.random.default_rng(6)
  indices, indptr = synth.fixed_count_csr(n, n, 50, seed=6)
  data = torch.from_numpy(rng.integers(-3, 4, size=indices.shape[0]).astype(np.float32)).to(cuda).reshape(1, -1)
  idx, ptr = (torch.from_numpy(a).to(cuda).reshape(1, -1) for a in (indices, indptr))
  events = torch.zeros((batch, n), dtype=torch.bool, device=cuda)
  call = lambda: bpl.event_csr_matvec_batching(data, idx, ptr, events, batch_size=batch, shape=(n, n), transpose=True)
  s = torch.cuda.Stream()
  torch.cuda.synchronize()
  g = torch.cuda.CUDAGraph()
  with torch.cuda.graph(g, stream=s):
    out = call()
  for i in range(3):
    events.copy_(torch.from_numpy(rng.random((batch, n)) < 0.1))
    torch.cuda.synchronize()
    g.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, call()), i  # (integers: exact in any order)


def test_scratch_memory_of_a_batch_of_a_small_network(cuda):
  # the batching descriptor says how many nonzeros there are: 20 entries of 1,000 x 1,000 with 50 per row hold 42 MB of runs
  # and a quarter of head room, not what 4,096 pairs for every column would take (655 MB)
  s = torch.cuda.Stream()
  rng = np.random.default_rng(8)
  indices = torch.from_numpy(rng.integers(0, 1000, (1, 50_000)).astype(np.int32)).to(cuda)
  indptr = (torch.arange(1001, dtype=torch.int32) * 50)[None].to(cuda)
  data = torch.ones((1, 50_000), device=cuda)
  events = torch.ones((20, 1000), dtype=torch.bool, device=cuda)
  torch.cuda.synchronize()
  with torch.cuda.stream(s):
    out = bpl.event_csr_matvec_batching(data, indices, indptr, events, batch_size=20, shape=(1000, 1000), transpose=True)
    has, _, size, _ = _query(s.cuda_stream)
  s.synchronize()
  assert has and size < 60e6, size
  assert torch.equal(out.cpu(), torch.bincount(indices[0].cpu(), minlength=1000).to(torch.float32).expand(20, -1))


@pytest.mark.parametrize("n_in", [151_552, 151_553, 311_296])
def test_normal_row_walk_is_captured_on_a_cold_stream(cuda, n_in, capfd):
  # few outputs, byte events: their bitmap lies in LDS and no scratch memory is needed, whatever the weights
  ev = torch.from_numpy(np.random.default_rng(n_in).random(n_in) < 0.1).to(cuda)
  kw = dict(w_mu=0.1, w_sigma=0.5, conn_prob=0.01, shape=(300, n_in), seed=5, outdim_parallel=True)
  want = bpl.event_matvec_prob_conn_normal_weight(ev, **kw)
  torch.cuda.synchronize()
  s, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
  capfd.readouterr()
  with torch.cuda.graph(g, stream=s):
    out = bpl.event_matvec_prob_conn_normal_weight(ev, **kw)
  assert "brainpylib_amd" not in capfd.readouterr().err
  assert not _query(s.cuda_stream)[0], "nothing was allocated"
  for _ in range(3):
    out.zero_()
    g.replay()
    torch.cuda.synchronize()
    # (the same addends in float64, in another order, rounded once)
    torch.testing.assert_close(out, want, rtol=3e-7, atol=1e-6)


def test_matmat_is_captured_where_there_is_no_room_for_generator_states(cuda, capfd):
  # the stream's scratch memory holds the transposed operand (64 rows of 4,000 inputs) and not the states of 3,000
  # columns: the waves of a captured call seed their own generators, with the same result
  hip = ctypes.CDLL("libamdhip64.so")
  handle = ctypes.c_void_p()
  assert hip.hipStreamCreate(ctypes.byref(handle)) == 0
  s, g = torch.cuda.ExternalStream(handle.value), torch.cuda.CUDAGraph()
  X = torch.from_numpy(np.random.default_rng(5).standard_normal((64, 4000)).astype(np.float32)).to(cuda)
  call = lambda n: bpl.matmat_prob_conn_uniform_weight(X, w_low=-0.5, w_high=1.5, conn_prob=0.01, shape=(4000, n), seed=5)
  want = call(3000)
  torch.cuda.synchronize()
  with torch.cuda.stream(s):
    call(100)
  s.synchronize()
  before = _query(s.cuda_stream)
  assert before[0] and before[2] < 3000 * 624 * 4
  capfd.readouterr()
  with torch.cuda.graph(g, stream=s):
    out = call(3000)
  assert "brainpylib_amd" not in capfd.readouterr().err
  assert _query(s.cuda_stream) == before, "nothing was allocated"
  for _ in range(3):
    out.zero_()
    g.replay()
    torch.cuda.synchronize()
    assert torch.equal(out, want)


@pytest.mark.parametrize("conn_prob", [0.005, 0.012])
def test_row_walk_is_captured_where_the_stream_has_rings_but_no_counters(cuda, capfd, conn_prob):
  # more than four batches of streams for each of 512 workgroups, and no counter to take them from: they are shared out evenly, and the
  # call, which succeeds, prints nothing.  (Rows of 240 synapses; those of 100 are walked by lanes, which need neither.)
  rng = np.random.default_rng(3)
  handle = ctypes.c_void_p()  # (a stream of its own: torch's come from a pool and may have counters from elsewhere)
  assert ctypes.CDLL("libamdhip64.so").hipStreamCreate(ctypes.byref(handle)) == 0
  s, g = torch.cuda.ExternalStream(handle.value), torch.cuda.CUDAGraph()
  x = torch.from_numpy(rng.random(100_000, dtype=np.float32)).to(cuda)
  torch.cuda.synchronize()
  with torch.cuda.stream(s):  # (bins of 0.75 GB: scratch memory, no counters)
    bpl.matvec_prob_conn_homo_weight(x, 0.5, conn_prob=0.01, shape=(100_000, 100_000), seed=1, outdim_parallel=False)
  s.synchronize()
  before = _query(s.cuda_stream)
  n_in = 20_000
  ev = torch.zeros(n_in, dtype=torch.bool, device=cuda)
  kw = dict(weight=1.0, conn_prob=conn_prob, shape=(140_001, n_in), seed=5, outdim_parallel=True)
  assert jitconn_by_lane("homo", 4, 140_001, n_in, conn_prob, event_bytes=1) == (conn_prob < 0.01)
  bpl.event_matvec_prob_conn_homo_weight(ev, **kw)
  torch.cuda.synchronize()
  capfd.readouterr()
  with torch.cuda.graph(g, stream=s):
    out = bpl.event_matvec_prob_conn_homo_weight(ev, **kw)
  assert "brainpylib_amd" not in capfd.readouterr().err
  assert _query(s.cuda_stream) == before, "nothing was allocated"
  for i in range(3):
    ev.copy_(torch.from_numpy(rng.random(n_in) < 0.1))
    out.zero_()
    torch.cuda.synchronize()
    g.replay()
    torch.cuda.synchronize()
    want = bpl.event_matvec_prob_conn_homo_weight(ev, **kw)
    assert want.sum() > 0 and torch.equal(out, want), i
