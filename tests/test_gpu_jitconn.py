"""GPU parity of the jitconn operators through the C ABI.

Generator contract: stream i is std::mt19937{seed + i}; output row i of a row-walk target
(input column i of an *_atomic_* target) is what the reference's CPU kernel computes for that
single stream.  Checked against (a) golden vectors produced by the reference's compiled CPU
kernels one stream at a time, (b) the per-stream oracle, (c) exact integer probes that pin the
generated index sets, (d) full-size properties."""
import ctypes
import json
import os

import numpy as np
import pytest
import torch

import brainpylib_amd as bpl
from brainpylib_amd import _lib
import benchdata as synth
from util import JIT_SHAPES, assert_close, assert_close_reordered, jitconn_by_lane

pytestmark = pytest.mark.gpu
GOLD = os.path.join(os.path.dirname(__file__), "golden")
KINDS_BUILT = ("homo", "uniform", "normal")


def kernel_call(inp, *, w_kind, w_a=0.0, w_b=0.0, log_p, seed, n_row, n_col, col_walk, dense, out_dtype=None,
                device="cuda:0"):
  """Calls the custom-call target directly (homo returns counts / plain sums)."""
  t = torch.from_numpy(np.ascontiguousarray(inp)).to(device)
  if t.dtype == torch.bool:
    odt = torch.float32 if out_dtype in (None, np.float32, "float32") else torch.float64
    suffix = ("_float" if odt == torch.float32 else "_double") + "_bool"
    prefix = "gpu_event_matvec"
  else:
    odt = t.dtype
    tn = "_float" if odt == torch.float32 else "_double"
    prefix, suffix = ("gpu_matvec", tn) if dense else ("gpu_event_matvec", tn + tn)
  if w_kind == "homo":
    opaque = _lib.build_jitconn_prob_homo_descriptor(n_row, n_col, seed, log_p)
  elif w_kind == "uniform":
    # descriptor carries (w_min, w_range); the range is formed in the result type like the CPU path's b - a
    np_dt = np.float32 if odt == torch.float32 else np.float64
    opaque = _lib.build_jitconn_prob_uniform_descriptor(n_row, n_col, seed, log_p, float(np_dt(w_a)),
                                                        float(np_dt(np_dt(w_b) - np_dt(w_a))))
  else:
    opaque = _lib.build_jitconn_prob_normal_descriptor(n_row, n_col, seed, log_p, w_a, w_b)
  out = torch.full((n_row,), 123.0, dtype=odt, device=device)  # poisoned: every element must be written
  name = prefix + ("_atomic" if col_walk else "") + "_prob_" + w_kind + "_v2" + suffix
  _lib.custom_call(name, [t, out], opaque)
  return out.cpu().numpy()


def _golden_cases():
  z = np.load(os.path.join(GOLD, "jitconn_cpu_reference.npz"))
  zs = np.load(os.path.join(GOLD, "jitconn_cpu_reference_streams.npz"))
  n = sum(1 for k in z.files if k.startswith("meta_"))
  for i in range(n):
    yield i, z["in_%d" % i], json.loads(str(z["meta_%d" % i])), zs["out_%d" % i]


def _abs_bound(oracle, inp, meta, dtype):
  """sum of |addends| per output element, for the reordering tolerance: rebuilt from the
  oracle's per-stream (index, weight) lists"""
  mag_in = np.abs(inp.astype(np.float64)) if meta["dense"] else (inp != 0).astype(np.float64)
  lp = oracle.log_p_of(meta["conn_prob"])
  n_outer, n_inner = (meta["n_col"], meta["n_row"]) if meta["col_walk"] else (meta["n_row"], meta["n_col"])
  bound = np.zeros(meta["n_row"])
  for s_ in range(n_outer):
    idx, w = oracle.jitconn_stream_weights(meta["seed"] + s_, meta["w_kind"], meta["w_a"], meta["w_b"], lp, n_inner,
                                           dtype=dtype)
    if meta["col_walk"]:
      np.add.at(bound, idx, np.abs(w.astype(np.float64)) * mag_in[s_])
    else:
      bound[s_] = (np.abs(w.astype(np.float64)) * mag_in[idx]).sum()
  return bound


def test_reference_golden_streams(cuda, oracle_mod):
  n = 0
  for i, inp, meta, want in _golden_cases():
    if meta["w_kind"] not in KINDS_BUILT:
      continue
    got = kernel_call(inp, w_kind=meta["w_kind"], w_a=meta["w_a"], w_b=meta["w_b"],
                      log_p=oracle_mod.log_p_of(meta["conn_prob"]), seed=meta["seed"], n_row=meta["n_row"],
                      n_col=meta["n_col"], col_walk=meta["col_walk"], dense=meta["dense"], out_dtype=meta["out_dtype"])
    if meta["w_kind"] == "homo" and not meta["dense"]:
      assert np.array_equal(got.astype(np.float64), want.astype(np.float64)), (i, meta)  # counts: exact
    else:
      dt = np.float32 if got.dtype == np.float32 else np.float64
      assert_close_reordered(got, want, _abs_bound(oracle_mod, inp, meta, dt), dt, what=str(meta))
    n += 1
  assert n == 450


@pytest.mark.parametrize("shape", JIT_SHAPES + [(64, 64), (3, 70000)])
@pytest.mark.parametrize("p", [0.01, 0.1, 0.5])
def test_index_sets_bit_exact_via_integer_probes(cuda, oracle_mod, shape, p):
  # dense float64 vectors 1, c and c^2 give count, sum and sum of squares of every row's index set,
  # all exact integers below 2^53: equal to the oracle's bit for bit
  n_row, n_col = shape
  lp = oracle_mod.log_p_of(p)
  c = np.arange(n_col, dtype=np.float64)
  print("case", shape, p, flush=True)
  for col_walk in (False, True):
    for vec in (np.ones(n_col), c, c * c):
      want = oracle_mod.jitconn_matvec(vec, log_p=lp, seed=1234, n_row=n_row, n_col=n_col, col_walk=col_walk,
                                       dense=True, per_stream_seed=True)
      got = kernel_call(vec, w_kind="homo", log_p=lp, seed=1234, n_row=n_row, n_col=n_col, col_walk=col_walk,
                        dense=True)
      assert np.array_equal(got, want), (shape, p, col_walk)


@pytest.mark.parametrize("n_out,n_in,p", [(3000, 1500, 0.05), (5000, 4000, 0.05), (9000, 40_000, 0.02),
                                          (20_000, 30_000, 0.03)])
def test_event_column_walk_in_every_regime(cuda, oracle_mod, n_out, n_in, p):
  # few input columns: every wave lists and seeds its own; from 2,048 columns on: a device list of the active
  # columns and generators seeded ahead, the pairs added with atomics; from ten million possible pairs on:
  # through bins.  Unit weight: the outputs are synapse counts, equal to the oracle's bit for bit, at little
  # and at much activity, twice in a row (the list's counter must be back at zero).
  lp = oracle_mod.log_p_of(p)
  rng = np.random.default_rng(n_in)
  for rate in (0.004, 0.3):
    ev = rng.random(n_in) < rate
    want = oracle_mod.jitconn_matvec(ev, log_p=lp, seed=99, n_row=n_out, n_col=n_in, col_walk=True, dense=False,
                                     per_stream_seed=True)
    for _ in range(2):
      got = kernel_call(ev, w_kind="homo", log_p=lp, seed=99, n_row=n_out, n_col=n_in, col_walk=True, dense=False)
      assert np.array_equal(got, want), (n_out, n_in, p, rate)
  # uniform weights and float events: sums of a few terms in any order
  evf = (rng.random(n_in) < 0.05).astype(np.float32)
  want = oracle_mod.jitconn_matvec(evf, log_p=lp, seed=5, n_row=n_out, n_col=n_in, col_walk=True, dense=False,
                                   per_stream_seed=True, w_kind="uniform", w_a=-1.0, w_b=2.0)
  got = kernel_call(evf, w_kind="uniform", w_a=-1.0, w_b=2.0, log_p=lp, seed=5, n_row=n_out, n_col=n_in, col_walk=True,
                    dense=False)
  np.testing.assert_allclose(got, want, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("n_in", [320_000, 1_500_000, 5_000_000])
def test_row_walk_with_a_two_level_event_bitmap(cuda, oracle_mod, n_in):
  # more inputs than the row walk ever keeps an exact bitmap of in LDS (311,296): a coarse
  # bitmap in LDS (one bit per 2, 8 and 32 inputs here) and the exact one in global memory, whose
  # word is looked at one batch late.  Bool and float events, all weight kinds; counts exact.
  n_out = 300
  rng = np.random.default_rng(n_in)
  ev = rng.random(n_in) < 0.02
  lp = oracle_mod.log_p_of(2000.0 / n_in)
  for inp in (ev, (ev * rng.uniform(0.5, 2.0, n_in)).astype(np.float32)):
    dense = None if inp.dtype == np.bool_ else False
    want = oracle_mod.jitconn_matvec(inp, log_p=lp, seed=77, n_row=n_out, n_col=n_in, dense=dense)
    got = kernel_call(inp, w_kind="homo", log_p=lp, seed=77, n_row=n_out, n_col=n_in, col_walk=False, dense=False)
    assert want.sum() > 0 and np.array_equal(got, want)
  for w_kind, a, b in (("uniform", 0.25, 1.75), ("normal", 0.5, 2.0)):
    want, mag = oracle_mod.jitconn_matvec(ev, w_kind=w_kind, w_a=a, w_b=b, log_p=lp, seed=77, n_row=n_out, n_col=n_in,
                                          return_abs=True)
    got = kernel_call(ev, w_kind=w_kind, w_a=a, w_b=b, log_p=lp, seed=77, n_row=n_out, n_col=n_in, col_walk=False,
                      dense=False)
    assert_close_reordered(got, want, mag, np.float32, what="two-level row walk %s" % w_kind)


def test_row_walk_lanes_past_the_end_of_a_row_count_nothing(cuda, oracle_mod):
  # two-level bitmap with EVERY event set (all coarse and exact bits are ones): the lanes of a row's last
  # batch that lie past the end of the row look up position 0, whose word of the exact bitmap holds no input, so a
  # row's count is its stream's synapse count exactly.  Rows of about 3 synapses: nearly every lane of every row's only batch is past the end.
  # (8,200 outputs: the walk that seeds its generators itself)
  for n_out, n_in in ((400, 311_297), (400, 320_000), (400, 1_310_720), (8_200, 320_000)):
    ev = np.ones(n_in, dtype=np.bool_)
    lp = oracle_mod.log_p_of(3.0 / n_in)
    got = kernel_call(ev, w_kind="homo", log_p=lp, seed=123, n_row=n_out, n_col=n_in, col_walk=False, dense=False)
    want = np.array([oracle_mod.jitconn_stream_indices(123 + r, lp, n_in)[1] for r in range(n_out)], dtype=np.float32)
    assert want.sum() > 0 and np.array_equal(got, want), n_in


def test_full_matrix_recovered_by_one_hot_events(cuda, oracle_mod):
  # every entry of a 100 x 200 implicit matrix, both walks, against the per-stream oracle's index lists
  n_row, n_col, seed = 100, 200, 77
  lp = oracle_mod.log_p_of(0.1)
  M = np.zeros((n_row, n_col))
  for r in range(n_row):
    idx, _ = oracle_mod.jitconn_stream_indices(seed + r, lp, n_col)
    M[r, idx] = 1
  got = np.zeros((n_row, n_col))
  for c in range(n_col):
    ev = np.zeros(n_col, dtype=bool)
    ev[c] = True
    got[:, c] = kernel_call(ev, w_kind="homo", log_p=lp, seed=seed, n_row=n_row, n_col=n_col, col_walk=False,
                            dense=False)
  assert np.array_equal(got, M)
  # column walk of the swapped shape generates the transpose of the same matrix
  gotT = np.zeros((n_col, n_row))
  for r in range(n_row):
    ev = np.zeros(n_row, dtype=bool)
    ev[r] = True
    gotT[:, r] = kernel_call(ev, w_kind="homo", log_p=lp, seed=seed, n_row=n_col, n_col=n_row, col_walk=True,
                             dense=False)
  assert np.array_equal(gotT, M.T)
  assert M[:, 0].sum() == 0  # index 0 is never connected


def test_closed_form_and_edges(cuda, oracle_mod):
  lp = oracle_mod.log_p_of(1.0)  # every skip is 1: indices 1..n-1
  v = np.arange(1, 301, dtype=np.float64)
  out = kernel_call(v, w_kind="homo", log_p=lp, seed=3, n_row=70, n_col=300, col_walk=False, dense=True)
  assert np.array_equal(out, np.full(70, v[1:].sum()))
  out = kernel_call(v[:70].copy(), w_kind="homo", log_p=lp, seed=3, n_row=300, n_col=70, col_walk=True, dense=True)
  want = np.full(300, v[:70].sum())
  want[0] = 0
  assert np.array_equal(out, want)
  # seed + stream wraps modulo 2^32
  ev = np.random.default_rng(0).random(500) < 0.5
  lp = oracle_mod.log_p_of(0.05)
  want = oracle_mod.jitconn_matvec(ev, log_p=lp, seed=2 ** 32 - 3, n_row=10, n_col=500, per_stream_seed=True)
  got = kernel_call(ev, w_kind="homo", log_p=lp, seed=2 ** 32 - 3, n_row=10, n_col=500, col_walk=False, dense=False)
  assert np.array_equal(got, want)
  # silent input, single element, and an invalid log_p that must be refused, not looped on
  got = kernel_call(np.zeros(500, bool), w_kind="homo", log_p=lp, seed=1, n_row=10, n_col=500, col_walk=True, dense=False)
  assert not got.any()
  got = kernel_call(np.ones(1, bool), w_kind="homo", log_p=lp, seed=1, n_row=5, n_col=1, col_walk=False, dense=False)
  assert not got.any()
  with pytest.raises(RuntimeError, match="log_p must be finite and negative"):
    kernel_call(ev, w_kind="homo", log_p=0.0, seed=1, n_row=10, n_col=500, col_walk=False, dense=False)


@pytest.mark.parametrize("shape", JIT_SHAPES)
@pytest.mark.parametrize("outdim_parallel", [True, False])
def test_wrapper_determinism_and_shape_swap(cuda, shape, outdim_parallel):
  # brainpylib/_src/jitconn_ops/tests/test_event_matvec.py:63-87
  rng = np.random.default_rng(1)
  for transpose in (False, True):
    ev = rng.random(shape[0] if transpose else shape[1]) < 0.1
    kw = dict(conn_prob=0.1, seed=1234, outdim_parallel=outdim_parallel)
    r1 = bpl.event_matvec_prob_conn_homo_weight(ev, 1.5, shape=shape, transpose=transpose, **kw)
    r2 = bpl.event_matvec_prob_conn_homo_weight(ev, 1.5, shape=shape, transpose=transpose, **kw)
    r3 = bpl.event_matvec_prob_conn_homo_weight(ev, 1.5, shape=shape[::-1], transpose=not transpose, **kw)
    assert torch.equal(r1, r2) and torch.equal(r1, r3)
    assert r1.shape[0] == (shape[1] if transpose else shape[0]) and r1.dtype == torch.float32
    u1 = bpl.event_matvec_prob_conn_uniform_weight(ev, w_low=-1.0, w_high=1.0, shape=shape, transpose=transpose, **kw)
    u3 = bpl.event_matvec_prob_conn_uniform_weight(ev, w_low=-1.0, w_high=1.0, shape=shape[::-1],
                                                   transpose=not transpose, **kw)
    assert torch.allclose(u1, u3, rtol=1e-5, atol=1e-6)
    fv = rng.standard_normal(ev.shape[0]).astype(np.float32)
    m1 = bpl.matvec_prob_conn_homo_weight(fv, 0.5, shape=shape, transpose=transpose, **kw)
    m3 = bpl.matvec_prob_conn_homo_weight(fv, 0.5, shape=shape[::-1], transpose=not transpose, **kw)
    assert torch.allclose(m1, m3, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("w_kind,a,b", [("homo", 0.0, 0.0), ("uniform", -1.0, 1.0), ("normal", 0.5, 2.0)])
def test_row_walk_and_column_walk_are_adjoint(cuda, oracle_mod, w_kind, a, b):
  # flipping transpose AND outdim_parallel gives M^T of the same M: <y, M x> == <M^T y, x>
  n_out, n_in = 300, 500
  rng = np.random.default_rng(5)
  x = rng.integers(-3, 4, n_in).astype(np.float64)
  y = rng.integers(-3, 4, n_out).astype(np.float64)
  lp = oracle_mod.log_p_of(0.2)
  Mx = kernel_call(x, w_kind=w_kind, w_a=a, w_b=b, log_p=lp, seed=11, n_row=n_out, n_col=n_in, col_walk=False, dense=True)
  MTy = kernel_call(y, w_kind=w_kind, w_a=a, w_b=b, log_p=lp, seed=11, n_row=n_in, n_col=n_out, col_walk=True, dense=True)
  assert abs(y @ Mx - MTy @ x) <= 1e-9 * max(1.0, abs(y @ Mx))


@pytest.mark.parametrize("w_kind,a,b", [("uniform", 0.25, 1.75), ("normal", 0.5, 2.0)])
def test_single_weights_against_oracle_streams(cuda, oracle_mod, w_kind, a, b):
  # one-hot dense inputs isolate single weights of a stream.  Uniform weights must equal the
  # oracle's draws bit for bit; normal weights go through logf/sqrtf (libm on the host, the
  # device's own on the GPU) and may differ in the last place.
  n_row, n_col, seed = 4, 3000, 9
  lp = oracle_mod.log_p_of(0.05)
  for dt in (np.float32, np.float64):
    for r in range(n_row):
      idx, w = oracle_mod.jitconn_stream_weights(seed + r, w_kind, a, b, lp, n_col, dtype=dt)
      assert len(idx) > 100
      # all weights of the row at once: W[k] lands in output k of a column walk over one-hot ... use
      # the row walk with a one-hot per probe for a handful of positions spread over several batches
      for k in (0, 1, 2, 63, 64, 65, len(idx) // 2, len(idx) - 2, len(idx) - 1):
        e = np.zeros(n_col, dtype=dt)
        e[idx[k]] = 1
        got = kernel_call(e, w_kind=w_kind, w_a=a, w_b=b, log_p=lp, seed=seed, n_row=n_row, n_col=n_col,
                          col_walk=False, dense=True)
        if w_kind == "uniform":
          assert got[r] == w[k], (dt, r, k)
        else:
          assert abs(got[r] - w[k]) <= 4 * np.finfo(dt).eps * max(1.0, abs(w[k])), (dt, r, k, got[r], w[k])


def test_normal_weights_whole_rows(cuda, oracle_mod):
  # dense float64 probes c and c^2 weighted by the normal draws: compares every (index, weight)
  # pairing of long rows (many parser batches, both skip roles, batch-boundary carries)
  n_row, n_col, seed = 64, 20000, 5
  lp = oracle_mod.log_p_of(0.1)
  c = np.arange(n_col, dtype=np.float64) / n_col
  for dt in (np.float32, np.float64):
    for vec in (np.ones(n_col, dtype=dt), c.astype(dt), (c * c).astype(dt)):
      want = oracle_mod.jitconn_matvec(vec, w_kind="normal", w_a=0.1, w_b=1.0, log_p=lp, seed=seed, n_row=n_row,
                                       n_col=n_col, dense=True, per_stream_seed=True)
      got = kernel_call(vec, w_kind="normal", w_a=0.1, w_b=1.0, log_p=lp, seed=seed, n_row=n_row, n_col=n_col,
                        col_walk=False, dense=True)
      meta = dict(dense=True, conn_prob=0.1, col_walk=False, n_row=n_row, n_col=n_col, seed=seed, w_kind="normal",
                  w_a=0.1, w_b=1.0)
      assert_close_reordered(got, want, _abs_bound(oracle_mod, vec, meta, dt), dt, what="normal rows")


def test_config_jitconn_event_full_size(cuda, oracle_mod):
  # 1e6 x 1e6, conn_prob 0.001 (~1e9 implicit synapses), events 1 %, seed 42: all four flag
  # combinations.  Row walks: 300 sampled rows against single-stream oracle calls.  Column walks:
  # the whole output against the oracle run over the ~1e4 active columns only.  Plus the adjoint
  # identity between the two walks on exact integer data.
  c = synth.config_jitconn_event()
  n = c["shape"][0]
  ev = c["events"]
  lp = oracle_mod.log_p_of(c["conn_prob"])
  seed = c["seed"]
  got_row = kernel_call(ev, w_kind="homo", log_p=lp, seed=seed, n_row=n, n_col=n, col_walk=False, dense=False)
  rows = np.random.default_rng(0).choice(n, 300, replace=False)
  for r in rows:
    idx, cnt = oracle_mod.jitconn_stream_indices(seed + int(r), lp, n)
    assert cnt == idx.shape[0]
    assert got_row[r] == ev[idx].sum(), r
  got_col = kernel_call(ev, w_kind="homo", log_p=lp, seed=seed, n_row=n, n_col=n, col_walk=True, dense=False)
  want_col = np.zeros(n)
  for col in np.flatnonzero(ev):
    idx, _ = oracle_mod.jitconn_stream_indices(seed + int(col), lp, n)
    np.add.at(want_col, idx, 1.0)
  assert np.array_equal(got_col.astype(np.float64), want_col)
  # the public wrappers: weight applied afterwards, transpose only swaps the (square) shape
  w = bpl.event_matvec_prob_conn_homo_weight(ev, c["weight"], conn_prob=c["conn_prob"], shape=c["shape"], seed=seed)
  assert np.array_equal(w.cpu().numpy(), got_row * np.float32(0.1))
  wt = bpl.event_matvec_prob_conn_homo_weight(ev, c["weight"], conn_prob=c["conn_prob"], shape=c["shape"], seed=seed,
                                              transpose=True, outdim_parallel=False)
  assert np.array_equal(wt.cpu().numpy(), got_col * np.float32(0.1))
  # adjoint: <y, M x> == <M^T y, x>, counts are exact in fp32 below 2^24
  y = np.random.default_rng(1).random(n) < 0.01
  MTy = kernel_call(y, w_kind="homo", log_p=lp, seed=seed, n_row=n, n_col=n, col_walk=True, dense=False)
  assert float(got_row.astype(np.float64) @ y) == float(MTy.astype(np.float64) @ ev)


@pytest.mark.parametrize("m", [1, 5, 8, 15, 33, 64, 70, 128, 130, 300, 600, 2048])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_matmat_against_oracle_and_vmapped_matvec(cuda, oracle_mod, m, dtype):
  # m values of the reference test (matmat_testcase.py:39-44) plus tile boundaries of the kernel and row counts
  # that take several passes of 128 rows (the last one partly filled)
  k, n, seed, p = 230, 150, 7, 0.2
  X = np.random.default_rng(m).standard_normal((m, k)).astype(dtype)
  lp = oracle_mod.log_p_of(p)
  print("case", m, dtype.__name__, flush=True)
  # uniform weights: same operations in the same order as the CPU loop -> bit-exact
  want = oracle_mod.jitconn_matmat(X, w_kind="uniform", w_a=-0.5, w_b=1.5, log_p=lp, seed=seed, n=n)
  got = bpl.matmat_prob_conn_uniform_weight(X, w_low=-0.5, w_high=1.5, conn_prob=p, shape=(k, n), seed=seed).cpu().numpy()
  assert got.shape == (m, n) and np.array_equal(got, want)
  # normal weights: logf/sqrtf of the device vs libm may differ in the last place
  want, mag = oracle_mod.jitconn_matmat(X, w_kind="normal", w_a=0.0, w_b=0.01, log_p=lp, seed=seed, n=n, return_abs=True)
  got_t = bpl.matmat_prob_conn_normal_weight(X, w_mu=0.0, w_sigma=0.01, conn_prob=p, shape=(k, n), seed=seed)
  got = got_t.cpu().numpy()
  assert_close_reordered(got, want, mag, dtype, what="matmat normal")
  # the reference tests' identity: matmat(X) == vmap(matvec(transpose=True))(X)
  for i in range(0, m, max(1, m // 4)):
    yi = bpl.matvec_prob_conn_normal_weight(X[i], w_mu=0.0, w_sigma=0.01, conn_prob=p, shape=(k, n), seed=seed,
                                            transpose=True)
    assert torch.allclose(got_t[i], yi, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("n", [32_768, 140_000])
def test_matmat_with_generators_seeded_ahead(cuda, oracle_mod, n):
  # from 32,768 columns of M on their generators are seeded ahead by a kernel of its own, 131,072 at a time
  # (140,000: two chunks, the second one short); uniform weights are bit-exact as with any other size
  m, k, seed, p = 9, 60, 11, 0.1
  X = np.random.default_rng(n).standard_normal((m, k)).astype(np.float32)
  lp = oracle_mod.log_p_of(p)
  want = oracle_mod.jitconn_matmat(X, w_kind="uniform", w_a=-0.5, w_b=1.5, log_p=lp, seed=seed, n=n)
  for _ in range(2):
    got = bpl.matmat_prob_conn_uniform_weight(X, w_low=-0.5, w_high=1.5, conn_prob=p, shape=(k, n), seed=seed).cpu().numpy()
    assert got.shape == (m, n) and np.array_equal(got, want)


@pytest.mark.parametrize("w_kind,a,b", [("homo", 0.0, 0.0), ("uniform", 0.25, 1.75), ("normal", 0.5, 2.0)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n_out,n_in,p", [(5001, 900, 0.001), (10_000, 4000, 0.0025), (70_063, 3, 1.0), (70_063, 40, 0.5), (140_000, 1500, 0.04)])
def test_row_walk_of_short_streams(cuda, oracle_mod, w_kind, a, b, dtype, n_out, n_in, p):
  # a lane to a stream: outputs that are not a multiple of 64, streams without a synapse, every index connected (what is longer, with
  # normal weights 140,000 rows of 60 and some others, goes by wave: test_row_walk_of_normal_weights_that_go_on_behind_the_first_words)
  rng = np.random.default_rng(n_out)
  ev, vec = rng.random(n_in) < 0.3, rng.uniform(0.5, 2.0, n_in).astype(dtype)
  oracle_mod.set_threads(min(16, len(os.sched_getaffinity(0))))
  kw = dict(w_kind=w_kind, w_a=a, w_b=b, log_p=oracle_mod.log_p_of(p), seed=21, n_row=n_out, n_col=n_in, out_dtype=dtype)
  for inp, dense in ((ev, False), (vec, True)):
    want, mag = oracle_mod.jitconn_matvec(inp, dense=dense, return_abs=True, **kw)
    got = kernel_call(inp, col_walk=False, dense=dense, **kw)
    if w_kind == "homo" and not dense: assert np.array_equal(got, want)
    assert_close_reordered(got, want, mag, dtype, what="row walk of short streams")
  oracle_mod.set_threads(1)


@pytest.mark.parametrize("signed", [False, True])
@pytest.mark.parametrize("n_out,mean", [(3000, 20.0), (130_000, 100.0), (300_000, 167.0)])
def test_sums_of_short_streams_in_double(cuda, oracle_mod, n_out, mean, signed):
  # A lane adds a whole row.  The vector is cut in two whose sums are exact in whatever order: 40 bits behind the point, and the
  # 13 bits and fewer that are left.  The result may be half a unit of the last place off plus what is lost of the lost parts: at
  # most 2^-53 of each, which are 2^-53 of a partial sum each, of which there are at most 250 (300,000 rows: some by wave, in
  # 64 sums of a few addends and a tree of six additions, as many half units of the sum of the sizes)
  n_in = 600_000 if mean > 150 else 20_000
  rng = np.random.default_rng(n_out)
  vec = rng.uniform(0.5, 2.0, n_in) * (rng.choice([-1.0, 1.0], n_in) if signed else 1.0)
  high = np.round(vec * 2.0 ** 40) * 2.0 ** -40
  oracle_mod.set_threads(min(16, len(os.sched_getaffinity(0))))
  kw = dict(w_kind="homo", log_p=oracle_mod.log_p_of(mean / n_in), seed=400_012, n_row=n_out, n_col=n_in, dense=True)
  (a, mag), b = oracle_mod.jitconn_matvec(high, return_abs=True, **kw), oracle_mod.jitconn_matvec(vec - high, **kw)
  counts = oracle_mod.jitconn_matvec(np.ones(n_in), **kw)
  oracle_mod.set_threads(1)
  assert np.finfo(np.longdouble).nmant >= 63
  want = a.astype(np.longdouble) + b.astype(np.longdouble)
  off = np.abs(kernel_call(vec, col_walk=False, **kw).astype(np.longdouble) - want).astype(np.float64)
  bound = 2.0 ** -53 * np.abs(want).astype(np.float64) * (1 + 2.0 ** -50) + 250 ** 2 * 2.0 ** -106 * mag
  bound[counts > 226] = 10 * 2.0 ** -53 * mag[counts > 226]
  assert np.all(off <= bound), (off / np.abs(want).astype(np.float64)).max()


def test_sums_of_short_streams_with_infinities(cuda, oracle_mod):
  # infinite addends give what a plain sum gives: an infinity, or NaN where both kinds meet
  n_out, n_in = 5000, 900
  vec = np.random.default_rng(3).uniform(0.5, 2.0, n_in)
  vec[5], vec[400], vec[77] = np.inf, -np.inf, np.finfo(np.float64).max
  kw = dict(w_kind="homo", log_p=oracle_mod.log_p_of(0.03), seed=3, n_row=n_out, n_col=n_in, dense=True)
  want = oracle_mod.jitconn_matvec(vec, **kw)
  assert np.isnan(want).any() and (want == np.inf).any() and (want == -np.inf).any() and (np.abs(want) < 1e3).any()
  got = kernel_call(vec, col_walk=False, **kw)
  finite = np.isfinite(want)
  np.testing.assert_array_equal(got[~finite], want[~finite])
  np.testing.assert_allclose(got[finite], want[finite], rtol=50 * 2.0 ** -53)  # (some 50 addends of one sign)


@pytest.mark.parametrize("w_kind,a,b", [("homo", 0.0, 0.0), ("uniform", 0.25, 1.75), ("normal", 0.5, 2.0)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n_out,n_in,p", [(900, 5001, 0.001), (30_000, 33_000, 0.0003), (3, 70_063, 1.0), (40, 70_063, 0.5),
                                          (17_000, 140_000, 0.0035), (2_200_000, 2100, 0.0001)])
def test_column_walk_of_short_streams(cuda, oracle_mod, w_kind, a, b, dtype, n_out, n_in, p):
  # a lane to a column: batches of 64 that do not come out even, one window and several, no bins at all (events with few pairs);
  # 2,100 columns of 220 are walked by waves, into windows of 15 bits
  rng = np.random.default_rng(n_out)
  ev, vec = rng.random(n_in) < 0.1, rng.uniform(0.5, 2.0, n_in).astype(dtype) * (rng.random(n_in) < 0.9)
  oracle_mod.set_threads(min(16, len(os.sched_getaffinity(0))))
  kw = dict(w_kind=w_kind, w_a=a, w_b=b, log_p=oracle_mod.log_p_of(p), seed=21, n_row=n_out, n_col=n_in, out_dtype=dtype,
            col_walk=True)
  for inp, dense in ((ev, False), (vec.astype(dtype), True)):
    want, mag = oracle_mod.jitconn_matvec(inp, dense=dense, return_abs=True, **kw)
    got = kernel_call(inp, dense=dense, **kw)
    if w_kind == "homo" and not dense: assert np.array_equal(got, want)
    assert_close_reordered(got, want, mag, dtype, what="column walk of short streams")
  oracle_mod.set_threads(1)


@pytest.mark.parametrize("w_kind,mean,most", [("homo", 167.0, 226), ("uniform", 104.0, 150)])
def test_row_walk_of_streams_that_outlast_their_lane(cuda, oracle_mod, w_kind, mean, most):
  # among streams of so many synapses in the mean a few need more words than a lane can draw (454): those are walked
  # again by their wave
  n_out, n_in = 300_000, 600_000
  ones = np.ones(n_in, bool)
  oracle_mod.set_threads(min(16, len(os.sched_getaffinity(0))))
  kw = dict(log_p=oracle_mod.log_p_of(mean / n_in), seed=400_012, n_row=n_out, n_col=n_in, w_kind=w_kind, w_a=1.0, w_b=1.0,
            out_dtype=np.float32)
  counts = oracle_mod.jitconn_matvec(ones, dense=False, **kw)  # (every weight is 1)
  assert counts.max() > most, "no stream is long enough"
  assert np.array_equal(kernel_call(ones, col_walk=False, dense=False, **kw), counts)
  kw.update(w_b=2.0)
  vec = np.random.default_rng(7).uniform(0.5, 2.0, n_in).astype(np.float32)
  want, mag = oracle_mod.jitconn_matvec(vec, dense=True, return_abs=True, **kw)
  assert_close_reordered(kernel_call(vec, col_walk=False, dense=True, **kw), want, mag, np.float32,
                         what="streams that outlast their lane")
  # the same streams as columns (homogeneous ones of that length are walked by waves): their wave finishes them
  kw.update(n_row=n_in, n_col=n_out, col_walk=True, w_b=1.0)
  ones = np.ones(n_out, np.float32)
  want = oracle_mod.jitconn_matvec(ones, dense=True, **kw)
  oracle_mod.set_threads(1)
  assert np.array_equal(kernel_call(ones, dense=True, **kw), want)


@pytest.mark.parametrize("n_out,mean,dtype,most", [(1_000_000, 92.0, np.float32, 139), (1_000_000, 38.0, np.float64, 60)])
def test_row_walk_of_normal_weights_that_go_on_behind_the_first_words(cuda, oracle_mod, n_out, mean, dtype, most):
  # A synapse takes 3.27 words, in double 4.55: the streams go on behind word 227, where words are made of new words, and of those of
  # 92 a few need more than the 454 that a lane can draw (139 synapses and more): their wave walks them.
  n_in, p = 3000, mean / 3000
  assert jitconn_by_lane("normal", np.dtype(dtype).itemsize, n_out, n_in, p, event_bytes=1)
  assert jitconn_by_lane("normal", np.dtype(dtype).itemsize, n_out, n_in, p)
  rng = np.random.default_rng(n_out)
  oracle_mod.set_threads(min(16, len(os.sched_getaffinity(0))))
  kw = dict(w_kind="normal", log_p=oracle_mod.log_p_of(p), seed=77, n_row=n_out, n_col=n_in, out_dtype=dtype)
  counts = oracle_mod.jitconn_matvec(np.ones(n_in, bool), dense=False, w_a=1.0, w_b=0.0, **kw)  # (every weight is 1)
  assert counts.max() >= most, counts.max()
  for inp, dense in ((rng.random(n_in) < 0.5, False), (rng.uniform(0.5, 2.0, n_in).astype(dtype), True)):
    want, mag = oracle_mod.jitconn_matvec(inp, dense=dense, return_abs=True, w_a=0.5, w_b=2.0, **kw)
    got = kernel_call(inp, col_walk=False, dense=dense, w_a=0.5, w_b=2.0, **kw)
    assert_close_reordered(got, want, mag, dtype, what="normal weights by lane")
  oracle_mod.set_threads(1)


@pytest.mark.parametrize("mean,dtype", [(80.0, np.float32), (30.0, np.float64)])
def test_column_walk_of_normal_weights_that_go_on_behind_the_first_words(cuda, oracle_mod, mean, dtype):
  n_in, n_out, p = 300_000, 20_000, mean / 20_000
  assert jitconn_by_lane("normal", np.dtype(dtype).itemsize, n_in, n_out, p, use=1)
  vec = np.random.default_rng(5).uniform(0.5, 2.0, n_in).astype(dtype)
  oracle_mod.set_threads(min(16, len(os.sched_getaffinity(0))))
  kw = dict(w_kind="normal", w_a=0.5, w_b=2.0, log_p=oracle_mod.log_p_of(p), seed=7, n_row=n_out, n_col=n_in, col_walk=True, dense=True)
  want, mag = oracle_mod.jitconn_matvec(vec, return_abs=True, **kw)
  oracle_mod.set_threads(1)
  assert_close_reordered(kernel_call(vec, **kw), want, mag, dtype, what="columns with normal weights by lane")


def test_column_walk_by_lane_in_several_launches(cuda, oracle_mod):
  # 4.8e8 synapses are more than the bins hold (3 GiB at 6 bytes and a quarter to spare): the columns are walked in two launches by
  # lane, with the bins emptied in between.  Whole numbers: every order of the additions gives the same sums.
  n_in, n_out, p = 8_000_000, 5000, 60.0 / 5000
  assert jitconn_by_lane("homo", 4, n_in, n_out, p, use=1) and n_in * 60.0 * 1.25 * 6 > 3 << 30
  rng = np.random.default_rng(8)
  vec = np.zeros(n_in, np.float32)
  on = rng.choice(n_in, 40_000, replace=False)
  vec[on] = rng.integers(1, 4, on.shape[0])
  kw = dict(log_p=oracle_mod.log_p_of(p), n_row=n_out)
  got = kernel_call(vec, w_kind="homo", seed=3, n_col=n_in, col_walk=True, dense=True, **kw)
  want = np.zeros(n_out)
  for c in on:
    idx, _ = oracle_mod.jitconn_stream_weights(3 + int(c), "homo", 0.0, 0.0, kw["log_p"], n_out, dtype=np.float32)
    want[idx] += vec[c]
  assert np.array_equal(got, want)


@pytest.mark.parametrize("w_kind,mean", [("homo", 15.0), ("uniform", 12.0), ("normal", 11.0)])
@pytest.mark.parametrize("rate", [0.004, 0.1, 0.6])
def test_column_walk_of_events_by_lane_into_bins(cuda, oracle_mod, w_kind, mean, rate):
  # a million columns have more than 1e7 synapses: bins, sized for an eighth of the columns (0.6: what finds them full goes to the
  # output directly).  Normal weights of that length go by wave.
  n_in, n_out, p = 1_000_000, 6007, mean / 6007
  assert jitconn_by_lane(w_kind, 4, n_in, n_out, p, use=2) == (w_kind != "normal") and n_in * mean > 1e7
  ev = np.random.default_rng(int(mean)).random(n_in) < rate
  oracle_mod.set_threads(min(16, len(os.sched_getaffinity(0))))
  kw = dict(w_kind=w_kind, w_a=0.25, w_b=1.75, log_p=oracle_mod.log_p_of(p), seed=7, n_row=n_out, n_col=n_in, col_walk=True, dense=False)
  want, mag = oracle_mod.jitconn_matvec(ev, return_abs=True, **kw)
  oracle_mod.set_threads(1)
  got = kernel_call(ev, **kw)
  if w_kind == "homo":
    assert np.array_equal(got, want)
  else:
    assert_close_reordered(got, want, mag, np.float32, what="event columns by lane into bins")


def test_matmat_of_more_tiles_than_a_launch_has_threads_for(cuda, oracle_mod):
  # X of 2,200 x 8,000,000 is transposed in 1.8e7 tiles of 32 x 32, 256 threads each: more than 2^32 (4e6 workgroups take them
  # in turn).  70 GB and their transpose, which is the scratch memory of a stream of its own.
  m, k, n, seed = 2_200, 8_000_000, 8, 5
  if torch.cuda.mem_get_info()[0] < 170 << 30:
    pytest.skip("150 GB of device memory are needed")
  handle = ctypes.c_void_p()
  hip = ctypes.CDLL("libamdhip64.so")
  assert hip.hipStreamCreate(ctypes.byref(handle)) == 0
  lp = oracle_mod.log_p_of(1e-5)
  X = torch.empty((m, k), device=cuda)
  for i in range(0, m, 50):
    X[i:i + 50].uniform_(0.5, 2.0)
  torch.cuda.synchronize()
  with torch.cuda.stream(torch.cuda.ExternalStream(handle.value)):
    got = bpl.matmat_prob_conn_uniform_weight(X, w_low=0.5, w_high=1.5, conn_prob=1e-5, shape=(k, n), seed=seed)
  torch.cuda.synchronize()
  for j in range(n):
    idx, w = oracle_mod.jitconn_stream_weights(seed + j, "uniform", 0.5, 1.5, lp, k, dtype=np.float32)
    assert idx.shape[0] > 20
    want = X[:, torch.from_numpy(idx.astype(np.int64)).to(cuda)].double() @ torch.from_numpy(w.astype(np.float64)).to(cuda)
    # (some 80 addends of one sign, added in float32 one after the other)
    torch.testing.assert_close(got[:, j].double(), want, rtol=idx.shape[0] * 2.0 ** -23, atol=0.0)
  del X, got, want
  torch.cuda.empty_cache()


@pytest.mark.parametrize("m,k,columns", [(3, 31, 0), (64, 33, 1), (65, 500, 63), (130, 64, 64), (9, 900, 65)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_matmat_from_one_workgroup_for_every_cu_on(cuda, oracle_mod, m, k, columns, dtype):
  # with more than four columns for every CU their generators are seeded beside the transposition of X, 64 to a wave
  # (up to there by the waves that walk them); tiles of 32 inputs and 64 rows of X, the last ones partly filled
  n = 4 * torch.cuda.get_device_properties(0).multi_processor_count + columns
  X = np.random.default_rng(k).standard_normal((m, k)).astype(dtype)
  want = oracle_mod.jitconn_matmat(X, w_kind="uniform", w_a=-0.5, w_b=1.5, log_p=oracle_mod.log_p_of(0.2), seed=3, n=n)
  got = bpl.matmat_prob_conn_uniform_weight(X, w_low=-0.5, w_high=1.5, conn_prob=0.2, shape=(k, n), seed=3).cpu().numpy()
  assert got.shape == (m, n) and np.array_equal(got, want)  # the same operations in the same order


def test_config_jitconn_matmat_full_size(cuda, oracle_mod):
  # 10,000 x 10,000 implicit matrix, conn_prob 0.1, N(0, 0.01^2) from seed 7, times B[10000, 128]:
  # out = (B^T @ M)^T in the reference's orientation (X = B^T, m = 128).
  c = synth.config_jitconn_matmat()
  X = np.ascontiguousarray(c["B"].T)
  oracle_mod.set_threads(min(16, len(os.sched_getaffinity(0))))
  lp = oracle_mod.log_p_of(c["conn_prob"])
  # the oracle on all 128 rows (every stream generated once and applied to every row of X), with
  # sum(|w x|) per output: the reordering term of the tolerance is computed, not estimated
  want, mag = oracle_mod.jitconn_matmat(X, w_kind="normal", w_a=c["w_mu"], w_b=c["w_sigma"], log_p=lp, seed=c["seed"],
                                        n=c["shape"][1], return_abs=True)
  # the definition itself (one matvec per row of X) on two rows
  rows = np.array([0, 127])
  by_rows = oracle_mod.jitconn_matmat(X[rows], w_kind="normal", w_a=c["w_mu"], w_b=c["w_sigma"], log_p=lp,
                                      seed=c["seed"], n=c["shape"][1], by_rows=True)
  oracle_mod.set_threads(1)
  assert np.array_equal(by_rows, want[rows])
  got = bpl.matmat_prob_conn_normal_weight(X, w_mu=c["w_mu"], w_sigma=c["w_sigma"], conn_prob=c["conn_prob"],
                                           shape=c["shape"], seed=c["seed"]).cpu().numpy()
  assert got.shape == (128, 10000)
  # the kernel adds in the oracle's order; what differs is the device's logf / sqrtf in the normal
  # weights (within 4 ulp each): 4 eps sum(|w x|) covers that too
  outside = assert_close_reordered(got, want, mag, np.float32, what="matmat 10,000 x 10,000 x 128")
  print("matmat full size: %d of %d outside plain rel 1e-5 / abs 1e-6; max abs err %.3e"
        % (outside, got.size, float(np.abs(got - want).max())), flush=True)


@pytest.mark.parametrize("w_kind,a,b", [("homo", 0.0, 0.0), ("uniform", 0.25, 1.75), ("normal", 0.5, 2.0)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_column_walk_through_bins_dense(cuda, oracle_mod, w_kind, a, b, dtype):
  # dense input, output wider than one 16,384-element window, > 2^20 pairs: the column walk appends
  # its pairs to bins that a second kernel adds.  Against the oracle's column walk (integer input:
  # homogeneous sums are exact) and against the row walk of the transposed flags (adjoint).
  n_out, n_in = 40_000, 2_500
  lp = oracle_mod.log_p_of(0.05)
  rng = np.random.default_rng(8)
  x = rng.integers(-3, 4, n_in).astype(dtype)
  got = kernel_call(x, w_kind=w_kind, w_a=a, w_b=b, log_p=lp, seed=21, n_row=n_out, n_col=n_in, col_walk=True,
                    dense=True)
  want, mag = oracle_mod.jitconn_matvec(x, w_kind=w_kind, w_a=a, w_b=b, log_p=lp, seed=21, n_row=n_out, n_col=n_in,
                                        col_walk=True, dense=True, return_abs=True)
  if w_kind == "homo":
    assert np.array_equal(got, want)
  else:
    assert_close_reordered(got, want, mag, dtype, what="binned column walk %s" % w_kind)
  y = rng.integers(-3, 4, n_out).astype(np.float64)
  x64 = x.astype(np.float64)
  Mx = kernel_call(x64, w_kind=w_kind, w_a=a, w_b=b, log_p=lp, seed=21, n_row=n_out, n_col=n_in, col_walk=True, dense=True)
  MTy = kernel_call(y, w_kind=w_kind, w_a=a, w_b=b, log_p=lp, seed=21, n_row=n_in, n_col=n_out, col_walk=False, dense=True)
  assert abs(y @ Mx - MTy @ x64) <= 1e-9 * max(1.0, abs(y @ Mx))


@pytest.mark.parametrize("w_kind,a,b", [("homo", 0.0, 0.0), ("uniform", 0.25, 1.75)])
@pytest.mark.parametrize("n_out,n_in,p,dtype", [(3_000_000, 300, 0.0015, np.float32), (3_000_000, 300, 0.0015, np.float64),
                                                (9_000_000, 100, 0.0015, np.float32)])
def test_column_walk_through_bins_wide_windows(cuda, oracle_mod, w_kind, a, b, n_out, n_in, p, dtype):
  # outputs of more than two million elements: the windows grow beyond the 16,384 accumulators a workgroup
  # holds at once (3,000,000: windows of 32,768 outputs added in two slices, pairs still packed with 16-bit
  # positions; 9,000,000: windows of 131,072 outputs in eight slices, whole pairs).  Integer input: the
  # homogeneous sums are exact.
  lp = oracle_mod.log_p_of(p)
  rng = np.random.default_rng(n_out % 1000)
  x = rng.integers(-3, 4, n_in).astype(dtype)
  x[x == 0] = 1
  got = kernel_call(x, w_kind=w_kind, w_a=a, w_b=b, log_p=lp, seed=5, n_row=n_out, n_col=n_in, col_walk=True, dense=True)
  want, mag = oracle_mod.jitconn_matvec(x, w_kind=w_kind, w_a=a, w_b=b, log_p=lp, seed=5, n_row=n_out, n_col=n_in,
                                        col_walk=True, dense=True, return_abs=True)
  assert mag.sum() > 1_048_576  # (enough pairs for the bins)
  if w_kind == "homo":
    assert np.array_equal(got, want)
  else:
    assert_close_reordered(got, want, mag, dtype, what="binned column walk, wide windows")


@pytest.mark.parametrize("w_kind,a,b", [("homo", 0.0, 0.0), ("normal", 0.5, 2.0)])
@pytest.mark.parametrize("n_out,n_in,p", [(4000, 4000, 0.02), (700, 90, 0.3), (5, 3, 0.9), (30_000, 2047, 0.01),
                                          (2 ** 24 + 5, 7, 2e-6), (2 ** 24 + 5, 140_000, 4e-7)])
def test_column_walk_dense_with_few_pairs(cuda, oracle_mod, w_kind, a, b, n_out, n_in, p):
  # dense input and fewer than 2^20 possible pairs: every column's generator is seeded ahead and the walk adds
  # its pairs to the output with atomics (no bins).  Against the oracle's column walk; integer input, so the
  # homogeneous sums are exact.  And a bound on the time: with every lane seeding its own column's generator
  # the first shape took 0.5 ms.
  lp = oracle_mod.log_p_of(p)
  x = np.random.default_rng(n_in).integers(-3, 4, n_in).astype(np.float32)
  kw = dict(w_kind=w_kind, w_a=a, w_b=b, log_p=lp, seed=33, n_row=n_out, n_col=n_in, col_walk=True, dense=True)
  got = kernel_call(x, **kw)
  want, mag = oracle_mod.jitconn_matvec(x, return_abs=True, **kw)
  if w_kind == "homo":
    assert np.array_equal(got, want)
  else:
    assert_close_reordered(got, want, mag, np.float32, what="dense column walk with few pairs")
  if n_out == 4000 and w_kind == "homo":
    xd = torch.from_numpy(x).cuda()
    call = lambda: bpl.matvec_prob_conn_homo_weight(xd, 0.5, conn_prob=p, shape=(n_out, n_in), seed=33, outdim_parallel=False)
    call()
    torch.cuda.synchronize()
    # best of five groups of five calls (a shared box or low clocks slow single groups down): about 70 us when the
    # generators are seeded ahead, 500 us when every lane seeds its own
    best = float("inf")
    for _ in range(5):
      e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
      e0.record()
      for _ in range(5):
        call()
      e1.record()
      torch.cuda.synchronize()
      best = min(best, e0.elapsed_time(e1) * 1e3 / 5)
    print("dense column walk 4,000 x 4,000: %.1f us per call (best of 5 groups)" % best, flush=True)
    assert best < 300.0


def test_column_walk_through_bins_sliced_windows(cuda, oracle_mod):
  # more than 2^21 outputs: the bins' windows are wider than their accumulators in LDS and are
  # added in slices
  n_out, n_in = 3_000_001, 1_500
  lp = oracle_mod.log_p_of(0.0004)
  rng = np.random.default_rng(9)
  x = rng.integers(-3, 4, n_in).astype(np.float32)
  for w_kind, a, b in (("homo", 0.0, 0.0), ("uniform", 0.25, 1.75)):
    got = kernel_call(x, w_kind=w_kind, w_a=a, w_b=b, log_p=lp, seed=5, n_row=n_out, n_col=n_in, col_walk=True, dense=True)
    want, mag = oracle_mod.jitconn_matvec(x, w_kind=w_kind, w_a=a, w_b=b, log_p=lp, seed=5, n_row=n_out, n_col=n_in,
                                          col_walk=True, dense=True, return_abs=True)
    if w_kind == "homo":
      assert np.array_equal(got, want)
    else:
      assert_close_reordered(got, want, mag, np.float32, what="sliced binned column walk")


def test_column_walk_through_bins_events_and_overflow(cuda, oracle_mod):
  # event input with n_in * n_out * p >= 5e7: bins sized for one active column in eight.  At 2 % activity
  # everything fits; with every column active most pairs overflow into direct atomics.  Counts are exact.
  n_out, n_in = 60_000, 90_000
  lp = oracle_mod.log_p_of(0.01)
  rng = np.random.default_rng(9)
  for rate in (0.02, 1.0):
    ev = rng.random(n_in) < rate
    print("rate", rate, flush=True)
    got = kernel_call(ev, w_kind="homo", log_p=lp, seed=5, n_row=n_out, n_col=n_in, col_walk=True, dense=False)
    want = oracle_mod.jitconn_matvec(ev, w_kind="homo", log_p=lp, seed=5, n_row=n_out, n_col=n_in, col_walk=True)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("w_kind,a,b", [("homo", 0.0, 0.0), ("uniform", 0.25, 1.75), ("normal", 0.1, 1.0)])
@pytest.mark.parametrize("active", [1, 16, 512 * 16, 512 * 17 + 1, 512 * 63, 512 * 64, 512 * 64 + 1])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_column_walk_last_batch_of_streams(cuda, oracle_mod, w_kind, a, b, active, dtype):
  # a workgroup seeds 64 streams at a time, and a batch of fewer stores no state beyond its own: 1, 16, 17 and 63 to a
  # workgroup, one whole batch, one more.  Rows of about 400 over ten windows, each ending within a batch of synapses.
  n_out, n_in = 40_000, 40_000
  lp = oracle_mod.log_p_of(0.01)
  rng = np.random.default_rng(active)
  ev = np.zeros(n_in, dtype=bool)
  ev[rng.permutation(n_in)[:active]] = True
  kw = dict(w_kind=w_kind, w_a=a, w_b=b, log_p=lp, seed=41, n_row=n_out, n_col=n_in, col_walk=True, dense=False)
  for x in ([ev] if dtype == np.float32 else [ev.astype(np.float64)]):
    got = kernel_call(x, **kw)
    want, mag = oracle_mod.jitconn_matvec(x, return_abs=True, **kw)
    if w_kind == "homo":
      assert np.array_equal(got, want)
    else:
      assert_close_reordered(got, want, mag, dtype, what="column walk, last batch %s" % w_kind)


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_random_shapes_walks_weights_and_inputs_against_oracle(cuda, oracle_mod, seed):
  # shapes up to two million inputs / outputs, both walks, all weight kinds, bool / float events and
  # dense vectors drawn at random: every target of the family against the oracle
  rng = np.random.default_rng(seed)
  for case in range(100):
    n_out = int(10 ** rng.uniform(0, 4.0))
    n_in = int(10 ** rng.uniform(0, 6.3))
    col_walk = bool(rng.random() < 0.5)
    if col_walk:
      n_out, n_in = int(10 ** rng.uniform(0, 6.3)), int(10 ** rng.uniform(0, 3.7))
    syn = 10 ** rng.uniform(0, 2.5)
    p = min(1.0, syn / max(n_out if col_walk else n_in, 1))
    lp = oracle_mod.log_p_of(p)
    w_kind = str(rng.choice(["homo", "uniform", "normal"]))
    a, b = (0.0, 0.0) if w_kind == "homo" else (0.25, 1.75)
    dtype = np.float32 if rng.random() < 0.7 else np.float64
    kind = str(rng.choice(["bool", "float", "dense"]))
    if kind == "bool":
      inp, dense = rng.random(n_in) < rng.choice([0.0, 0.02, 0.5, 1.0]), False
    elif kind == "float":
      inp, dense = ((rng.random(n_in) < 0.3) * rng.uniform(0.5, 2, n_in)).astype(dtype), False
    else:
      inp, dense = rng.integers(-3, 4, n_in).astype(dtype), True
    stream_seed = int(rng.integers(0, 2 ** 31))
    print("case", case, n_out, n_in, col_walk, "%.2e" % p, w_kind, kind, dtype.__name__, flush=True)
    want, mag = oracle_mod.jitconn_matvec(inp, w_kind=w_kind, w_a=a, w_b=b, log_p=lp, seed=stream_seed, n_row=n_out,
                                          n_col=n_in, col_walk=col_walk, dense=(None if kind == "bool" else dense),
                                          return_abs=True)
    got = kernel_call(inp, w_kind=w_kind, w_a=a, w_b=b, log_p=lp, seed=stream_seed, n_row=n_out, n_col=n_in,
                      col_walk=col_walk, dense=dense)
    if w_kind == "homo":
      assert np.array_equal(got, want)  # counts / sums of small integers
    else:
      assert_close_reordered(got, want, mag, np.float32 if kind == "bool" else dtype, what="case %d" % case)



@pytest.mark.parametrize("w_kind,a,b", [("homo", 0.0, 0.0), ("uniform", 0.25, 1.75), ("normal", 0.5, 2.0)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_first_generation_dense_targets_give_the_cpu_paths_matrix(cuda, oracle_mod, w_kind, a, b, dtype):
  # gpu_matvec_prob_*_v1_*: the descriptor carries conn_prob itself; on the reference's CPU path the
  # version does not change the result (matvec.py:296-308), so the oracle is the same row walk.
  n_row, n_col, seed = 70, 3000, 21
  rng = np.random.default_rng(3)
  tn = "_float" if dtype == np.float32 else "_double"
  np_dt = dtype
  for p, vec in ((0.07, rng.integers(-3, 4, n_col).astype(dtype)), (0.5, np.arange(n_col).astype(dtype)),
                 (1.0, np.ones(n_col, dtype=dtype))):
    lp = oracle_mod.log_p_of(p)
    want = oracle_mod.jitconn_matvec(vec, w_kind=w_kind, w_a=a, w_b=b, log_p=lp, seed=seed, n_row=n_row, n_col=n_col,
                                     dense=True, per_stream_seed=True)
    if w_kind == "homo":
      opaque = _lib.build_jitconn_prob_homo_descriptor(n_row, n_col, seed, p)
    elif w_kind == "uniform":
      opaque = _lib.build_jitconn_prob_uniform_descriptor(n_row, n_col, seed, p, float(np_dt(a)),
                                                          float(np_dt(np_dt(b) - np_dt(a))))
    else:
      opaque = _lib.build_jitconn_prob_normal_descriptor(n_row, n_col, seed, p, a, b)
    t = torch.from_numpy(vec).to("cuda:0")
    out = torch.full((n_row,), 123.0, dtype=t.dtype, device="cuda:0")
    _lib.custom_call("gpu_matvec_prob_" + w_kind + "_v1" + tn, [t, out], opaque)
    got = out.cpu().numpy()
    v2 = kernel_call(vec, w_kind=w_kind, w_a=a, w_b=b, log_p=lp, seed=seed, n_row=n_row, n_col=n_col, col_walk=False,
                     dense=True)
    assert np.array_equal(got, v2), (w_kind, p)  # one kernel behind both names
    if w_kind == "homo":
      assert np.array_equal(got.astype(np.float64), want.astype(np.float64)), p  # integer data: exact sums
      if p >= 1.0:
        assert np.all(got == n_col - 1)  # closed form: every index from 1 on
    else:
      meta = dict(dense=True, conn_prob=p, col_walk=False, n_row=n_row, n_col=n_col, seed=seed, w_kind=w_kind,
                  w_a=a, w_b=b)
      assert_close_reordered(got, want, _abs_bound(oracle_mod, vec, meta, dtype), dtype, what="v1 " + w_kind)


def test_version_argument_of_the_dense_wrappers(cuda):
  rng = np.random.default_rng(8)
  shape = (200, 300)
  kw = dict(conn_prob=0.1, shape=shape, seed=77)
  for transpose in (False, True):
    v = rng.standard_normal(shape[0] if transpose else shape[1]).astype(np.float32)
    calls = ((bpl.matvec_prob_conn_homo_weight, (v, 0.3), {}),
             (bpl.matvec_prob_conn_uniform_weight, (v,), dict(w_low=-1.0, w_high=2.0)),
             (bpl.matvec_prob_conn_normal_weight, (v,), dict(w_mu=0.1, w_sigma=0.5)))
    for fn, args, extra in calls:
      y1 = fn(*args, transpose=transpose, version='v1', **extra, **kw)
      y2 = fn(*args, transpose=transpose, version='v2', **extra, **kw)
      assert torch.equal(y1, y2), fn.__name__
      with pytest.raises(_lib.GPUOperatorNotFound):  # the reference registers no atomic v1 target either
        fn(*args, transpose=transpose, outdim_parallel=False, version='v1', **extra, **kw)
      with pytest.raises(AssertionError):
        fn(*args, transpose=transpose, version='v3', **extra, **kw)
  # the raw probability is validated where it is converted
  t = torch.zeros(10, dtype=torch.float32, device="cuda:0")
  out = torch.zeros(10, dtype=torch.float32, device="cuda:0")
  with pytest.raises(RuntimeError):
    _lib.custom_call("gpu_matvec_prob_homo_v1_float", [t, out], _lib.build_jitconn_prob_homo_descriptor(10, 10, 1, -0.5))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n_syn", [1, 2, 3, 22, 79, 80, 81, 82, 127, 128, 129, 130, 159, 160, 161, 255, 256, 257, 1000])
def test_normal_weights_worked_off_in_groups(cuda, oracle_mod, n_syn, dtype):
  # A wave works the weights of 128 synapses (80 in double) off at a time.  With conn_prob 1 a stream holds
  # every index once: streams that end just before, at and behind the end of a group, in every operator.
  rng = np.random.default_rng(n_syn)
  lp, m = oracle_mod.log_p_of(1.0), 37
  vec = rng.uniform(0.5, 2.0, n_syn).astype(dtype)
  ev = (rng.random(n_syn) < 0.3) | (np.arange(n_syn) == n_syn - 1)
  kw = dict(w_kind="normal", w_a=0.5, w_b=2.0, log_p=lp, seed=11)
  print("case", n_syn, dtype.__name__, flush=True)
  for inp, dense in ((vec, True), (ev, False)):
    want, mag = oracle_mod.jitconn_matvec(inp, n_row=m, n_col=n_syn, dense=dense, return_abs=True, out_dtype=dtype, **kw)
    got = kernel_call(inp, n_row=m, n_col=n_syn, col_walk=False, dense=dense, out_dtype=dtype, **kw)
    assert_close_reordered(got, want, mag, dtype, what="normal weights, row walk")
  x = rng.uniform(0.5, 2.0, m).astype(dtype)
  want, mag = oracle_mod.jitconn_matvec(x, n_row=n_syn, n_col=m, col_walk=True, dense=True, return_abs=True, **kw)
  got = kernel_call(x, n_row=n_syn, n_col=m, col_walk=True, dense=True, **kw)
  assert_close_reordered(got, want, mag, dtype, what="normal weights, column walk")
  X = rng.uniform(0.5, 2.0, (70, n_syn)).astype(dtype)
  want, mag = oracle_mod.jitconn_matmat(X, n=m, return_abs=True, **kw)
  got = bpl.matmat_prob_conn_normal_weight(torch.from_numpy(X).cuda(), w_mu=0.5, w_sigma=2.0, conn_prob=1.0,
                                           shape=(n_syn, m), seed=11).cpu().numpy()
  assert_close_reordered(got, want, mag, dtype, what="normal weights, matmat")


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n_in", [90_112, 90_113, 151_552, 151_553, 311_296, 311_297])
@pytest.mark.parametrize("p", [0.003, 0.0002, 0.00005])
def test_normal_weights_on_both_sides_of_the_bitmaps_and_skip_paths(cuda, oracle_mod, p, n_in, dtype):
  # bitmaps exact in LDS, up to the last one and the first in two levels (for more rows than here they begin at 151,552 inputs,
  # double 90,112: test_row_walk_on_both_sides_of_the_exact_bitmaps), and
  # conn_probs whose skips are tried on the upper word alone, on both words, and in 13 bits of fraction less
  rng = np.random.default_rng(n_in)
  ev = rng.random(n_in) < 0.2
  kw = dict(w_kind="normal", w_a=0.5, w_b=2.0, log_p=oracle_mod.log_p_of(p), seed=5, n_row=301, n_col=n_in)
  print("case", p, n_in, dtype.__name__, flush=True)
  want, mag = oracle_mod.jitconn_matvec(ev, dense=False, return_abs=True, out_dtype=dtype, **kw)
  assert_close_reordered(kernel_call(ev, col_walk=False, dense=False, out_dtype=dtype, **kw), want, mag, dtype,
                         what="normal weights, events")


@pytest.mark.parametrize("mean", [70.0, 240.0])
@pytest.mark.parametrize("w_kind,dtype,last", [("homo", np.float32, 268_288), ("uniform", np.float32, 235_520),
                                               ("uniform", np.float64, 219_136), ("normal", np.float32, 151_552),
                                               ("normal", np.float64, 90_112)])
def test_row_walk_on_both_sides_of_the_exact_bitmaps(cuda, oracle_mod, w_kind, dtype, last, mean):
  # (rows of 240 synapses are walked by waves, most of those of 70 by lanes, which have no bitmaps)
  # (outputs, inputs): exact bitmaps of up to 311,296 inputs where one workgroup a CU has all rows; two workgroups of
  # fewer waves; two turns of one; two 16-wave workgroups, up to `last` inputs (16,384 outputs: one)
  place = {"homo": 311_296, "uniform": 311_296, "normal": 151_552 if dtype == np.float32 else 153_600}[w_kind]
  rng = np.random.default_rng(last)
  for n_out, n_in in ((301, 311_296), (301, 311_297), (4_101, place), (4_101, place + 1), (6_000, place), (8_191, place),
                      (16_384, 311_296), (16_385, last), (16_385, last + 1)):
    ev = rng.random(n_in) < 0.2
    kw = dict(w_kind=w_kind, w_a=0.5, w_b=2.0, log_p=oracle_mod.log_p_of(mean / n_in), seed=9, n_row=n_out, n_col=n_in)
    print("case", n_out, n_in, flush=True)
    assert mean < 240 or not jitconn_by_lane(w_kind, np.dtype(dtype).itemsize, n_out, n_in, mean / n_in, event_bytes=1)
    want, mag = oracle_mod.jitconn_matvec(ev, dense=False, return_abs=True, out_dtype=dtype, **kw)
    got = kernel_call(ev, col_walk=False, dense=False, out_dtype=dtype, **kw)
    if w_kind == "homo":
      assert np.array_equal(got, want)
    else:
      assert_close_reordered(got, want, mag, dtype, what="row walk, %s weights" % w_kind)


def _stream_that_skips_to_the_end_of_the_integers(w_kind, n_in):
  """(seed, log_p, the index that the second skip would lead to from 2^32 - 16 on, counted around): the first skip of the
  stream is 2^32 - 16, the second one so short that a walk that went on would find an input."""
  for seed in range(200_000):
    words = np.random.RandomState(seed).randint(0, 1 << 32, 64, dtype=np.uint64).astype(np.float64)
    log_u = lambda i: np.log((words[i] + words[i + 1] * 2.0 ** 32) * 2.0 ** -64)
    at = {"homo": 2, "uniform": 3, "normal": 2}[w_kind]
    if w_kind == "normal":
      while (2 * words[at] * 2.0 ** -32 - 1) ** 2 + (2 * words[at + 1] * 2.0 ** -32 - 1) ** 2 > 1:
        at += 2
      at += 2
    log_p = log_u(0) / (2.0 ** 32 - 16.5)
    second = np.ceil(log_u(at) / log_p)
    if np.ceil(log_u(0) / log_p) == 2.0 ** 32 - 16 and 100 < second < n_in - 100:
      return seed, log_p, int(second) - 16
  raise AssertionError("no such stream")


@pytest.mark.parametrize("w_kind", KINDS_BUILT)
@pytest.mark.parametrize("dtype", [np.bool_, np.float32])
def test_a_skip_to_just_below_two_to_the_32_ends_the_row(cuda, oracle_mod, w_kind, dtype):
  n_in = 400_000  # (a two-level bitmap, whose positions begin at 32)
  seed, log_p, index = _stream_that_skips_to_the_end_of_the_integers(w_kind, n_in)
  ev = np.zeros(n_in, dtype)
  ev[index] = 1
  kw = dict(w_kind=w_kind, w_a=0.5, w_b=2.0, log_p=log_p, seed=seed, n_row=1, n_col=n_in)
  assert oracle_mod.jitconn_matvec(ev, dense=False, **kw)[0] == 0
  assert kernel_call(ev, col_walk=False, dense=False, **kw)[0] == 0


@pytest.mark.parametrize("counter", [0, 1])
@pytest.mark.parametrize("polls", [0, 3])
@pytest.mark.parametrize("n_out,groups", [(64, 1), (1_000, 1), (8_200, 3), (9_001, 40)])
def test_waves_that_do_not_wait_for_their_generators_write_their_rows_all_the_same(cuda, n_out, groups, polls, counter):
  # one to many batches per workgroup; the counters are found as they were left, so each form runs twice
  import ctypes
  n_in, seed, log_p = 5_000, 11, float(np.log(1 - 0.02))
  ev = np.random.default_rng(n_out).random(n_in) < 0.3
  want = kernel_call(ev, w_kind="homo", log_p=log_p, seed=seed, n_row=n_out, n_col=n_in, col_walk=False, dense=False)
  events = torch.from_numpy(ev).cuda()
  check = _lib.lib().bpl_selfcheck_jitconn_rowwalk
  check.argtypes = [ctypes.c_void_p] * 3 + [ctypes.c_uint32] * 3 + [ctypes.c_double] + [ctypes.c_uint32] * 2 + [ctypes.c_int]
  print("case", n_out, groups, polls, counter, flush=True)
  for _ in range(2):
    out = torch.full((n_out,), -1.0, device="cuda")
    rc = check(torch.cuda.current_stream().cuda_stream, events.data_ptr(), out.data_ptr(), n_out, n_in, seed, log_p, polls,
               groups, counter)
    assert rc == 0, _lib.last_error()
    np.testing.assert_array_equal(out.cpu().numpy(), want)


@pytest.mark.parametrize("n_out,per_row", [(33_001, 30), (60_000, 100), (81_921, 250), (135_000, 20), (33_001, 240), (60_000, 240),
                                           (135_000, 240)])
def test_row_walk_whose_batches_are_shared_out_or_taken(cuda, oracle_mod, n_out, per_row):
  # two batches for some workgroups, seeded side by side and one after the other; taken from the counter from two and a
  # half (rows of 200 synapses and more) and from four batches a workgroup on.  Rows of 240 and 250 are walked by waves, the shorter
  # ones by lanes, but for 60,000 uniform ones of 100.
  n_in = 3000
  ev = np.random.default_rng(n_out).random(n_in) < 0.1
  kw = dict(log_p=oracle_mod.log_p_of(per_row / n_in), seed=5, n_row=n_out, n_col=n_in, w_a=0.25, w_b=1.75)
  print("case", n_out, per_row, flush=True)
  for w_kind in ("homo", "uniform"):
    assert per_row < 240 or not jitconn_by_lane(w_kind, 4, n_out, n_in, per_row / n_in, event_bytes=1)
    want, mag = oracle_mod.jitconn_matvec(ev, w_kind=w_kind, dense=False, per_stream_seed=True, return_abs=True, **kw)
    for _ in range(3):
      got = kernel_call(ev, w_kind=w_kind, col_walk=False, dense=False, **kw)
      if w_kind == "homo":
        assert np.array_equal(got, want)
      else:
        assert_close_reordered(got, want, mag, np.float32, what="row walk, batches shared out or taken")


@pytest.mark.parametrize("n_out,n_in", [(8192, 3000), (10_007, 200_000), (20_000, 400_000), (70_001, 5000)])
def test_row_walk_with_generators_seeded_inside_the_kernel(cuda, oracle_mod, n_out, n_in):
  # from 8,192 outputs the row walk seeds its generators itself, 64 streams at a time, into rings of
  # seeded states that its workgroups keep in device memory: whole outputs against the per-stream
  # oracle for every weight kind, event (LDS bitmap / two-level bitmap / packed float events) and
  # dense input, output counts that are and are not multiples of 64, fewer batches than workgroups,
  # twice in a row (the second call finds the rings of the first).
  rng = np.random.default_rng(n_out)
  lp = oracle_mod.log_p_of(200.0 / n_in)
  ev = rng.random(n_in) < 0.1
  fev = (ev * rng.uniform(0.5, 2.0, n_in)).astype(np.float32)
  vec = rng.integers(-3, 4, n_in).astype(np.float64)
  print("case", n_out, n_in, flush=True)
  for _ in range(2):
    for inp, dense in ((ev, False), (fev, False), (vec, True)):
      want = oracle_mod.jitconn_matvec(inp, log_p=lp, seed=5, n_row=n_out, n_col=n_in, dense=dense, per_stream_seed=True)
      got = kernel_call(inp, w_kind="homo", log_p=lp, seed=5, n_row=n_out, n_col=n_in, col_walk=False, dense=dense)
      assert want.any() and np.array_equal(got.astype(np.float64), want.astype(np.float64)), (inp.dtype, dense)
  for w_kind, a, b in (("uniform", 0.25, 1.75), ("normal", 0.5, 2.0)):
    for inp, dense, dt in ((ev, False, np.float32), (vec.astype(np.float32), True, np.float32), (vec, True, np.float64)):
      want, mag = oracle_mod.jitconn_matvec(inp, w_kind=w_kind, w_a=a, w_b=b, log_p=lp, seed=5, n_row=n_out, n_col=n_in,
                                            dense=dense, per_stream_seed=True, return_abs=True)
      got = kernel_call(inp, w_kind=w_kind, w_a=a, w_b=b, log_p=lp, seed=5, n_row=n_out, n_col=n_in, col_walk=False,
                        dense=dense)
      assert_close_reordered(got, want, mag, dt, what="fused row walk %s" % w_kind)
