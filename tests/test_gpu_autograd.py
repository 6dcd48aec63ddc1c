"""Differentiation rules of the operators (the reference's JVP / transpose rules,
event_csr_matvec.py:439-463, cusparse_matvec.py:281-308, jitconn event_matvec.py:242-273),
checked against torch's own autograd through the equivalent dense float64 product on the CPU."""
import numpy as np
import pytest
import torch
import torch.autograd.forward_ad as fwAD

import benchdata as synth
import brainpylib_amd as bpl
from util import random_csr

pytestmark = pytest.mark.gpu
SHAPES = [(60, 90), (90, 60), (200, 200)]


def _dense(data, indices, indptr, shape):
  """Differentiable dense float64 matrix on the CPU."""
  counts = np.diff(indptr)
  row = torch.from_numpy(np.repeat(np.arange(shape[0]), counts))
  col = torch.from_numpy(indices.astype(np.int64))
  vals = data if data.shape[0] > 1 else data.expand(col.shape[0])
  return torch.zeros(shape, dtype=torch.float64).index_put((row, col), vals, accumulate=True)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("homo", [False, True])
def test_event_csr_matvec_gradients(cuda, shape, transpose, homo):
  data_np, indices, indptr = random_csr(shape, 0.3, seed=shape[0] + 13, dtype=np.float64)
  if homo:
    data_np = np.array([0.8])
  rng = np.random.default_rng(2)
  n_in = shape[0] if transpose else shape[1]
  n_out = shape[1] if transpose else shape[0]
  ev_np = (rng.random(n_in) < 0.3) * rng.uniform(0.5, 2.0, n_in)
  ct_np = rng.standard_normal(n_out)
  # reference gradients: dense product with the events as a 0/1 vector for the weights ...
  d_ref = torch.tensor(data_np, requires_grad=True)
  M = _dense(d_ref, indices, indptr, shape)
  M = M.T if transpose else M
  (M @ torch.tensor((ev_np != 0).astype(np.float64)) @ torch.tensor(ct_np)).backward()
  # ... and the product that is linear in the events for the events (the rule's own definition)
  e_ref = torch.tensor(ev_np, requires_grad=True)
  (M.detach() @ e_ref @ torch.tensor(ct_np)).backward()

  data = torch.tensor(data_np, device="cuda", requires_grad=True)
  # weights: boolean events
  out = bpl.event_csr_matvec(data, indices, indptr, ev_np != 0, shape=shape, transpose=transpose)
  out.backward(torch.tensor(ct_np, device="cuda"))
  if homo:
    torch.testing.assert_close(data.grad.cpu(), d_ref.grad, rtol=1e-10, atol=1e-10)
  else:
    torch.testing.assert_close(data.grad.cpu(), d_ref.grad, rtol=1e-12, atol=1e-12)
  # events: float events carry a gradient
  events = torch.tensor(ev_np, device="cuda", requires_grad=True)
  out = bpl.event_csr_matvec(data.detach(), indices, indptr, events, shape=shape, transpose=transpose)
  out.backward(torch.tensor(ct_np, device="cuda"))
  torch.testing.assert_close(events.grad.cpu(), e_ref.grad, rtol=1e-10, atol=1e-10)
  # forward mode: tangents of weights and events together
  d_dot, e_dot = rng.standard_normal(data_np.shape), rng.standard_normal(n_in)
  with fwAD.dual_level():
    dd = fwAD.make_dual(data.detach(), torch.tensor(d_dot, device="cuda"))
    ee = fwAD.make_dual(events.detach(), torch.tensor(e_dot, device="cuda"))
    tangent = fwAD.unpack_dual(bpl.event_csr_matvec(dd, indices, indptr, ee, shape=shape, transpose=transpose)).tangent
  Md = _dense(torch.tensor(d_dot), indices, indptr, shape)
  Md = Md.T if transpose else Md
  want = Md @ torch.tensor((ev_np != 0).astype(np.float64)) + M.detach() @ torch.tensor(e_dot)
  torch.testing.assert_close(tangent.cpu(), want, rtol=1e-10, atol=1e-10)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("homo", [False, True])
def test_csr_matvec_gradients(cuda, shape, transpose, homo):
  data_np, indices, indptr = random_csr(shape, 0.3, seed=shape[0] + 17, dtype=np.float64, weights="uniform")
  if homo:
    data_np = np.array([0.8])
  rng = np.random.default_rng(3)
  n_in = shape[0] if transpose else shape[1]
  n_out = shape[1] if transpose else shape[0]
  v_np, ct_np = rng.standard_normal(n_in), rng.standard_normal(n_out)
  d_ref = torch.tensor(data_np, requires_grad=True)
  v_ref = torch.tensor(v_np, requires_grad=True)
  M = _dense(d_ref, indices, indptr, shape)
  M = M.T if transpose else M
  (M @ v_ref @ torch.tensor(ct_np)).backward()
  data = torch.tensor(data_np, device="cuda", requires_grad=True)
  vec = torch.tensor(v_np, device="cuda", requires_grad=True)
  out = bpl.cusparse_csr_matvec(data, indices, indptr, vec, shape=shape, transpose=transpose)
  out.backward(torch.tensor(ct_np, device="cuda"))
  torch.testing.assert_close(data.grad.cpu(), d_ref.grad, rtol=1e-10, atol=1e-10)
  torch.testing.assert_close(vec.grad.cpu(), v_ref.grad, rtol=1e-10, atol=1e-10)
  d_dot, v_dot = rng.standard_normal(data_np.shape), rng.standard_normal(n_in)
  with fwAD.dual_level():
    dd = fwAD.make_dual(data.detach(), torch.tensor(d_dot, device="cuda"))
    vv = fwAD.make_dual(vec.detach(), torch.tensor(v_dot, device="cuda"))
    tangent = fwAD.unpack_dual(bpl.cusparse_csr_matvec(dd, indices, indptr, vv, shape=shape, transpose=transpose)).tangent
  Md = _dense(torch.tensor(d_dot), indices, indptr, shape)
  Md = Md.T if transpose else Md
  want = Md @ torch.tensor(v_np) + M.detach() @ torch.tensor(v_dot)
  torch.testing.assert_close(tangent.cpu(), want, rtol=1e-10, atol=1e-10)


# rows, columns, mean row length: one partial step; rows shorter than a quad (windows of more than 64 rows to a step);
# vectors that fit the 139 to 151 KB staged in LDS, one element more than what fits (beside sums and products 36,608 floats
# or 17,792 doubles, beside products alone 38,656 or 18,816), the last staged size and one more (gathered from L2 only);
# rows that run through many waves' ranges
@pytest.mark.parametrize("n_row,n_col,mean", [(3, 9, 2), (9000, 200, 1), (300, 35_328, 900), (2000, 35_329, 300),
                                              (900, 17_664, 10), (20_000, 141_312, 40), (700, 141_313, 800),
                                              (10, 300_000, 20_000), (500, 36_609, 40), (500, 38_657, 40),
                                              (500, 17_793, 40), (500, 18_817, 40)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("transpose", [False, True])
def test_gradients_of_weights_and_vector_from_one_walk(cuda, n_row, n_col, mean, dtype, transpose):
  rng = np.random.default_rng(n_row)
  counts = np.minimum(rng.poisson(mean * np.exp(rng.standard_normal(n_row) - 0.5)), n_col)
  counts[rng.random(n_row) < 0.2] = 0
  counts[-1] = 0  # (rows without nonzeros, the last one among them)
  counts[0] = max(counts[0], 2)
  idx, ptr = synth.counted_csr(counts, n_col, seed=n_row)
  row = torch.from_numpy(np.repeat(np.arange(n_row), counts))
  col = torch.from_numpy(idx.astype(np.int64))
  print("case", n_row, n_col, dtype, transpose, idx.shape[0], flush=True)
  n_in, n_out = (n_row, n_col) if transpose else (n_col, n_row)
  g = torch.Generator().manual_seed(n_col)
  data, vec, ct = (torch.randn(n, dtype=dtype, generator=g) for n in (idx.shape[0], n_in, n_out))
  src, dst = (row, col) if transpose else (col, row)
  want = vec[src] * ct[dst]  # one product per weight: the same bits
  addend = (data * ct[dst]).to(torch.float64)  # the sums' addends, rounded once each as the kernels round them
  want_vec = torch.zeros(n_in, dtype=torch.float64).index_add_(0, src, addend)
  mag = torch.zeros(n_in, dtype=torch.float64).index_add_(0, src, addend.abs())
  # (second round: index and weight arrays that do not begin at a multiple of 16 bytes)
  for first in (0, 1):
    d = torch.cat([torch.zeros(first, dtype=dtype), data]).cuda()[first:].requires_grad_()
    i = torch.cat([torch.zeros(first, dtype=torch.int32), torch.from_numpy(idx)]).cuda()[first:]
    v = vec.cuda().requires_grad_()
    y = bpl.cusparse_csr_matvec(d, i, torch.from_numpy(ptr).cuda(), v, shape=(n_row, n_col), transpose=transpose)
    got, got_vec = torch.autograd.grad(y, (d, v), ct.cuda())
    assert torch.equal(got.cpu(), want)
    # transposed: the walk's float64 sums in another order, rounded once to dtype; else the transposed product, whose
    # partial sums are of dtype (the bound of two orders of summation in that precision)
    order = torch.float64 if transpose else dtype
    bound = torch.finfo(dtype).eps * want_vec.abs() + 4 * torch.finfo(order).eps * mag
    assert bool(((got_vec.cpu().to(torch.float64) - want_vec).abs() <= bound).all())
    # the weights' gradient alone (no sums), of float events; the events' values enter it
    y = bpl.event_csr_matvec(d, i, torch.from_numpy(ptr).cuda(), v.detach(), shape=(n_row, n_col), transpose=transpose)
    assert torch.equal(torch.autograd.grad(y, d, ct.cuda())[0].cpu(), want)


# infinities and NaN in the weights and in both vectors: they stay in the rows and products that they belong to, also where a
# neighbour shares a load of four nonzeros, a wave's range or the masked lanes of a step with them
@pytest.mark.parametrize("n_row,n_col,mean", [(40, 30, 3), (3000, 700, 2), (500, 40_000, 60), (6, 150_000, 9000)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_gradients_with_infinities_and_nan(cuda, n_row, n_col, mean, dtype):
  rng = np.random.default_rng(n_col)
  counts = np.minimum(rng.poisson(mean, n_row), n_col)
  idx, ptr = synth.counted_csr(counts, n_col, seed=n_row)
  row, col = np.repeat(np.arange(n_row), counts), idx.astype(np.int64)
  w, v, ct = (rng.standard_normal(n) for n in (idx.shape[0], n_row, n_col))
  for a in (w, v, ct):  # (column 0 and row 0 among them: masked lanes point there)
    a[rng.choice(a.shape[0], max(1, a.shape[0] // 50), replace=False)] = np.inf
    a[rng.choice(a.shape[0], max(1, a.shape[0] // 50), replace=False)] = np.nan
  ct[0], v[0] = np.nan, -np.inf
  w, v, ct = (torch.from_numpy(a).to(dtype) for a in (w, v, ct))
  d, t = w.cuda().requires_grad_(), v.cuda().requires_grad_()
  y = bpl.cusparse_csr_matvec(d, idx, ptr, t, shape=(n_row, n_col), transpose=True)
  got, sums = (g.cpu() for g in torch.autograd.grad(y, (d, t), ct.cuda()))
  assert torch.equal(torch.nan_to_num(got, 7.0), torch.nan_to_num(v[row] * ct[col], 7.0))
  assert torch.equal(got.isnan(), (v[row] * ct[col]).isnan())
  addend = (w * ct[col]).to(torch.float64)
  want = torch.zeros(n_row, dtype=torch.float64).index_add_(0, torch.from_numpy(row), addend)
  mag = torch.zeros(n_row, dtype=torch.float64).index_add_(0, torch.from_numpy(row), addend.abs())
  finite = want.isfinite()
  assert torch.equal(sums.isnan(), want.isnan()) and torch.equal(sums[want.isinf()].to(torch.float64), want[want.isinf()])
  # (float64 sums in another order, rounded once)
  bound = torch.finfo(dtype).eps * want.abs() + 4 * torch.finfo(torch.float64).eps * mag
  assert bool(((sums.to(torch.float64) - want).abs() <= bound)[finite].all()) and (bool(finite.any()) or mean > 1000)


# arrays longer than indptr says, by less than a quad and by more than the walk has threads; a matrix without nonzeros and
# one without rows.  Nothing depends on what lies beyond: its gradient is zero, whatever its columns are.
@pytest.mark.parametrize("n_row,mean,extra", [(50, 7, 3), (2000, 40, 300_000), (2000, 0, 1000), (0, 0, 5)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("product", ["cusparse_csr_matvec", "event_csr_matvec"])
def test_gradients_of_padded_index_arrays(cuda, n_row, mean, extra, dtype, transpose, product):
  n_col = 900
  rng = np.random.default_rng(extra)
  counts = np.minimum(rng.poisson(mean, n_row), n_col)
  idx, ptr = synth.counted_csr(counts, n_col, seed=extra) if n_row else (np.zeros(0, np.int32), np.zeros(1, np.int32))
  nnz = idx.shape[0]
  row, col = torch.from_numpy(np.repeat(np.arange(n_row), counts)), torch.from_numpy(idx.astype(np.int64))
  g = torch.Generator().manual_seed(n_row)
  data = torch.randn(nnz + extra, dtype=dtype, generator=g)
  n_in, n_out = (n_row, n_col) if transpose else (n_col, n_row)
  vec, ct = (torch.rand(n_in, generator=g) < 0.5).to(dtype), torch.randn(n_out, dtype=dtype, generator=g)
  src, dst = (row, col) if transpose else (col, row)
  d, v = data.cuda().requires_grad_(), vec.cuda().requires_grad_()
  idx = torch.cat([torch.from_numpy(idx), torch.full((extra,), n_col - 1, dtype=torch.int32)]).cuda()
  for wanted in ((d,), (d, v)):
    y = getattr(bpl, product)(d, idx, torch.from_numpy(ptr).cuda(), v, shape=(n_row, n_col), transpose=transpose)
    torch.full_like(d, float("nan"))  # (memory that an unwritten result would show)
    got = torch.autograd.grad(y, wanted, ct.cuda())
    assert torch.equal(got[0][:nnz].cpu(), vec[src] * ct[dst]) and not got[0][nnz:].any()
  want = torch.zeros(n_in, dtype=torch.float64).index_add_(0, src, (data[:nnz] * ct[dst]).to(torch.float64))
  mag = torch.zeros(n_in, dtype=torch.float64).index_add_(0, src, (data[:nnz] * ct[dst]).abs().to(torch.float64))
  # (two orders of summation in the result's precision)
  bound = torch.finfo(dtype).eps * want.abs() + 4 * torch.finfo(dtype).eps * mag
  assert bool(((got[1].cpu().to(torch.float64) - want).abs() <= bound).all())


@pytest.mark.parametrize("kind", ["homo", "uniform", "normal"])
@pytest.mark.parametrize("transpose", [False, True])
@pytest.mark.parametrize("outdim_parallel", [False, True])
def test_jitconn_matvec_gradients(cuda, oracle_mod, kind, transpose, outdim_parallel):
  # the implicit matrix, made explicit column by column with unit vectors through the oracle
  shape = (70, 50)
  kw = dict(conn_prob=0.2, shape=shape, seed=99, transpose=transpose, outdim_parallel=outdim_parallel)
  n_in = shape[0] if transpose else shape[1]
  n_out = shape[1] if transpose else shape[0]
  if kind == "homo":
    call = lambda v: bpl.matvec_prob_conn_homo_weight(v, 1.5, **kw)
  elif kind == "uniform":
    call = lambda v: bpl.matvec_prob_conn_uniform_weight(v, w_low=-1.0, w_high=2.0, **kw)
  else:
    call = lambda v: bpl.matvec_prob_conn_normal_weight(v, w_mu=0.5, w_sigma=2.0, **kw)
  eye = torch.eye(n_in, dtype=torch.float64, device="cuda")
  M = torch.stack([call(eye[i]) for i in range(n_in)], dim=1)  # (n_out, n_in)
  rng = np.random.default_rng(4)
  v = torch.tensor(rng.standard_normal(n_in), device="cuda", requires_grad=True)
  ct = torch.tensor(rng.standard_normal(n_out), device="cuda")
  out = call(v)
  torch.testing.assert_close(out.detach(), M @ v.detach(), rtol=1e-10, atol=1e-10)
  out.backward(ct)
  torch.testing.assert_close(v.grad, M.T @ ct, rtol=1e-10, atol=1e-10)
  v_dot = torch.tensor(rng.standard_normal(n_in), device="cuda")
  with fwAD.dual_level():
    tangent = fwAD.unpack_dual(call(fwAD.make_dual(v.detach(), v_dot))).tangent
  torch.testing.assert_close(tangent, M @ v_dot, rtol=1e-10, atol=1e-10)
  # event operator with float events: same matrix applied to the 0/1 vector; gradient as above
  if kind == "homo":
    ecall = lambda e: bpl.event_matvec_prob_conn_homo_weight(e, 1.5, **kw)
  elif kind == "uniform":
    ecall = lambda e: bpl.event_matvec_prob_conn_uniform_weight(e, w_low=-1.0, w_high=2.0, **kw)
  else:
    ecall = lambda e: bpl.event_matvec_prob_conn_normal_weight(e, w_mu=0.5, w_sigma=2.0, **kw)
  ev = torch.tensor((rng.random(n_in) < 0.3) * rng.uniform(0.5, 2.0, n_in), device="cuda", requires_grad=True)
  out = ecall(ev)
  torch.testing.assert_close(out.detach(), M @ (ev.detach() != 0).double(), rtol=1e-10, atol=1e-10)
  out.backward(ct)
  torch.testing.assert_close(ev.grad, M.T @ ct, rtol=1e-10, atol=1e-10)


def test_homogeneous_jitconn_weight_gradient(cuda):
  w = torch.tensor(0.7, device="cuda", requires_grad=True)
  ev = np.random.default_rng(5).random(300) < 0.2
  out = bpl.event_matvec_prob_conn_homo_weight(ev, w, conn_prob=0.1, shape=(200, 300), seed=3)
  out.sum().backward()
  counts = bpl.event_matvec_prob_conn_homo_weight(ev, 1.0, conn_prob=0.1, shape=(200, 300), seed=3)
  torch.testing.assert_close(w.grad, counts.sum())


def test_csr_coo_utilities(cuda):
  data, indices, indptr = random_csr((40, 30), 0.3, seed=5)
  row, col = bpl.csr_to_coo(indices, indptr)
  assert np.array_equal(row.numpy(), np.repeat(np.arange(40), np.diff(indptr)))
  assert np.array_equal(col.numpy(), indices)
  perm = np.random.default_rng(6).permutation(indices.shape[0])
  ix, ip = bpl.coo_to_csr(row.numpy()[perm], indices[perm], num_row=40)
  assert np.array_equal(ip.numpy(), indptr)
  for r in range(40):  # same entries per row, in the order the COO arrays listed them
    assert np.array_equal(ix.numpy()[ip[r]:ip[r + 1]], indices[perm][row.numpy()[perm] == r])
  dense = bpl.csr_to_dense(data, indices, indptr, shape=(40, 30)).numpy()
  want = np.zeros((40, 30), np.float32)
  want[row.numpy(), indices] = data
  assert np.array_equal(dense, want)
