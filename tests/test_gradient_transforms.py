"""Transforms over the backward pass of the CSR products (a batch of cotangents, forward over reverse, a second
derivative): the products behind the gradient of the weights have to stay visible to them.  The custom calls are
replaced by dense products, so that the rules themselves run on the CPU."""
import pytest
import torch
import torch.autograd.forward_ad as fwAD

from brainpylib_amd import event_ops, sparse_ops
from util import random_csr


def _dense(data, indices, indptr, shape):
  row, col = sparse_ops.csr_to_coo(indices, indptr)
  dense = torch.zeros(shape, dtype=data.dtype)
  return dense.index_put((row.long(), col.long()), data, accumulate=True)


@pytest.fixture(params=["csr", "event"])
def product(request, monkeypatch):
  def launch(data, indices, indptr, vector, shape, transpose, *_):
    dense = _dense(data, indices, indptr, shape)
    return (dense.T if transpose else dense) @ vector.to(data.dtype)
  monkeypatch.setattr(sparse_ops, "_launch", launch)
  monkeypatch.setattr(event_ops, "_launch", launch)
  if request.param == "csr":
    return lambda *a: sparse_ops._CSRMatvec.apply(*a, "vector")
  return event_ops._EventCSRMatvec.apply


def _problem(transpose):
  shape = (7, 11)
  _, idx, ptr = random_csr(shape, 0.4, 4)
  gen = torch.Generator().manual_seed(1)
  n_in, n_out = shape if transpose else shape[::-1]
  data, vec = (torch.randn(n, generator=gen, dtype=torch.float64) for n in (len(idx), n_in))
  vec = (vec > 0).to(torch.float64)
  ct = torch.randn((3, n_out), generator=gen, dtype=torch.float64)
  idx, ptr = torch.from_numpy(idx), torch.from_numpy(ptr)
  row, col = (t.long() for t in sparse_ops.csr_to_coo(idx, ptr))
  src, dst = (row, col) if transpose else (col, row)
  return shape, idx, ptr, data.requires_grad_(), vec, ct, vec[src] * ct[:, dst], src, dst


@pytest.mark.parametrize("transpose", [False, True])
def test_batch_of_cotangents(product, transpose):
  shape, idx, ptr, data, vec, ct, want, _, _ = _problem(transpose)
  out = product(data, idx, ptr, vec, shape, transpose)
  got, = torch.autograd.grad(out, data, ct, is_grads_batched=True)
  assert torch.equal(got, want)


@pytest.mark.parametrize("transpose", [False, True])
def test_tangent_of_the_cotangent(product, transpose):
  shape, idx, ptr, data, vec, ct, want, _, _ = _problem(transpose)
  out = product(data, idx, ptr, vec, shape, transpose)
  with fwAD.dual_level():
    got, = torch.autograd.grad(out, data, fwAD.make_dual(ct[0], ct[1]))
    primal, tangent = fwAD.unpack_dual(got)
  assert torch.equal(primal, want[0])
  assert tangent is not None and torch.equal(tangent, want[1])


@pytest.mark.parametrize("transpose", [False, True])
def test_derivative_by_the_cotangent(product, transpose):
  shape, idx, ptr, data, vec, ct, want, src, dst = _problem(transpose)
  ct = ct[0].clone().requires_grad_()
  out = product(data, idx, ptr, vec, shape, transpose)
  got, = torch.autograd.grad(out, data, ct, create_graph=True)
  assert torch.equal(got.detach(), want[0])
  second, = torch.autograd.grad(got.sum(), ct)
  torch.testing.assert_close(second, torch.zeros_like(second).index_add_(0, dst, vec[src]), rtol=1e-14, atol=1e-14)


@pytest.mark.parametrize("transpose", [False, True])
def test_padded_index_arrays(product, transpose, monkeypatch):
  # arrays longer than indptr says: the matrix ends where indptr ends, and what lies beyond has gradient zero
  shape, idx, ptr, data, vec, ct, want, _, _ = _problem(transpose)
  launch = sparse_ops._launch
  nnz, extra = idx.shape[0], 4
  monkeypatch.setattr(sparse_ops, "_launch", lambda d, i, *a: launch(d[:nnz], i[:nnz], *a))
  monkeypatch.setattr(event_ops, "_launch", lambda d, i, *a: launch(d[:nnz], i[:nnz], *a))
  data = torch.cat([data.detach(), torch.ones(extra, dtype=data.dtype)]).requires_grad_()
  idx = torch.cat([idx, torch.full((extra,), 2 ** 31 - 1, dtype=idx.dtype)])
  out = product(data, idx, ptr, vec, shape, transpose)
  got, = torch.autograd.grad(out, data, ct, is_grads_batched=True)
  assert torch.equal(got[:, :nnz], want) and not got[:, nnz:].any()
