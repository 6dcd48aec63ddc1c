"""Argument checking of the host-side operator wrappers (same conditions as the reference's
wrappers; no GPU needed: the checks run before a device is touched)."""
import ctypes
import inspect

import numpy as np
import pytest
import torch

import brainpylib_amd as bpl

IDX = np.zeros(6, dtype=np.int32)
PTR = np.zeros(5, dtype=np.int32)  # shape[0] = 4


def test_event_csr_matvec_checks():
  # brainpylib/_src/event_ops/event_csr_matvec.py:75-99
  ev4, ev7 = np.zeros(4, bool), np.zeros(7, bool)
  with pytest.raises(ValueError, match="size of data"):
    bpl.event_csr_matvec(np.zeros(3, np.float32), IDX, PTR, ev7, shape=(4, 7))
  with pytest.raises(ValueError, match="scalar or 1D"):
    bpl.event_csr_matvec(np.zeros((2, 3), np.float32), IDX, PTR, ev7, shape=(4, 7))
  with pytest.raises(ValueError, match="indices should be a 1D vector with int32 or uint32"):
    bpl.event_csr_matvec(1.0, IDX.astype(np.int64), PTR, ev7, shape=(4, 7))
  with pytest.raises(ValueError, match="indptr should be a 1D vector with int32 or uint32"):
    bpl.event_csr_matvec(1.0, IDX, PTR.astype(np.int64), ev7, shape=(4, 7))
  with pytest.raises(ValueError, match="events should be a 1D"):
    bpl.event_csr_matvec(1.0, IDX, PTR, np.zeros((7, 1), bool), shape=(4, 7))
  with pytest.raises(ValueError, match="length-2"):
    bpl.event_csr_matvec(1.0, IDX, PTR, ev7, shape=(4, 7, 1))
  with pytest.raises(ValueError, match=r"Shape mismatch, mat \(4, 7\) @ vec \(4,\)"):
    bpl.event_csr_matvec(1.0, IDX, PTR, ev4, shape=(4, 7))
  with pytest.raises(ValueError, match=r"Shape mismatch, vec \(7,\) @ mat \(4, 7\)"):
    bpl.event_csr_matvec(1.0, IDX, PTR, ev7, shape=(4, 7), transpose=True)
  with pytest.raises(ValueError, match="events should be bool or have the dtype of data"):
    bpl.event_csr_matvec(np.zeros(6, np.float32), IDX, PTR, np.zeros(7, np.float64), shape=(4, 7))


def test_csr_matvec_checks():
  # brainpylib/_src/sparse_ops/sparse_csr_matvec.py:70-82
  v = np.zeros(7, np.float32)
  with pytest.raises(ValueError, match="Only support methods"):
    bpl.csr_matvec(1.0, IDX, PTR, v, shape=(4, 7), method="fast")
  with pytest.raises(TypeError, match="Only support float32 and float64"):
    bpl.csr_matvec(np.zeros(6, np.int32), IDX, PTR, v, shape=(4, 7))
  with pytest.raises(TypeError, match="types of data and vector"):
    bpl.csr_matvec(np.zeros(6, np.float64), IDX, PTR, v, shape=(4, 7))
  with pytest.raises(ValueError, match="Shape mismatch"):
    bpl.csr_matvec(np.zeros(6, np.float32), IDX, PTR, np.zeros(4, np.float32), shape=(4, 7))


@pytest.mark.skipif(torch.cuda.is_available(), reason="checks the no-device error")
def test_no_cpu_fallback():
  with pytest.raises(RuntimeError, match="no CPU path"):
    bpl.event_csr_matvec(1.0, IDX, PTR, np.zeros(7, bool), shape=(4, 7))
  with pytest.raises(RuntimeError, match="no CPU path"):
    bpl.csr_matvec(1.0, IDX, PTR, np.zeros(7, np.float32), shape=(4, 7))


def test_check_csr_accepts_a_matrix_and_names_what_is_wrong_with_the_others():
  # the operators trust their index arrays as the reference's kernels do; this is the opt-in pass over them
  idx = np.array([0, 6, 2, 2, 5, 1], dtype=np.int32)
  ptr = np.array([0, 2, 2, 5, 6], dtype=np.int32)
  bpl.check_csr(idx, ptr, shape=(4, 7))
  bpl.check_csr(idx.astype(np.uint32), ptr.astype(np.uint32), shape=(4, 7))
  bpl.check_csr(np.zeros(0, np.int32), np.zeros(5, np.int32), shape=(4, 7))
  with pytest.raises(ValueError, match=r"indices should lie in \[0, 6\)"):
    bpl.check_csr(idx, ptr, shape=(4, 6))
  with pytest.raises(ValueError, match="indices should lie"):
    bpl.check_csr(np.array([0, -1, 2, 2, 5, 1], dtype=np.int32), ptr, shape=(4, 7))
  with pytest.raises(ValueError, match="indices should lie"):
    bpl.check_csr(np.array([0, 2 ** 31 + 3, 2, 2, 5, 1], dtype=np.uint32), ptr, shape=(4, 7))
  with pytest.raises(ValueError, match="never decrease"):
    bpl.check_csr(idx, np.array([0, 3, 2, 5, 6], dtype=np.int32), shape=(4, 7))
  with pytest.raises(ValueError, match="end at len"):
    bpl.check_csr(idx, np.array([0, 2, 2, 5, 7], dtype=np.int32), shape=(4, 7))
  with pytest.raises(ValueError, match="start at 0"):
    bpl.check_csr(idx, np.array([1, 2, 2, 5, 6], dtype=np.int32), shape=(4, 7))
  with pytest.raises(ValueError, match="shape\\[0\\] \\+ 1 = 4 entries"):
    bpl.check_csr(idx, ptr, shape=(3, 7))
  with pytest.raises(ValueError, match="int32 or uint32"):
    bpl.check_csr(idx.astype(np.int64), ptr, shape=(4, 7))


def test_python_scalars_are_kept_by_bit_pattern():
  # 0.0 and -0.0 compare equal and NaN does not equal itself: the host copies of Python numbers are
  # looked up by the value's bits
  import math
  from brainpylib_amd import _tensors
  a, b = _tensors.as_tensor(0.0), _tensors.as_tensor(-0.0)
  assert not math.copysign(1.0, a.item()) < 0 and math.copysign(1.0, b.item()) < 0
  assert _tensors.as_tensor(-0.0) is b and _tensors.as_tensor(0.0) is a
  n1, n2 = _tensors.as_tensor(float("nan")), _tensors.as_tensor(float("nan"))
  assert n1 is n2 and math.isnan(n1.item())
  assert _tensors.as_tensor(True).dtype == torch.bool and _tensors.as_tensor(1).dtype == torch.float32


def test_numbers_as_weights_are_told_apart_by_their_bits():
  from brainpylib_amd._tensors import number_operand
  for a, b in ((0.0, -0.0), (1, 2), (0.5, 0.25), (3, 3.5)):
    assert number_operand(a).host is not number_operand(b).host
    for v in (a, b):
      host = number_operand(v).host
      assert host is number_operand(v).host
      assert host.shape == (1,) and host.dtype == torch.float32
      assert host.item() == v and np.signbit(host.item()) == np.signbit(v)
  nan = number_operand(float("nan"))
  assert np.isnan(nan.host.item()) and nan is number_operand(float("nan"))


def test_native_enqueue_refuses_what_is_no_call():
  gpu_ops = pytest.importorskip("brainpylib_amd.gpu_ops")
  from brainpylib_amd import _lib
  address = ctypes.cast(_lib.target("event_csr_matvec_homo_float_bool"), ctypes.c_void_p).value
  for args in ((), (address, 0), (address, 0, "text"), (address, 0, b"") + (torch.zeros(1),) * 17):
    with pytest.raises(TypeError):
      gpu_ops.enqueue(*args)
  with pytest.raises(ValueError):
    gpu_ops.enqueue(0, 0, b"")
  with pytest.raises(AttributeError):
    gpu_ops.enqueue(address, 0, b"", 1)
  # a target's own error comes back as the exception and leaves nothing behind
  for _ in range(2):
    with pytest.raises(RuntimeError, match="event_csr_matvec_homo_float_bool"):
      gpu_ops.enqueue(address, 0, b"short", torch.zeros(1))
  assert not _lib.last_error()


def test_custom_call_takes_what_ctypes_takes():
  from brainpylib_amd import _lib

  class Stream:  # (as torch's streams are)
    _as_parameter_ = ctypes.c_void_p(0)
  one = torch.zeros(1)
  opaque = ctypes.create_string_buffer(b"short")
  for stream, descriptor, buffers in ((0, b"short", [one]), (ctypes.c_void_p(0), b"short", [one]), (Stream(), b"short", [one]),
                                      (0, opaque, [one]), (0, b"short", [one] * 17)):
    with pytest.raises(RuntimeError, match="event_csr_matvec_homo_float_bool"):  # (the target's own error)
      _lib.custom_call("event_csr_matvec_homo_float_bool", buffers, descriptor, stream=stream)
  assert not _lib.last_error()


def test_signature_of_an_autograd_function_binds_other_calls_as_inspect_does():
  from brainpylib_amd._tensors import keep_signature

  @keep_signature
  class F:
    @staticmethod
    def forward(a, b, c=3):
      return a
  sig = inspect.signature(F.forward)
  assert sig.bind(1, 2, 4).args == (1, 2, 4)
  usual = inspect.Signature(list(sig.parameters.values()))
  bound = sig.bind(1, 2, 4)
  bound.apply_defaults()
  assert bound == usual.bind(1, 2, 4)
  assert bound.kwargs == {} and bound.arguments == {"a": 1, "b": 2, "c": 4}
  bound = sig.bind(1, b=2)
  bound.apply_defaults()
  assert bound.args == (1, 2, 3)
  with pytest.raises(TypeError):
    sig.bind(1)


def test_tangents_are_found_where_torch_does_not_tell_its_level(monkeypatch):
  import types
  import torch.autograd.forward_ad as fwAD
  from brainpylib_amd import _tensors
  monkeypatch.setattr(_tensors, "forward_ad", types.SimpleNamespace(unpack_dual=fwAD.unpack_dual))
  t = torch.ones(2)
  assert not _tensors.has_tangent(t)
  with fwAD.dual_level():
    assert _tensors.has_tangent(fwAD.make_dual(t, t)) and not _tensors.has_tangent(t)


@pytest.mark.parametrize("context", ["inference_mode", "grad", "jvp", "vmap"])
def test_numbers_first_seen_inside_a_mode_or_transform_are_kept_as_plain_tensors(context, monkeypatch):
  # (the meta device stands for a GPU)
  from brainpylib_amd import _tensors
  for table in ("_PY_SCALARS", "_PY_NUMBERS", "_HOST_SCALARS"):
    monkeypatch.setattr(_tensors, table, {})
  device = torch.device("meta")
  own = torch.tensor([0.75])

  def first_call(x):
    _tensors.number_to_device(_tensors.number_operand(0.6), device)
    _tensors.as_tensor(0.7)
    _tensors.to_device(own, device)
    return (x * x).sum()
  x = torch.ones(3)
  if context == "inference_mode":
    with torch.inference_mode():
      first_call(x)
  elif context == "grad":
    torch.func.grad(first_call)(x)
  elif context == "jvp":
    torch.func.jvp(first_call, (x,), (x,))
  else:
    torch.func.vmap(first_call)(torch.ones(2, 3))
  number = _tensors.number_operand(0.6)
  kept = [number.host, number.copies[device], _tensors.as_tensor(0.6), _tensors.as_tensor(0.7), _tensors.to_device(own, device)]
  assert kept[1] is _tensors.number_to_device(number, device)
  for t in kept:
    t.data_ptr()  # (raises for a transform's wrapper)
    assert not t.is_inference()
    y = torch.ones(1, device=t.device, requires_grad=True)
    (y * t).sum().backward()  # (saves t)
  assert torch.equal(number.host, torch.tensor([0.6])) and _tensors.as_tensor(0.7).item() == np.float32(0.7)


def test_a_host_number_with_a_tangent_keeps_it_on_its_way_to_the_device(monkeypatch):
  # (the meta device stands for a GPU)
  import torch.autograd.forward_ad as fwAD
  from brainpylib_amd import _tensors
  monkeypatch.setattr(_tensors, "_HOST_SCALARS", {})
  device = torch.device("meta")
  t = torch.tensor([0.5])
  plain = _tensors.to_device(t, device)
  with fwAD.dual_level():
    assert _tensors.to_device(t, device) is plain
    moved = _tensors.to_device(fwAD.make_dual(t, torch.tensor([2.0])), device)
    assert fwAD.unpack_dual(moved).tangent is not None
  assert _tensors.to_device(t, device) is plain


def test_device_copies_of_numbers_stay_where_graphs_and_streams_may_read_them(monkeypatch):
  # (the meta device stands for a GPU)
  from brainpylib_amd import _tensors
  for table in ("_PY_SCALARS", "_PY_NUMBERS", "_HOST_SCALARS"):
    monkeypatch.setattr(_tensors, table, {})
  device = torch.device("meta")
  copy = lambda v: _tensors.number_to_device(_tensors.number_operand(v), device)
  most = _tensors._MOST_HOST_SCALARS
  kept = [copy(i + 0.5) for i in range(most)]
  late = copy(-1.0)
  assert _tensors._MOST_HOST_SCALARS <= 4096 and len(_tensors._HOST_SCALARS) == most
  assert all(any(t is k for k in _tensors._HOST_SCALARS.values()) for t in (kept[0], kept[-1]))
  assert copy(0.5) is kept[0] and copy(most - 0.5) is kept[-1]
  assert copy(-1.0) is not late and torch.device("meta") not in _tensors.number_operand(-1.0).copies
