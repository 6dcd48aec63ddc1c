"""Argument plumbing shared by the operator wrappers: everything becomes a contiguous torch
CUDA tensor (device memory is PyTorch-ROCm's; nothing is computed with torch)."""
import ctypes
import inspect
import struct
import threading

import numpy as np
import torch
from torch.autograd import forward_ad

FLOAT_DTYPES = (torch.float32, torch.float64)
_INDEX_DTYPES = (torch.int32, torch.uint32)


_PY_SCALARS = {}  # host tensors of Python numbers seen as operands (read-only)


def _is_plain(t):
  if type(t) is not torch.Tensor or t.is_inference():
    return False
  try:
    t.data_ptr()
  except RuntimeError:  # a wrapper of a function transform
    return False
  return True


def _plain(make):
  """``make()``, a tensor that later calls are given too: one that belongs to no inference mode, function transform or
  dispatch mode that happens to be active at the first of them.  All of these are a thread's own, so where leaving inference
  mode is not enough the tensor is made by another thread (on the caller's stream)."""
  with torch.inference_mode(False):
    t = make()
  if _is_plain(t):
    return t
  made = []
  stream = torch.cuda.current_stream() if torch.cuda.is_available() else None

  def work():
    try:
      with torch.cuda.stream(stream):
        made.append(make())
    except Exception as e:  # (raised below, in the caller's thread)
      made.append(e)
  thread = threading.Thread(target=work)
  thread.start()
  thread.join()
  if isinstance(made[0], Exception):
    raise made[0]
  return made[0]


def as_tensor(a):
  """Unwraps brainpy-like arrays (objects with `.value`) and wraps numpy / python data as a torch
  tensor WITHOUT moving it, so that argument checks can run before a device is needed.
  Python floats become float32 (the reference's default float)."""
  if hasattr(a, "value") and not isinstance(a, (torch.Tensor, np.ndarray)):
    a = a.value
  if isinstance(a, torch.Tensor):
    return a
  if isinstance(a, (bool, int, float)):
    # keyed by the value's bits, so that 0.0 and -0.0 are two entries and a NaN finds its own
    key = (type(a), struct.pack("<d", a) if isinstance(a, float) else a)
    t = _PY_SCALARS.get(key)
    if t is None:
      if len(_PY_SCALARS) >= 256:
        _PY_SCALARS.clear()
      dtype = torch.bool if isinstance(a, bool) else torch.float32
      t = _PY_SCALARS[key] = _plain(lambda: torch.tensor(a, dtype=dtype, device="cpu"))
    return t
  arr = np.asarray(a)
  if arr.dtype == np.uint32:
    return torch.from_numpy(np.ascontiguousarray(arr).view(np.int32)).view(torch.uint32)
  if arr.ndim == 0:
    return torch.tensor(arr.item(), dtype=_np_to_torch(arr.dtype))
  return torch.from_numpy(np.ascontiguousarray(arr))


class _NumberTensor:
  """A Python number as a host tensor of shape (1,), with that tensor's copies on devices."""
  __slots__ = ("host", "copies")

  def __init__(self, value):
    scalar = as_tensor(value)
    self.host = _plain(lambda: scalar.reshape(1))
    self.copies = {}


_PY_NUMBERS = {}


def number_operand(value):
  """The _NumberTensor of a Python int or float (a homogeneous weight), made once per value."""
  # keyed by the value's bits, as in as_tensor
  key = struct.pack("<d", value) if type(value) is float else value
  number = _PY_NUMBERS.get(key)
  if number is None:
    if len(_PY_NUMBERS) >= 256:
      _PY_NUMBERS.clear()
    number = _PY_NUMBERS[key] = _NumberTensor(value)
  return number


def number_to_device(number, device):
  copy = number.copies.get(device)
  if copy is None:
    copy, kept = _scalar_copy(number.host, device)
    if kept:
      number.copies[device] = copy
  return copy


def device_of(*args):
  """The device the call runs on: that of the first CUDA tensor argument, else the current one."""
  for a in args:
    if isinstance(a, torch.Tensor) and a.is_cuda:
      return a.device
  if not torch.cuda.is_available():
    raise RuntimeError("brainpylib_amd needs a HIP device: there is no CPU path in this package.")
  return torch.device("cuda", torch.cuda.current_device())


def has_tangent(t):
  # (outside a dual level, where unpack_dual finds no tangent either, its named tuple is most of the cost; the level is
  # torch's own name, and without it every tensor is looked at)
  return getattr(forward_ad, "_current_level", 0) >= 0 and t.is_floating_point() and forward_ad.unpack_dual(t).tangent is not None


# Device copies of one-element host operands.  One that is here stays: queued calls on other streams and captured graphs
# may still read it.  What comes when the table is full (512 bytes of device memory an entry) is copied for its call alone.
_HOST_SCALARS = {}
_MOST_HOST_SCALARS = 4096


def _bits(t):
  """The bytes of a host tensor of one element."""
  try:
    return t.numpy().tobytes()
  except RuntimeError:
    if not _is_plain(t):
      raise
    return ctypes.string_at(t.data_ptr(), t.element_size())  # (inside a function transform, where numpy() is not to be had)


def _scalar_copy(t, device):
  """A one-element host tensor on a device, and whether the table of copies holds it."""
  key = (_bits(t), t.dtype, tuple(t.shape), device)  # (the bits: -0.0 is not 0.0, NaN equals itself)
  hit = _HOST_SCALARS.get(key)
  if hit is not None:
    return hit, True
  copy = _plain(lambda: t.to(device).contiguous())
  if len(_HOST_SCALARS) >= _MOST_HOST_SCALARS:
    return copy, False
  return _HOST_SCALARS.setdefault(key, copy), True  # (another thread may have been first)


def to_device(t, device):
  if t.device != device:
    if t.numel() == 1 and t.device.type == 'cpu' and not t.requires_grad and not has_tangent(t):
      # A one-element host operand (a homogeneous weight given as a Python number): its device copy
      # is made once per value.  A pageable host-to-device copy per call would cost more than the
      # kernels of a small network.  The operators only read their operands.
      return _scalar_copy(t, device)[0]
    t = t.to(device)
  return t.contiguous()


def _np_to_torch(dt):
  return {np.dtype(np.float32): torch.float32, np.dtype(np.float64): torch.float64,
          np.dtype(np.int32): torch.int32, np.dtype(np.int64): torch.int64,
          np.dtype(np.bool_): torch.bool, np.dtype(np.uint8): torch.uint8}.get(np.dtype(dt), torch.float32)


def is_index_dtype(dt):
  return dt in _INDEX_DTYPES


class _PositionalSignature(inspect.Signature):
  """The signature of a ``forward`` that is only called with all its arguments by position: there is nothing to match."""
  __slots__ = ()

  def bind(self, *args, **kwargs):
    if kwargs or len(args) != len(self.parameters):
      return super().bind(*args, **kwargs)
    return _PositionalArguments(self, args)


class _PositionalArguments(inspect.BoundArguments):
  """Arguments that were all given by position; by name only if somebody asks."""
  __slots__ = ("args",)

  def __init__(self, signature, args):
    self._signature = signature
    self.args = args

  @property
  def arguments(self):
    return dict(zip(self._signature.parameters, self.args))

  @property
  def kwargs(self):
    return {}

  def apply_defaults(self):
    pass


def keep_signature(function):
  """Class decorator for autograd functions: torch binds the arguments of one with a ``setup_context`` through
  ``inspect.signature(forward).bind`` on every call, which costs more host time than the call it prepares; the
  signature kept on ``forward`` passes arguments given by position through."""
  function.forward.__signature__ = _PositionalSignature(
    list(inspect.signature(function.forward).parameters.values()))
  return function
