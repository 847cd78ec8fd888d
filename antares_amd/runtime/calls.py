"""Operators whose calls are replayed in native code.

``Operator`` (``csrc/host/calls.cpp``) is the base class of everything callable in ``autort.ops``.  A call whose
signature - dtypes, shapes, devices, contiguity and 16-byte alignment of the tensors, which of them share memory, which
arguments are given - has a recipe is replayed from it without entering Python; any other call reaches the subclass's
``_call(pending, ...)``, which checks the arguments, runs the operator and leaves the recipe with ``pending`` (None when none
is wanted, or the arguments are nothing a recipe can be kept for).
"""
from __future__ import annotations

import ctypes
from ctypes import c_void_p

import torch

from . import capi

try:
    from . import _calls
    _Base = _calls.Operator
except ImportError as _e:                     # not built: operators can still be made (lowering, compiling), not called
    _calls, _reason = None, str(_e)

    class _Base:
        tuned = config = fast_path = None

        def _bind(self, names, dynamic):
            pass

        def __call__(self, *args, **kwargs):
            raise capi.ArtError(f'antares_amd/runtime/_calls.so cannot be loaded ({_reason}): build it with `python -m antares_amd.build`')


class Operator(_Base):
    """Copies and pickles like an object of Python's: with its attributes, without its recipes."""

    def _bind(self, names, dynamic):
        self._parameters = (names, dynamic)
        super()._bind(names, dynamic)

    def __getstate__(self):
        return {**vars(self), **{n: getattr(self, n) for n in ('tuned', 'config', 'fast_path') if getattr(self, n) is not None}}

    def __setstate__(self, state):
        for name, value in state.items():
            setattr(self, name, value)
        self._bind(*self._parameters)


_ready = False


def setup():
    """Hands the native side the library's launch entry point; before the first recipe is kept."""
    global _ready
    if not _ready:
        lib = capi.lib()
        _calls.setup(ctypes.cast(lib.art_launch, c_void_p).value, ctypes.cast(lib.art_last_error, c_void_p).value, capi.ArtError,
                     torch.nn.Parameter)
        _ready = True


def forget():
    """Every recipe is worked out again at its next call (the rules of a launch plan have changed)."""
    if _calls is not None:
        _calls.forget()


class Stream:
    """The stream of the call, as an argument."""


STREAM = Stream()
_Tensor = torch.Tensor


class Number:
    """Number ``index`` of the call's list argument, passed on as it is: its value now, and its place in later calls."""
    __slots__ = ('value', 'slot', 'kind')

    def __init__(self, value, slot: int, kind: str):
        self.value, self.slot, self.kind = value, slot, kind


class _ViewOfAnArgument(Exception):
    pass


def address(t: torch.Tensor) -> int:
    """Where a tensor's elements are; an error for a wrapper (torch.func, functionalisation) that has none."""
    at = t.data_ptr()
    if not at and t.numel():
        raise capi.ArtError(f'a tensor of shape {list(t.shape)} has no memory')
    return at


def _value(a, stream: int):
    if a is STREAM:
        return stream
    if isinstance(a, _Tensor):
        return address(a)
    return a.value if a.__class__ is Number else a


def values(args, stream: int) -> list:
    """Arguments as ctypes takes them: tensors by their address, STREAM as the handle, a Number as its value."""
    return [a if a.__class__ is int else (a.data_ptr() or address(a)) if a.__class__ is _Tensor else _value(a, stream) for a in args]


class Call:
    """What one call of an operator launches, in order: kernels and entry points of the library, with tensors as
    tensors, the stream as STREAM, list numbers as Number, and constants.  ``replay``: False when the next call of the same
    signature may go another way (there was no memory for the usual one)."""

    __slots__ = ('stream', 'steps', 'replay')

    def __init__(self, stream: int):
        self.stream = stream
        self.steps = []
        self.replay = True

    def library(self, fn, *args):
        given = values(args, self.stream)
        self.steps.append((fn, None, None, args))
        capi.check(fn(*given))

    def kernel(self, func, grid: int, block: int, args):
        given = values(args, self.stream)
        self.steps.append((func, (grid, 1, 1), (block, 1, 1), args))
        capi.launch(func, (grid, 1, 1), (block, 1, 1), self.stream, given)

    def keep(self, op: Operator, pending, results, device_stream: bool):
        """Leaves the recipe of this call with the operator.  Tensors that are not among the call's arguments are
        allocated afresh by every later call; a view of an argument is neither, and a call that uses one leaves no recipe."""
        if pending is None or not self.replay:
            return
        setup()
        key, slots, device = pending
        place, owned = {}, set()
        for i, s in enumerate(slots):             # one tensor in two places is part of the signature
            if isinstance(s, torch.Tensor):
                place.setdefault(id(s), i)
                owned.add(s.untyped_storage().data_ptr())
        fresh = []

        def index(t):
            at = place.get(id(t))
            if at is None:
                if t.numel() and t.untyped_storage().data_ptr() in owned:
                    raise _ViewOfAnArgument
                at = place[id(t)] = len(slots) + len(fresh)
                fresh.append(t)
            return at

        def encode(fn, a):
            if isinstance(a, torch.Tensor):
                return ('p', index(a))
            if a is STREAM:
                return ('s',)
            if isinstance(a, Number):
                return (a.kind, a.slot)
            if isinstance(a, float):
                return ('f', a)
            return ('i', int(a or 0))
        launches = []
        try:
            for fn, grid, block, args in self.steps:
                address = fn.value if grid is not None else ctypes.cast(fn, c_void_p).value
                launches.append((address, grid, block, [encode(fn, a) for a in args]))
            outs = [index(t) for t in results]
        except _ViewOfAnArgument:
            return
        if len(fresh) <= 16:
            op._commit(key, len(slots), device, int(device_stream), [(t.dtype, tuple(t.shape)) for t in fresh], launches, outs)
