"""Calls replayed in native code, as far as that needs no GPU: what a recipe passes on to an entry point (here a
recording callback), with arguments that are numbers."""
import collections
import copy
import ctypes
import pickle
import sys

import pytest
import torch
import torch.utils._python_dispatch

from antares_amd.autort import builtin_ops, patterns
from antares_amd.autort.op import ExportedOp
from antares_amd.runtime import calls


class Recording(calls.Operator):
    """Passes the numbers of `extra` on to a callback: as whole numbers, or as floats."""

    def __init__(self, kind='I', during=None):
        self.kind, self.seen, self.python_calls = kind, [], 0

        def entry(*values):
            self.seen.append(values[0])
            if during is not None:
                during()
            return 0
        # whole numbers are int arguments of the library's entry points
        self.entry = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_int if kind == 'I' else ctypes.c_float)(entry)
        self._bind(('x', 'extra'), ('extra',))

    def _call(self, pending, x=None, extra=None):
        self.python_calls += 1
        value = int(extra[0]) if self.kind == 'I' else float(extra[0])
        call = calls.Call(0)
        call.library(self.entry, calls.Number(value, 2, self.kind))
        call.keep(self, pending, [], device_stream=False)


@pytest.mark.parametrize('values', [(5, 6, 2 ** 31 - 1, -1, 0), (5.0, 6.0, 7.9, -7.9, 0.0), (True, False, True)])
def test_a_whole_number_is_passed_on_whatever_kind_of_number_it_is(values):
    op = Recording('I')
    for v in values * 2:
        op(None, extra=[v])
        op(extra=(v,))
    assert op.seen == [int(v) for v in values * 2 for _ in range(2)] and op.python_calls == 2


def test_a_position_that_changes_its_kind():
    op = Recording('I')
    for v in (5, 6.0, 7, 8.0, 9.5, True, 10, 11.5, 12) * 2:
        op(None, extra=[v])
    assert op.seen == [5, 6, 7, 8, 9, 1, 10, 11, 12] * 2


def test_a_float_is_passed_on_whatever_kind_of_number_it_is():
    op = Recording('F')
    values = (0.5, 0.25, 3, 4, 1e30) * 3
    for v in values:
        op(None, extra=[v])
    assert op.seen == [ctypes.c_float(float(v)).value for v in values] and op.python_calls == 2


def test_a_number_that_is_none_raises_what_it_raises_at_the_first_call():
    op = Recording('I')
    for first in (True, False):
        for v, error in ((float('nan'), ValueError), (float('inf'), OverflowError), (-float('inf'), OverflowError)):
            with pytest.raises(error):
                op(None, extra=[v])
        op(None, extra=[3.0])
    assert op.python_calls == 4 and op.seen == [3, 3]


def test_a_number_given_as_a_tensor_leaves_no_recipe(monkeypatch):
    """The value of a tensor that no launch takes may be part of the call's constants: the next call has another one."""
    monkeypatch.setattr(builtin_ops, 'current_stream_handle', lambda: 0)
    kept = []
    monkeypatch.setattr(calls.Call, 'keep', lambda self, *a, **k: kept.append(self))
    entry = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p)(lambda *a: 0)
    x, out, number, empty = torch.ones(4), torch.empty(4), torch.tensor([3]), torch.empty(0)

    def run(slots, *args):
        kept.clear()
        builtin_ops._run(None, None if slots is None else (b'', slots, -1), out, entry, *args)
        return len(kept)
    assert run((x, out), x, 3) == 1
    assert run((x, out, [5], 5), x, calls.Number(5, 3, 'I')) == 1
    assert run((x, None, empty), x, 3) == 1               # a tensor without elements has no value
    assert run((x, out, [number], number), x, int(number)) == 0
    assert run((x, number, out), x, int(number)) == 0
    assert run(None, x, 3) == 0


def test_a_view_of_an_argument_leaves_no_recipe(monkeypatch):
    monkeypatch.setattr(calls, 'setup', lambda: None)
    kept = []

    class Keeping:
        def _commit(self, *recipe):
            kept.append(recipe)
    entry = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p)(lambda *a: 0)
    x, fresh = torch.ones(4), torch.empty(4)

    def keep(arg, result):
        kept.clear()
        call = calls.Call(0)
        call.library(entry, arg)
        call.keep(Keeping(), (b'', (x,), -1), [result], device_stream=False)
        return len(kept)
    assert keep(x, fresh) == 1 and keep(fresh, x) == 1 and keep(x[:0], x) == 1
    assert keep(x[:2], fresh) == 0 and keep(x, x[1:]) == 0 and keep(x.view(2, 2), fresh) == 0


class GpuShaped(torch.Tensor):
    """Dtype, shape and device of a GPU tensor, without one."""

    @staticmethod
    def __new__(cls, *shape):
        return torch.Tensor._make_wrapper_subclass(cls, shape, dtype=torch.float32, device='cuda:0')

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        raise NotImplementedError(func)


class Reached(Exception):
    pass


class Noting(calls.Operator):
    def __init__(self):
        self.pending = []
        self._bind(('x', 'extra'), ())

    def _call(self, pending, x=None, extra=None):
        self.pending.append(pending)
        raise Reached


TRANSFORMS = [
    lambda f: torch.vmap(f)(GpuShaped(3, 4)),
    lambda f: torch.vmap(torch.vmap(f))(GpuShaped(3, 4, 5)),
    lambda f: torch.func.grad(f)(GpuShaped(3, 4)),
    lambda f: torch.func.functionalize(f)(GpuShaped(3, 4))]


@pytest.mark.parametrize('transform', TRANSFORMS)
def test_a_tensor_without_memory_reaches_the_python_method(transform):
    """Inside torch.func's transformations a GPU tensor is a plain torch.Tensor without storage, or without memory."""
    op = Noting()

    def call(x):
        assert type(x) is torch.Tensor and x.is_cuda
        with pytest.raises(Reached):
            op(x)
        with pytest.raises(Reached):
            op(None, extra=[x])
        raise Reached
    with pytest.raises(Reached):
        transform(call)
    assert op.pending == [None, None]


@pytest.mark.skipif(torch.cuda.is_available(), reason='the error of a machine without a GPU')
def test_an_error_of_torch_in_a_replayed_call_is_a_python_exception():
    entry = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p)(lambda *a: 0)

    class Streaming(calls.Operator):
        def __init__(self):
            self._bind(('x',), ())

        def _call(self, pending, x=None):
            call = calls.Call(0)
            call.library(entry, calls.STREAM)
            call.keep(self, pending, [], device_stream=False)
    op = Streaming()
    op(None)
    for _ in range(3):
        with pytest.raises(RuntimeError):               # no device, hence no current stream
            op(None)


def test_a_tensor_without_memory_is_refused_before_the_launch():
    called = []
    entry = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_void_p)(lambda *a: called.append(a) or 0)

    def launch(x):
        call = calls.Call(0)
        with pytest.raises(RuntimeError):
            call.library(entry, x)
        with pytest.raises(RuntimeError):
            call.kernel(None, 1, 64, [x])
        raise Reached
    for transform in TRANSFORMS:
        with pytest.raises(Reached):
            transform(launch)
    assert not called


@pytest.mark.parametrize('as_list', [True, False])
def test_arguments_live_until_the_call_is_over(as_list):
    """Other threads run while a recipe's entry points do, and may change a list argument."""
    value, counts = float('1234.5'), []
    extra = [value] if as_list else (value,)

    def during():
        if op.seen[1:] and as_list:
            extra.clear()
        counts.append(sys.getrefcount(value))
    op = Recording('F', during)
    op(None, extra=[value])                              # leaves the recipe
    counts.clear()
    before = sys.getrefcount(value)
    op(None, extra=extra)
    assert op.seen == [1234.5] * 2 and op.python_calls == 1
    assert counts == [before + (0 if as_list else 1)]           # the list's reference is gone, the call's is there
    assert sys.getrefcount(value) == before - as_list


def exported(name, **kw):
    return ExportedOp('output0[N] = input0[N] + input1[N]', ['input0=float32[N:64]', 'input1=float32[N:64]'], name=name, **kw)


def by_hand(name):
    op = ExportedOp(patterns.W4A16_IR, patterns.W4A16_INPUTS, name=name, config='tune:3', tuned={'k': {'value': 2}})
    assert op.fast_path is not None
    return op


@pytest.mark.parametrize('duplicate', [copy.copy, copy.deepcopy])
@pytest.mark.parametrize('make', [exported, by_hand, lambda name: builtin_ops.RmsNorm(torch.float16), lambda name: builtin_ops.PartitionEvenFirst()])
def test_operators_can_be_copied(make, duplicate):
    op = make('copied')
    holder = torch.nn.Module()
    holder.op = op
    twin, held = duplicate(op), copy.deepcopy(holder).op
    assert held is not op
    for t in (twin, held):
        assert type(t) is type(op) and vars(t).keys() == vars(op).keys() and t.name == op.name
        assert t.tuned == op.tuned and t.config == op.config and (t.fast_path is None) == (op.fast_path is None)
    assert twin is not op and (op.tuned is None or (twin.tuned is op.tuned) == (duplicate is copy.copy))
    twin.fast_path = None                                # its own attributes
    twin.tuned = {'other': {'value': 1}}
    assert op.tuned != twin.tuned and (op.fast_path is None) == (make is not by_hand)


def test_a_copy_is_called_like_the_operator_it_is_a_copy_of():
    op = Recording('I')
    op(None, extra=[1])
    op(None, extra=[2])
    twin = copy.copy(op)
    for i in (3, 4, 5):
        twin(None, extra=[i])
    twin(extra=[6], x=None)
    op(None, extra=[7])
    assert op.seen == [1, 2, 3, 4, 5, 6, 7] and (op.python_calls, twin.python_calls) == (1, 2)


def test_built_in_operators_can_be_pickled():
    for op in (builtin_ops.RmsNorm(torch.float32), builtin_ops.Rotary('rotary_f32', False), builtin_ops.GemvW4Fused(), builtin_ops.PartitionEvenFirst()):
        twin = pickle.loads(pickle.dumps(op))
        assert type(twin) is type(op) and vars(twin) == vars(op) and twin.tuned == op.tuned


@pytest.mark.parametrize('attribute', ['fast_path', 'tuned', 'config'])
def test_an_attribute_that_is_replaced_ends_the_recipes(attribute):
    """Also where the new object takes the old one's place in memory."""
    op = Recording('I')
    for i in range(20):
        setattr(op, attribute, None)
        setattr(op, attribute, (lambda: i) if attribute == 'fast_path' else {'i': i})
        for _ in range(3):
            op(None, extra=[i])
        assert op.python_calls == i + 1
    if attribute != 'fast_path':
        getattr(op, attribute)['i'] = 'changed'              # and one that is changed in place
        op(None, extra=[1])
        assert op.python_calls == 21
        setattr(op, attribute, collections.OrderedDict(i=1))     # whose changes leave no trace
        for _ in range(2):
            op(None, extra=[1])
        assert op.python_calls == 23
    delattr(op, attribute)
    assert getattr(op, attribute) is None


def test_calls_under_a_dispatch_mode_or_with_filled_memory_are_not_replayed():
    class Mode(torch.utils._python_dispatch.TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))
    op = Recording('I')
    for i in (0, 1, 2):
        op(None, extra=[i])
    assert op.python_calls == 1
    with Mode():
        op(None, extra=[3])
        op(None, extra=[4])
    assert op.python_calls == 3
    before = torch.are_deterministic_algorithms_enabled()
    try:
        torch.use_deterministic_algorithms(True)
        op(None, extra=[5])
        op(None, extra=[6])
    finally:
        torch.use_deterministic_algorithms(before)
    assert op.python_calls == 5
    op(None, extra=[7])
    assert op.python_calls == 5 and op.seen == [0, 1, 2, 3, 4, 5, 6, 7]


class Sized(calls.Operator):
    """Its signature is the size: every size has a recipe of its own."""

    def __init__(self):
        self.python_calls, self.pending, self.seen = 0, 0, []
        self.entry = ctypes.CFUNCTYPE(ctypes.c_int, ctypes.c_int)(lambda n: self.seen.append(n) or 0)
        self._bind(('size',), ())

    def _call(self, pending, size):
        self.python_calls += 1
        self.pending += pending is not None
        call = calls.Call(0)
        call.library(self.entry, size)
        call.keep(self, pending, [], device_stream=False)


def test_recipes_that_are_not_used_are_made_only_for_signatures_met_again():
    """Making one costs as much as a call: where every call has another signature, it is not worth it."""
    op = Sized()
    for size in range(1000):
        op(size)
    assert 8 <= op.pending < 16                          # the credit; and the marks are 32 bits of a hash
    for size in range(1000):
        op(size)
    made = op.pending
    assert made > 800                                    # two signatures in one place of the marks take it from each other
    for size in range(1000):
        op(size)
    assert op.pending - made < 200 and op.seen == [size for _ in range(3) for size in range(1000)]


def test_recipes_that_are_used_are_made_at_the_first_call():
    op = Sized()
    for size in range(1000):
        for _ in range(3):
            op(size)
    assert op.python_calls == 1000
    for size in range(2000, 2008):                       # eight of them may wait for their use
        op(size)
    for size in range(2000, 2008):
        op(size)
    assert op.python_calls == 1008


def test_an_argument_that_is_missing_is_not_one_that_is_none():
    entry = ctypes.CFUNCTYPE(ctypes.c_int)(lambda: 0)

    class Two(calls.Operator):
        def __init__(self):
            self._bind(('a', 'b', 'c'), ())

        def _call(self, pending, a, b, c=None):
            call = calls.Call(0)
            call.library(entry)
            call.keep(self, pending, [], device_stream=False)
    op = Two()
    for _ in range(4):
        op(None, None)
        op(b=None, a=None)
        with pytest.raises(TypeError):
            op(None)
        with pytest.raises(TypeError):
            op(b=None)
        with pytest.raises(TypeError):
            op(None, None, None, None)
        with pytest.raises(TypeError):
            op(None, None, a=None)
        with pytest.raises(TypeError):
            op(None, None, d=None)


def test_the_table_is_emptied_when_it_is_full():
    op = Sized()
    for size in range(9000):
        for _ in range(3):
            op(size)
    assert op.seen == [size for size in range(9000) for _ in range(3)] and op.python_calls == 9000
    op(8999)                                             # made after the table was emptied
    assert op.python_calls == 9000
    op(0)
    op(0)
    assert op.python_calls == 9001
