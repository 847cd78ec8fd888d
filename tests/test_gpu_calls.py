"""Calls replayed in native code: what belongs to a signature (shapes, alignment, one tensor in two places, which
arguments are given) leads to a recipe of its own, what does not (addresses, numbers in `extra`) is taken from the call,
and a call that cannot be replayed still raises what it raised before."""
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def op():
    import autort
    return autort.export(ir='output0[N] = input0[N] + input1[N]', inputs=['input0=float32[N:64]', 'input1=float32[N:64]'], name='calls_add')


@pytest.mark.parametrize('n', [0, 1, 3, 4, 1000, 4099])
def test_every_signature_gets_its_own_recipe(op, n):
    import autort
    print(f'[case] calls n={n}', flush=True)
    dev = autort.device()
    for offset in (0, 1, 4):                                 # aligned, not aligned, aligned again
        for _ in range(3):
            a, b = torch.randn(n + 4, device=dev)[offset:n + offset], torch.randn(n, device=dev)
            assert a.numel() == n and torch.equal(op(a, b), a + b)
            assert torch.equal(op(a, a), a + a)              # one tensor in two places ...
            assert torch.equal(op(b, a), a + b)              # ... is not what two tensors are
            out = torch.empty(n, device=dev)
            assert op(a, b, out=out) is out and torch.equal(out, a + b)
            assert op(a, b, out) is out
            kept = a.clone()
            assert op(a, b, out=a) is a and torch.equal(a, kept + b)


def test_errors_are_raised_after_a_replayed_call_too(op):
    import autort
    dev = autort.device()
    a = torch.randn(100, device=dev)
    op(a, a)
    op(a, a)
    for bad in ((a,), (a, a.half()), (a, a.cpu()), (a, torch.randn(200, device=dev)[::2]), (a, 1.0), (a, a, torch.empty(7, device=dev)), (a, torch.randn(99, device=dev))):
        with pytest.raises(Exception):
            op(*bad)
    with pytest.raises(TypeError):
        op(a, input1=a)
    assert torch.equal(op(a, a), a + a)


def test_numbers_in_extra_and_the_stream_are_taken_from_the_call():
    import autort
    dev = autort.device()
    x, w = torch.randn(256, device=dev), torch.randn(256, device=dev)
    vsum = (x * x).sum().view(1)
    for inv_n in (1 / 256, 1 / 64, 1.0, 1):
        want = x * torch.rsqrt(vsum * inv_n + 1e-5) * w
        assert torch.allclose(autort.ops.rmsnorm_f32(x, vsum, w, extra=[inv_n]), want, rtol=1e-4, atol=1e-5)
    q = torch.randn(2, 2, 64, device=dev)
    inv = torch.rand(128, device=dev)
    for pos in (0, 1, 77, torch.tensor([77], dtype=torch.int32, device=dev), torch.tensor([3], dtype=torch.int32, device=dev)):
        angle = float(pos) * inv[:64]
        want = torch.cat([q[:, 0] * angle.cos() - q[:, 1] * angle.sin(), q[:, 1] * angle.cos() + q[:, 0] * angle.sin()], 1)
        got = autort.ops.rotary_f32(q, inv, torch.empty(2, 128, device=dev), extra=[pos])
        assert torch.allclose(got, want, rtol=1e-4, atol=1e-4)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        g = torch.cuda.CUDAGraph()
        out = torch.zeros(256, device=dev)
        autort.ops.rmsnorm_f32(x, vsum, w, out, extra=[1.0])
        side.synchronize()
        with torch.cuda.graph(g, stream=side):               # recorded on the capturing stream: not run yet
            autort.ops.rmsnorm_f32(x, vsum, w, out, extra=[0.25])
        first = out.clone()
        g.replay()
    side.synchronize()
    assert not torch.equal(first, out) and torch.allclose(out, x * torch.rsqrt(vsum * 0.25 + 1e-5) * w, rtol=1e-4, atol=1e-5)


def test_several_threads_call_one_operator(op):
    import autort
    dev = autort.device()
    wrong = []

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for k in range(50):
                a = torch.full((64 + (i + k) % 7,), float(i), device=dev)
                if not torch.equal(op(a, a), a + a):
                    wrong.append((i, k))
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


# a position is taken by its value in every call, also where an earlier call of the signature had another kind of number
@pytest.mark.parametrize('positions', [(5.0, 6.0, 77.9), (5, 6.0, 7, True, 8.0)])
@pytest.mark.parametrize('name', ['rotary_f32', 'rotate_f32'])
def test_a_position_may_be_any_number(name, positions):
    import autort
    print(f'[case] {name} {positions}', flush=True)
    dev = autort.device()
    x, inv = torch.randn(2, 2, 64, device=dev), torch.rand(128, device=dev)
    for pos in positions * 3:
        angle = float(int(pos)) * inv[:64]
        if name == 'rotary_f32':
            want = torch.cat([x[:, 0] * angle.cos() - x[:, 1] * angle.sin(), x[:, 1] * angle.cos() + x[:, 0] * angle.sin()], 1)
            got = autort.ops.rotary_f32(x, inv, torch.empty(2, 128, device=dev), extra=[pos])
        else:
            data = x.view(2, 128)[0]
            re, im = data[0::2], data[1::2]
            want = torch.stack([re * angle.cos() - im * angle.sin(), im * angle.cos() + re * angle.sin()], 1).view(128)
            got = autort.ops.rotate_f32(inv[:64].view(1, 64), data, torch.empty(128, device=dev), extra=[pos])
        assert torch.allclose(got, want, rtol=1e-4, atol=1e-4)


def test_a_number_given_as_a_tensor_is_read_in_every_call():
    import autort
    dev = autort.device()
    x, w = torch.randn(256, device=dev), torch.randn(256, device=dev)
    vsum = (x * x).sum().view(1)
    for inv_n in (1 / 256, 1 / 64, 1.0):
        want = x * torch.rsqrt(vsum * inv_n + 1e-5) * w
        for extra in ([torch.tensor(inv_n, device=dev)], [torch.tensor([inv_n], device=dev), 1e-5]):
            assert torch.allclose(autort.ops.rmsnorm_f32(x, vsum, w, extra=extra), want, rtol=1e-4, atol=1e-5)
    qkv, inv = torch.randn(3, 3 * 256, device=dev).half(), torch.rand(128, device=dev).half()
    for first in (0, 2, 5):
        got, want = ([torch.zeros(3, 2, 128, device=dev).half()] + [torch.zeros(8, 256, device=dev).half() for _ in range(2)] for _ in range(2))
        autort.ops.rope_qkv_store_rows_f16(qkv, inv, *got, extra=[torch.tensor([first], device=dev)])
        autort.ops.rope_qkv_store_rows_f16(qkv, inv, *want, extra=[first])
        assert all(torch.equal(a, b) for a, b in zip(got, want)) and torch.equal(got[2][first:first + 3], qkv[:, 512:])


def test_a_tensor_of_positions_in_the_place_of_the_list():
    import autort
    dev = autort.device()
    x, inv = torch.randn(2, 2, 64, device=dev), torch.rand(128, device=dev)
    for pos in (3, 4, 5, 6):
        got = autort.ops.rotary_f32(x, inv, torch.empty(2, 128, device=dev), extra=torch.tensor([pos], dtype=torch.int32, device=dev))
        assert torch.equal(got, autort.ops.rotary_f32(x, inv, torch.empty(2, 128, device=dev), extra=[pos]))


def test_errors_of_torch_are_python_exceptions_in_replayed_calls_too(op):
    import autort
    dev = autort.device()
    big = torch.zeros(32 << 20, device=dev)
    for _ in range(3):
        op(big, big)
    for transform in (lambda f: torch.vmap(f)(torch.zeros(2, 64, device=dev)), lambda f: torch.func.functionalize(f)(torch.zeros(64, device=dev)),
                      lambda f: torch.func.grad(lambda x: f(x).sum())(torch.zeros(64, device=dev))):
        with pytest.raises(RuntimeError):
            transform(lambda x: op(x, x))
    kept = [op(big, big) for _ in range(2)]
    del kept
    torch.cuda.empty_cache()
    try:
        torch.cuda.set_per_process_memory_fraction(1e-4)
        with pytest.raises(torch.OutOfMemoryError):
            op(big, big)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert not op(big, big).any()


def conv_op(name):
    import autort
    return autort.export(ir='output0[N, F, HO, WO] +=! input0[N, C, HO + KH - 1, WO + KW - 1].when([HO + KH - 1 >= 0, HO + KH - 1 < 28, WO + KW - 1 >= 0, '
                            'WO + KW - 1 < 28], 0.0) * input1[F, C, KH, KW] where HO in 28, WO in 28',
                         inputs=['input0=float32[N:4, C:64, H:28, W:28]', 'input1=float32[F:64, C:64, KH:3, KW:3]'], name=name)


@pytest.mark.parametrize('order', ['over its image first', 'apart first'])
def test_a_convolution_over_its_image_and_one_apart_from_it_do_not_depend_on_each_other(order):
    import autort
    dev = autort.device()
    op = conv_op('calls_conv_' + order.split()[0])
    g = torch.Generator().manual_seed(1)
    x, w = torch.randn(4, 64, 28, 28, generator=g), torch.randn(64, 64, 3, 3, generator=g) / 24
    want, bound = (torch.nn.functional.conv2d(a, b, padding=1) for a, b in ((x.double(), w.double()), (x.double().abs(), w.double().abs())))
    taken = []
    handler = op.fast_path
    op.fast_path = lambda *a: taken.append(handler(*a)) or taken[-1]

    def check(got):
        assert ((got.cpu().double() - want).abs() <= 2.0 ** -23 * 9 * 64 * bound).all()
    for where in (['over', 'apart', 'behind'] if order.startswith('over') else ['apart', 'behind', 'over']) * 3:
        print(f'[case] convolution {where}', flush=True)
        memory = torch.zeros(2 * x.numel(), device=dev)
        image = memory[:x.numel()].view_as(x).copy_(x)
        at = {'over': 0, 'apart': None, 'behind': x.numel()}[where]        # behind: the first element past the image
        check(op(image, w.to(dev), out=None if at is None else memory[at:at + x.numel()].view_as(x)))
    assert sorted(taken) == [False, True, True]          # a recipe each: by hand where the memory is apart


def test_which_tensors_share_memory_is_part_of_the_signature():
    from antares_amd.runtime import calls
    import autort
    dev = autort.device()

    class Keys(calls.Operator):
        def __init__(self):
            self._bind(('a', 'b', 'c', 'extra'), ())

        def _call(self, pending, *args, **kwargs):
            return pending and pending[0]
    op = Keys()

    def key(*args, **kwargs):
        return op(*args, **kwargs) or op(*args, **kwargs)          # pending when a recipe is wanted: once the credit is spent, for a signature met again
    m = torch.zeros(64, device=dev)
    a, b, c = m[0:16], m[16:32], m[32:48]
    base = key(a, b, c)
    assert base == key(a, c, b) == key(b, c, a) == key(c.clone(), b, a) and base != key(a, b, [c])
    keys = [base, key(a, a, c), key(a, b, a), key(a, b, b), key(a, m[12:28], c), key(a, b, m[12:28]), key(a, b, m[20:36]),
            key(m[4:20], m[12:28], m[20:36]), key(m[4:20], m[8:24], m[12:28])]
    assert len(set(keys)) == len(keys)
    assert key(a, m[4:20], c) == key(b, m[12:28], c) == key(a, m[0:16], c)  # how they overlap is not
    assert key(a, b, extra=[c]) != key(a, b, extra=[b])
    none = m[:0]
    assert key(none, m[:0], c) == key(none, m[4:4], a)                     # nothing to share without elements


def test_copies_of_an_operator_are_called_like_it(op):
    import copy
    import autort
    dev = autort.device()
    fresh = autort.export(ir=op.ir, inputs=op.input_specs, name='calls_add_fresh')
    norm = autort.ops.rmsnorm_f32
    a, b = torch.randn(1000, device=dev), torch.randn(1000, device=dev)
    op(a, b)
    for twin in (copy.deepcopy(fresh), copy.copy(fresh), copy.copy(op)):
        assert all(torch.equal(twin(a, b), a + b) for _ in range(3))
    assert all(torch.equal(copy.deepcopy(norm)(a, None, b), norm(a, None, b)) for _ in range(2))


def test_a_lazy_copy_is_written_apart_from_its_original(op):
    import autort
    dev = autort.device()
    a, b, kept = torch.randn(1000, device=dev), torch.randn(1000, device=dev), torch.zeros(1000, device=dev)
    for _ in range(4):
        out = torch._lazy_clone(kept)
        assert torch.equal(op(a, b, out=out), a + b) and not kept.any()
        both = torch._lazy_clone(kept)
        assert torch.equal(op(torch._lazy_clone(a), b, out=both), a + b) and not kept.any()


def test_a_growing_cache_and_a_first_position_that_moves_on():
    """Attention over a row more every time (another signature), and rows stored at another position (a number of `extra`)."""
    import autort
    dev = autort.device()
    q, k, v, f = torch.randn(2, 128, device=dev), torch.randn(20, 2, 128, device=dev), torch.randn(20, 2, 128, device=dev), torch.tensor([0.1], device=dev)
    qkv, inv = torch.randn(3, 3 * 256, device=dev).half(), torch.rand(128, device=dev).half()
    qo, kc, vc = torch.zeros(3, 2, 128, device=dev).half(), torch.zeros(20, 256, device=dev).half(), torch.zeros(20, 256, device=dev).half()
    for _ in range(3):
        for s in range(1, 21):
            want = torch.einsum('hs,shd->hd', torch.softmax(torch.einsum('hd,shd->hs', q, k[:s]) * 0.1, -1), v[:s])
            assert torch.allclose(autort.ops.attention_f32(q, k[:s], v[:s], f), want, rtol=1e-4, atol=1e-5)
        for first in (0, 5, 17, 2.0):
            vc.zero_()
            autort.ops.rope_qkv_store_rows_f16(qkv, inv, qo, kc, vc, extra=[first])
            assert torch.equal(vc[int(first):int(first) + 3], qkv[:, 512:]) and vc.any(1).sum() == 3
        for outside in (18, -1):
            with pytest.raises(RuntimeError):
                autort.ops.rope_qkv_store_rows_f16(qkv, inv, qo, kc, vc, extra=[outside])


@pytest.mark.parametrize('first', [True, False])
def test_calls_run_without_room_for_their_scratch_memory(first):
    """Memory runs out (a limit on what torch may take): a first call and a replayed one take a kernel that needs less, and once there
    is room again the call is as before."""
    import autort
    from antares_amd.runtime import capi
    dev = autort.device()
    print(f'[case] calls without room, first={first}', flush=True)
    n, c, hw, f = 30, 246, 20, 32
    ir = (f'output0[N, F, HO, WO] +=! input0[N, C, HO + KH - 1, WO + KW - 1].when([HO + KH - 1 >= 0, HO + KH - 1 < {hw}, WO + KW - 1 >= 0, WO + KW - 1 < {hw}], 0.0) '
          f'* input1[F, C, KH, KW] where HO in {hw}, WO in {hw}')
    op = autort.export(ir=ir, inputs=[f'input0=float32[N:{n}, C:{c}, H:{hw}, W:{hw}]', f'input1=float32[F:{f}, C:{c}, KH:3, KW:3]'], name=f'conv_room_{int(first)}')
    shape = (0, n, c, hw, hw, f, hw, hw, 1, 1)
    lib = capi.lib()
    form = lib.art_conv2d_choose(*shape)
    assert form & 255 > 3 and lib.art_conv2d_scratch_bytes(*shape, form) > 24 << 20 and lib.art_conv2d_form(*shape, 0)
    g = torch.Generator().manual_seed(3)
    x, w = torch.randn(n, c, hw, hw, generator=g), torch.randn(f, c, 3, 3, generator=g)
    want = torch.nn.functional.conv2d(x[:2].double(), w.double(), padding=1)
    xd, wd, y = x.to(dev), w.to(dev), torch.empty(n, f, hw, hw, device=dev)

    def off():
        got = y[:2].cpu().double()
        y.zero_()
        return float((got - want).norm() / want.norm())
    if not first:
        for _ in range(2):
            op(xd, wd, out=y)
        assert off() < 1e-6
    try:
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        # room for the filter (a block of 2 MiB) and no copy of the image
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (8 << 20)) / torch.cuda.get_device_properties(dev).total_memory)
        held = []
        with pytest.raises(torch.OutOfMemoryError):            # what is left in blocks of 24 MiB is taken
            while len(held) < 1000:
                held.append(torch.empty(24 << 20, dtype=torch.uint8, device=dev))
        for _ in range(2):
            op(xd, wd, out=y)
            assert off() < 1e-6
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    op(xd, wd, out=y)
    usual = y.clone()
    op(xd, wd, out=y)
    assert torch.equal(y, usual) and off() < 1e-6
