"""Which calls the handlers of hand-written kernels take, decided on the host: no GPU."""
import pytest
import torch

from antares_amd.autort import patterns
from antares_amd.autort.op import ExportedOp
from antares_amd.runtime import capi

CONV = ('output0[N, F, HO, WO] +=! input0[N, C, HO + KH - 1, WO + KW - 1].when([HO + KH - 1 >= 0, HO + KH - 1 < 28, WO + KW - 1 >= 0, '
        'WO + KW - 1 < 28], 0.0) * input1[F, C, KH, KW] where HO in 28, WO in 28')
CONV_INPUTS = ['input0=float32[N:4, C:64, H:28, W:28]', 'input1=float32[F:64, C:64, KH:3, KW:3]']


class GpuShaped(torch.Tensor):
    """Dtype, shape and device of a GPU tensor, without one."""

    @staticmethod
    def __new__(cls, shape):
        return torch.Tensor._make_wrapper_subclass(cls, shape, dtype=torch.float32, device='cuda:0')

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        raise NotImplementedError(func)


class Launches:
    def __init__(self):
        self.taken = []

    def library(self, fn, *args):
        self.taken.append(fn.__name__)


def taken_by(op, *tensors):
    """What the hand-written kernel's handler launches for these tensors; [] when it leaves the call to the generic kernels."""
    bound = dict(zip(op.declared + op.fresh_outputs, tensors))
    env = op.fused.bind_dims({n: tuple(bound[n].shape) for n in op._declared_in_graph})
    call = Launches()
    ran = op.fast_path(op, bound, env, call)
    assert ran == bool(call.taken)
    return call.taken


@pytest.mark.parametrize('spec,shape,dense', [
    (None, (4, 64, 28, 28), True), (None, (4 * 64 * 28 * 28,), True),                # the program's own result, in any shape
    ('output0=float32[4, 64, 28, 28]', (4, 64, 28, 28), True),
    ('output0=float32[N:4, F:64, A:32, B:28]', (4, 64, 32, 28), False), ('output0=float32[N:4, F:64, A:28, B:32]', (4, 64, 28, 32), False),
    ('output0=float32[N:4, F:64, A:32, B:28]', (4, 64, 28, 28), True),              # of the size of the result in this call
    ('output0=float32[5, 64, 28, 28]', (5, 64, 28, 28), False), ('output0=float32[4, 65, 28, 28]', (4, 65, 28, 28), False)])
def test_a_convolution_into_part_of_a_larger_result_is_left_to_the_generic_kernels(spec, shape, dense):
    op = ExportedOp(CONV, CONV_INPUTS + ([spec] if spec else []), name='conv_part')
    x, w, y = torch.zeros(4, 64, 28, 28), torch.zeros(64, 64, 3, 3), torch.zeros(shape)
    assert taken_by(op, x, w, y) == (['art_conv2d'] if dense else [])


@pytest.mark.parametrize('spec,shape,fits', [
    ('output0=float32[N, F, A, B]', (4, 64, 28, 28), True), ('output0=float32[N, F, A, B]', (4, 64, 30, 29), True),
    ('output0=float32[N, F, A, B]', (4, 64, 27, 28), False), ('output0=float32[N, F, A, B]', (4, 64, 28, 27), False),
    ('output0=float32[4, 64, 28, 20]', (4, 64, 28, 20), False), ('output0=float32[3, 64, 28, 28]', (3, 64, 28, 28), False)])
def test_a_declared_result_too_small_for_the_program_is_refused(monkeypatch, spec, shape, fits):
    class Checked(Exception):
        pass

    def init(device):
        raise Checked
    monkeypatch.setattr(capi, 'init', init)              # what follows the checks
    op = ExportedOp(CONV, CONV_INPUTS + [spec], name='conv_room')
    with pytest.raises(Checked if fits else ValueError):
        op._call(None, *(GpuShaped(s) for s in ((4, 64, 28, 28), (64, 64, 3, 3), shape)))


@pytest.mark.parametrize('K', [4, 31, 32, 63, 64, 512])
def test_float32_products_on_the_vector_units_keep_short_sums(K):
    """Where the generic lowering spreads k over a wavefront or a block (its launch plan says so), its sums are short: the tile kernel
    takes such a product with its short sums (form 4) or not at all, whatever an older module file has kept; elsewhere without them."""
    lib = capi.lib()
    op = ExportedOp(patterns.GEMM_F32_IR, patterns.GEMM_F32_INPUTS, name='gemm_thin')
    plan, sizes = op.plans[0], (1, 8, 31, 32, 33, 63, 64, 65, 255, 1000, 4096, 16384)

    class Codes(Launches):
        def library(self, fn, *args):
            self.taken.append(256 * args[-3] + args[-2])
    for M in sizes:
        for N in sizes[1:]:
            own, code = lib.art_gemm_tile_form(1, M, N, K, 0, 0, 1), lib.art_gemm_tile_form(1, M, N, K, 0, 0, 0)
            short = plan.choose({'M': M, 'N': N, 'K': K}, {n: 0 for n in plan.args})[0].split('_')[-1] in ('w', 'b')
            assert (own >> 8 == 4) == short and own >> 8 and code in (0, own), (M, N, K, own, code)
            if M * N > 1 << 16:
                continue
            op.tuned = {f'gemm_tile.form|1,{M},{K},{N}': {'value': 256 * (1 if short else 4) + 1, 'us': 0.0}}
            call = Codes()
            op.fast_path(op, dict(a=torch.zeros(M, K), b=torch.zeros(K, N), c=torch.zeros(M, N)), {}, call)
            assert call.taken == ([code] if code else []), (M, N, K)


@pytest.mark.parametrize('kind,M,N,K,generic,here', [
    (0, 24, 61, 446, 3.9, 6.2), (0, 1440, 56, 24, 3.3, 4.0), (0, 47, 9, 4106, 4.3, 11.7), (0, 1088, 24, 192, 8.5, 4.3), (0, 8, 3968, 1024, 113, 6.4),
    (0, 8, 128, 7904, 31, 7.6), (1, 64, 6, 832, 3.5, 8.9), (1, 72, 8, 16352, 23, 31), (1, 45, 704, 192, 15.5, 7.7),
    (1, 5, 9920, 5376, 1870, 68), (2, 920, 1, 370, 3.1, 4.6), (2, 31, 2, 6301, 4.2, 8.8), (2, 23, 963, 105, 6.9, 4.1)])
def test_thin_products_go_to_the_kernel_that_was_measured_to_be_faster(kind, M, N, K, generic, here):
    """One of each kind of kernel that the generic lowering has without matrix instructions; times in us on an MI355X."""
    assert bool(capi.lib().art_gemm_tile_form(kind, M, N, K, 0, 0, 0)) == (here < generic)


@pytest.mark.parametrize('kind,M,N,K,generic,here', [
    (0, 4672, 4992, 32, 20.4, 24.9), (0, 2216, 7464, 216, 41.1, 33.6), (0, 7212, 8134, 615, 390, 175), (0, 2028, 15937, 171, 102, 53),
    (2, 4608, 15168, 64, 56, 66), (2, 1856, 3456, 48, 8.2, 9.8), (2, 5369, 3613, 80, 55, 19), (2, 3592, 15416, 48, 114, 42), (2, 4096, 4096, 4096, 106, 98)])
def test_products_that_are_mostly_stores_go_to_the_kernel_that_was_measured_to_be_faster(kind, M, N, K, generic, here):
    """Whole vectors of k and whole lines of results: the generic kernels on the matrix instructions; odd ones: the tile kernel."""
    assert bool(capi.lib().art_gemm_tile_form(kind, M, N, K, 0, 0, 0)) == (here < generic)


@pytest.mark.parametrize('f16', [0, 1])
def test_convolutions_are_taken_by_forms_whose_sums_are_no_longer_than_the_generic_ones(f16):
    """Where the generic lowering has no matrix instructions (its launch plan says so): float32 form 7, float16 blocks of 64 x 64 (any
    block below 64 terms, which are a chain there).  Elsewhere float16 with less than a chunk of channels, not whole eighths of them: blocks of 64 x 64.  Also for a form that a module
    file has kept."""
    lib, dtype = capi.lib(), 'float16' if f16 else 'float32'
    cast = '.to(`float32`)' if f16 else ''
    for n, c, hw, f in ((1, 16, 40, 31), (2, 1, 20, 64), (8, 3, 40, 64), (5, 24, 2, 2424), (1, 208, 4, 1160), (3, 32, 7, 32), (2, 33, 40, 21), (9, 9, 28, 200), (4, 4, 30, 96),
                        (10, 11, 51, 146), (17, 25, 29, 88), (6, 24, 28, 96), (4, 16, 30, 64), (32, 128, 28, 128), (3, 40, 3, 1040)):
        shape = (f16, n, c, hw, hw, f, hw, hw, 1, 1)
        op = ExportedOp(f'o[N, F, HO, WO] +=! x[N, C, HO + KH, WO + KW]{cast} * w[F, C, KH, KW]{cast} where HO in {hw}, WO in {hw}',
                        [f'x={dtype}[N:{n}, C:{c}, H:{hw + 2}, W:{hw + 2}]', f'w={dtype}[F:{f}, C:{c}, KH:3, KW:3]'], name=f'conv_sums_{f16}')
        env = op.fused.bind_dims({'x': (n, c, hw + 2, hw + 2), 'w': (f, c, 3, 3)})
        vector = op.plans[0]._matrix_choice(env)[0] is None
        allowed = [v for v in range(1, 8) if lib.art_conv2d_exact_enough(*shape, v)]
        if vector:
            assert allowed == (list(range(1, 8 - f16)) if c < 8 else [7] if not f16 else [1, 4] if c <= 16 or c % 8 == 0 or c >= 48 else [1]), (shape, allowed)
        elif f16 and c < 32 and c % 8:
            assert allowed == ([1, 4] if c > 4 else []), (shape, allowed)
        else:
            assert set(allowed) >= {1, 2, 3, 4, 5, 6}, (shape, allowed)
        choice = lib.art_conv2d_choose(*shape)
        assert not choice or (choice & 255) in allowed, (shape, choice, allowed)


def test_a_kept_convolution_form_with_longer_sums_is_not_used():
    class Codes(Launches):
        def library(self, fn, *args):
            self.taken.append(args[-2])
    n, c, hw, f = 17, 25, 29, 88
    ir = CONV.replace('28', str(hw)).replace('input0[N, C, HO + KH - 1, WO + KW - 1]', 'input0[N, C, HO + KH - 1, WO + KW - 1].to(`float32`)') \
        .replace('input1[F, C, KH, KW]', 'input1[F, C, KH, KW].to(`float32`)')
    op = ExportedOp(ir, [f'input0=float16[N:{n}, C:{c}, H:{hw}, W:{hw}]', f'input1=float16[F:{f}, C:{c}, KH:3, KW:3]'], name='conv_kept')
    bound = {'input0': torch.zeros(n, c, hw, hw).half(), 'input1': torch.zeros(f, c, 3, 3).half(), 'output0': torch.zeros(n, f, hw, hw)}
    env = op.fused.bind_dims({k: tuple(v.shape) for k, v in bound.items()})
    choice = capi.lib().art_conv2d_choose(1, n, c, hw, hw, f, hw, hw, 1, 1)
    for kept, used in ((5, choice), (1, 1)):
        op.tuned = {f'conv2d.form|1,{n},{c},{hw},{hw},{f},{hw},{hw},1,1': {'value': kept, 'us': 0.0}}
        call = Codes()
        assert op.fast_path(op, bound, env, call) and call.taken == [used]


@pytest.mark.parametrize('f16,n,c,f,hw,generic,here', [
    (0, 1, 24, 32, 15, 7.6, 13.7), (0, 58, 12, 4, 158, 82, 621), (0, 30, 9, 8, 104, 28, 144), (0, 7, 34, 4058, 6, 17, 25), (0, 6, 9, 294, 76, 39, 50),
    (0, 4, 3, 14, 159, 14, 42), (0, 1, 257, 1658, 1, 8.1, 34), (1, 63, 20, 4, 90, 59, 107), (1, 2, 65, 2887, 8, 13.5, 17.7), (1, 10, 3, 2, 151, 7.6, 58),
    (0, 2, 232, 24, 52, 375, 37), (0, 205, 40, 24, 33, 6457, 213), (0, 9, 216, 64, 17, 23, 20), (0, 8, 3, 105, 42, 14.9, 10.7), (1, 28, 40, 16, 42, 319, 19),
    (1, 9, 240, 104, 13, 19, 13.8), (1, 197, 19, 80, 24, 51, 36), (1, 40, 3, 50, 87, 159, 74), (1, 32, 128, 128, 28, 40, 18.5)])
def test_convolutions_go_to_the_kernel_that_was_measured_to_be_faster(f16, n, c, f, hw, generic, here):
    """Few channels, features or points and very many of them; times in us on an MI355X."""
    assert bool(capi.lib().art_conv2d_choose(f16, n, c, hw, hw, f, hw, hw, 1, 1)) == (here < generic)


@pytest.mark.parametrize('f16,n,c,f,hw,before,direct', [
    (0, 4, 40, 104, 8, 12.9, 4.6), (0, 2, 232, 24, 52, 35.8, 20.9), (0, 1, 24, 32, 15, 7.6, 4.2), (1, 1, 104, 176, 9, 9.4, 5.4), (1, 32, 128, 128, 28, 18.4, 60),
    (0, 11, 176, 104, 34, 63, 92), (1, 26, 120, 32, 37, 19, 36)])
def test_convolutions_in_one_launch_where_that_was_measured_to_be_faster(f16, n, c, f, hw, before, direct):
    """Few products; times in us on an MI355X."""
    assert bool(capi.lib().art_conv2d_direct(f16, n, c, hw, hw, f, hw, hw, 1, 1)) == (direct < before)


@pytest.mark.parametrize('f16,n,c,f,h,w,before,direct', [
    (1, 47, 80, 11, 16, 104, 34.6, 59.9), (1, 72, 88, 4, 14, 103, 46.8, 79.9), (1, 95, 88, 1, 16, 83, 40.5, 58.9), (1, 37, 80, 2, 3, 97, 10.8, 13.1),
    (0, 22, 88, 10, 116, 65, 333, 136), (0, 87, 36, 6, 3, 63, 35.3, 14.5)])
def test_convolutions_of_wide_images_in_one_launch_where_that_was_measured_to_be_faster(f16, n, c, f, h, w, before, direct):
    """Blocks of which a compute unit holds two; times in us on an MI355X."""
    assert bool(capi.lib().art_conv2d_direct(f16, n, c, h, w, f, h, w, 1, 1)) == (direct < before)


@pytest.mark.parametrize('f16,n,c,hw,forms', [(1, 2, 8, 9, [8, 9, 10]), (1, 2, 12, 9, []), (0, 2, 12, 9, [8, 9, 10]), (0, 2, 6, 9, []), (0, 2, 8, 100, [8, 9]), (0, 2, 8, 110, [8]),
                                              (0, 2, 8, 120, []), (0, 1, 8, 15, [8, 9, 10])])
def test_convolutions_in_one_launch_take_whole_pieces_of_the_filter_and_short_runs(f16, n, c, hw, forms):
    """A feature's taps in 16-byte pieces; runs of four points per lane at the most: a block's own, two rows and a bit."""
    assert [v for v in (8, 9, 10) if capi.lib().art_conv2d_form(f16, n, c, hw, hw, 32, hw, hw, 1, 1, v)] == forms


@pytest.mark.parametrize('form', [-8, 11, 12, 40, 41, 255, 256 + 8, 256 + 40, 512 + 10, 1 << 30])
@pytest.mark.parametrize('f16', [0, 1])
def test_convolutions_refuse_forms_that_there_are_not(f16, form):
    """No entry works with a number that names no form (a shift by the difference to 8 is as long as one likes)."""
    lib, shape = capi.lib(), (f16, 2, 16, 9, 9, 32, 9, 9, 1, 1)
    assert lib.art_conv2d_form(*shape, form) == lib.art_conv2d_exact_enough(*shape, form) == lib.art_conv2d_scratch_bytes(*shape, form) == 0
    assert lib.art_conv2d(None, None, None, None, *shape, form, None) != 0 and f'form {form}' in lib.art_last_error().decode()


@pytest.mark.parametrize('f16,n,c,h,w,f', [(1, 64, 512, 128, 128, 512), (0, 64, 64, 100, 100, 17), (1, 256, 64, 112, 112, 64), (0, 32, 256, 56, 56, 256),
                                           (1, 2, 2048, 14, 14, 2048), (0, 1, 40, 12000, 60, 48), (0, 9, 216, 17, 17, 64)])
def test_convolutions_take_a_bounded_copy_of_the_image(f16, n, c, h, w, f):
    """128 MiB for the copy, whatever the batch (64 more for slices), beside the filter; one image of more is gathered."""
    lib, shape = capi.lib(), (f16, n, c, h, w, f, h, w, 1, 1)
    form = lib.art_conv2d_choose(*shape)
    assert form
    beside = lib.art_conv2d_scratch_bytes(*shape, form) - lib.art_conv2d_packed_bytes(f16, c, f)
    assert beside <= (128 << 20) + (64 << 20 if form >> 8 else 0) + 4096
    assert form <= 3 or -(-c // (32 if f16 else 16)) * (h + 2) * (w + 2) * 64 <= 128 << 20
    gathered = lib.art_conv2d_form(*shape, 0)               # for callers that have no room for a copy
    assert gathered <= 3 and (not gathered or lib.art_conv2d_exact_enough(*shape, gathered)) and (gathered or w > 80 or f < 32)


def test_slices_of_a_product_take_a_bounded_part_of_the_memory():
    """128 MiB at the most, also for a number of slices that a module file has kept."""
    lib = capi.lib()
    for kind, M, N, K in ((0, 2723, 9534, 15561), (1, 7351, 3031, 12535), (1, 3568, 3460, 3723), (2, 3173, 2863, 14926)):
        slices = lib.art_gemm_tile_form(kind, M, N, K, 0, 0, 1) & 255
        assert slices == 1 or slices * M * N * 4 <= 128 << 20

    class Codes(Launches):
        def library(self, fn, *args):
            self.taken.append(256 * args[-3] + args[-2])
    M, N, K = 1200, 1300, 700
    op = ExportedOp(patterns.GEMM_F32_IR, patterns.GEMM_F32_INPUTS, name='gemm_kept')
    bound, choice = dict(a=torch.zeros(M, K), b=torch.zeros(K, N), c=torch.zeros(M, N)), lib.art_gemm_tile_form(1, M, N, K, 0, 0, 0)
    for kept, used in ((256 + 22, choice), (256 + 21, 256 + 21)):
        op.tuned = {f'gemm_tile.form|1,{M},{K},{N}': {'value': kept, 'us': 0.0}}
        call = Codes()
        op.fast_path(op, bound, {}, call)
        assert call.taken == [used]


def test_calls_without_room_for_their_scratch_memory_take_a_form_that_needs_less(monkeypatch):
    """Where memory runs out: a product in one slice, a convolution that gathers its image, then the generic kernels; none of them
    leaves a recipe for later calls."""
    lib, room = capi.lib(), [1 << 40]
    empty = torch.empty

    def limited(count, **kw):
        if count * kw['dtype'].itemsize > room[0]:
            raise torch.OutOfMemoryError('no room')
        return empty(count, **kw)
    monkeypatch.setattr(torch, 'empty', limited)

    class Codes(Launches):
        replay = True

        def library(self, fn, *args):
            self.taken.append(args[-2] if fn.__name__ == 'art_conv2d' else 256 * args[-3] + args[-2])

    def taken(op, bound, env):
        call = Codes()
        return op.fast_path(op, bound, env, call), call.taken, call.replay
    M, N, K = 300, 300, 3000
    code = lib.art_gemm_tile_form(1, M, N, K, 0, 0, 0)
    assert code & 255 > 1
    op, bound = ExportedOp(patterns.GEMM_F32_IR, patterns.GEMM_F32_INPUTS, name='gemm_room'), dict(a=torch.zeros(M, K), b=torch.zeros(K, N), c=torch.zeros(M, N))
    assert taken(op, bound, {}) == (True, [code], True)
    room[0] = 1000
    assert taken(op, bound, {}) == (True, [code & ~255 | 1], False)
    room[0] = 1 << 40
    shape = (0, 4, 64, 28, 28, 64, 28, 28, 1, 1)
    op = ExportedOp(CONV, CONV_INPUTS, name='conv_scratch')
    bound = dict(zip(op.declared + op.fresh_outputs, (torch.zeros(4, 64, 28, 28), torch.zeros(64, 64, 3, 3), torch.zeros(4, 64, 28, 28))))
    env = op.fused.bind_dims({k: tuple(v.shape) for k, v in bound.items()})
    form, gathered = lib.art_conv2d_choose(*shape), lib.art_conv2d_form(*shape, 0)
    assert form & 255 > 3 and 1 <= gathered <= 3
    assert taken(op, bound, env) == (True, [form], True)
    room[0] = lib.art_conv2d_packed_bytes(0, 64, 64)
    assert taken(op, bound, env) == (True, [gathered], False)
    room[0] -= 1
    assert taken(op, bound, env) == (False, [], False)


def test_forms_of_the_int4_product():
    """Every form runs where it is asked for; one that cannot number or address its rows and columns is replaced, and what
    no form takes is refused: offsets of a block's x and of its sums of a K split end below 4 GiB, weights of 4 GiB and more come with two forms."""
    form = capi.lib().art_gemm_w4a16_form
    for code in (1, 2, 4, 5, 8, 9, 10, 11):
        for splits in (1, 3):
            assert form(250, 1024, 1056, 0, 0, 256 * code + splits) == 256 * code + splits
    assert form(64, 4096, 4096, 0, 0, 3) & 255 == 3 and form(64, 4096, 4096, 0, 0, 3) >> 8 in (1, 2)
    assert form(64, 256, 4096, 0, 0, 2304 + 9) == 2304 + 2                                # no more splits than groups
    for code in (3, 6, 7, 12, 255):
        assert form(64, 4096, 4096, 0, 0, 256 * code) == 0
    assert form(64, 4096, 4104, 0, 0, 0) == 0 and form(64, 4160, 4096, 0, 0, 0) == 0 and form(0, 4096, 4096, 0, 0, 0) == 0
    assert form(257, 1024, 1056, 0, 0, 2304 + 1) >> 8 not in (0, 9) and form(512, 1024, 1056, 0, 0, 2816 + 1) == 2816 + 1
    assert form(4, 384, 1 << 26, 0, 0, 0) == 1024 + 1 and form(4, 384, (1 << 26) + 16, 0, 0, 0) == 0
    assert form(32, (1 << 26) - 128, 16, 0, 0, 256 + 1) == 256 + 1
    assert form(32, 1 << 26, 16, 0, 0, 256 + 1) & 255 > 1 and form(64, 1 << 25, 16, 0, 0, 512 + 1) not in (0, 512 + 1) and form(4, (1 << 26) + 128, 16, 0, 0, 0) == 0
    for code, taken in ((1, 1), (2, None), (5, None), (4, 4), (8, None), (9, None)):
        got = form(200, 256 * 128, 262144, 0, 0, 256 * code + 1)
        assert got and (got == 256 * code + 1) == (taken is not None)
        assert form(200, 255 * 128, 262144, 0, 0, 256 * code + 1) == 256 * code + 1
    assert form(1, 256, 1 << 22, 0, 0, 2048 + 2) == 2048 + 2
    assert form(1, 256, (1 << 22) + 16, 0, 0, 2048 + 2) not in (0, 2048 + 2)


def test_int4_products_take_the_blocks_that_are_fastest_over_weights_from_hbm():
    """Sizes where the estimates of two forms are close and one of them is far slower with a model's weights: two blocks of 32 rows
    that unpack the same weights against one of 64 (64 rows over 11008 x 4096 18.5 us and 15.9), and narrow blocks over all of K of rows
    whole KiB apart (8 rows over 4096 x 4096 10.1 and 7.8 us, over 5120 x 5120 14.0 and 9.2).  Where the narrow blocks are faster they stay."""
    form = capi.lib().art_gemm_w4a16_form
    assert form(64, 11008, 4096, 0, 0, 0) >> 8 == 2
    for residual in (0, 1):
        assert form(64, 4096, 12288, 0, residual, 0) >> 8 == 2 and form(250, 11008, 4096, 0, residual, 0) >> 8 == 5
        assert form(8, 4096, 4096, 0, residual, 0) & 255 > 1 and form(8, 5120, 5120, 0, residual, 0) & 255 > 1
    assert form(16, 1024, 1024, 0, 0, 0) == 2304 + 1 and form(16, 1024, 4096, 0, 0, 0) == 2304 + 1 and form(16, 4096, 11008, 0, 0, 0) == 2560 + 1
    # a pass that turns or gates adds more than eight K-splits in two trips to memory (19 rows over 6016 x 384 9.9 us, in eight splits 6.4)
    assert form(19, 6016, 384, 2, 0, 0) & 255 <= 8 and form(32, 6528, 384, 2, 0, 0) & 255 <= 8
