"""fp16 GEMM on the matrix cores against the oracle (fp32 accumulate, fp16 out; rtol/atol 1e-2)."""
import numpy as np
import pytest
import torch

from antares_amd import workloads

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures('oracle_built')]
FP16_TOL = dict(rtol=1e-2, atol=1e-2)


@pytest.fixture(scope='module')
def gemm():
    import autort
    from antares_amd.autort import patterns
    return autort, autort.export(ir=patterns.GEMM_F16_IR, inputs=patterns.GEMM_F16_INPUTS, name='gemm_f16')


def oracle_gemm(a, b):
    """fp32-accumulated product of the fp16 operands, rounded to fp16 (float64 sums are exact enough to stand in
    for the fp32 loop nest at these sizes; the oracle's own loop nest is used for the small case below)."""
    return (a.astype(np.float64) @ b.astype(np.float64)).astype(np.float32).astype(np.float16)


def test_small_against_loop_nest_oracle(gemm):
    from antares_amd.autort import patterns
    from antares_amd.ir import parse_program
    from oracle.cpu_backend import CpuModule
    autort, op = gemm
    print('[case] gemm 256x256x64 vs loop nest', flush=True)
    g = torch.Generator().manual_seed(1)
    a = (torch.randn(256, 64, generator=g) * 0.5).half()
    b = (torch.randn(64, 256, generator=g) * 0.5).half()
    want = CpuModule(parse_program(patterns.GEMM_F16_IR, patterns.GEMM_F16_INPUTS), fast_math=False)(a=a.numpy(), b=b.numpy())['c']
    got = op(a.to(autort.device()), b.to(autort.device())).cpu().numpy()
    assert np.allclose(got.astype(np.float32), want.astype(np.float32), **FP16_TOL)


@pytest.mark.parametrize('M,N,K', [(256, 256, 64), (256, 512, 128), (512, 256, 192), (1024, 2048, 1024), (4096, 4096, 4096),
                                   # edge tiles: any M, N % 8 == 0
                                   (1, 256, 64), (100, 264, 128), (257, 248, 64), (300, 1000, 192), (64, 4096, 4096), (777, 8, 64)])
def test_against_float64_product(gemm, M, N, K):
    autort, op = gemm
    print(f'[case] gemm {M}x{N}x{K}', flush=True)
    g = torch.Generator().manual_seed(M + N + K)
    a = (torch.randn(M, K, generator=g) * 0.02).half()
    b = (torch.randn(K, N, generator=g) * 0.02).half()
    dev = autort.device()
    got = op(a.to(dev), b.to(dev))
    assert op.fast_path is not None and got.dtype == torch.float16 and got.shape == (M, N)
    want = torch.from_numpy(oracle_gemm(a.numpy(), b.numpy()))
    assert torch.allclose(got.cpu().float(), want.float(), **FP16_TOL)
    # identity and one-hot structure: pins operand order / transposition
    if M == N == 256:
        eye = torch.eye(256, dtype=torch.float16)
        bb = (torch.randn(256, 256, generator=g)).half()
        f = autort.export(ir=op.ir, inputs=['a=float16[M:256, K:256]', 'b=float16[K:256, N:256]'], name='gemm_f16_sq')
        assert torch.equal(f(eye.to(dev), bb.to(dev)).cpu(), bb)
        assert torch.equal(f(bb.to(dev), eye.to(dev)).cpu(), bb)


@pytest.mark.parametrize('threads', [256, 512])
@pytest.mark.parametrize('M,N,K', [(256, 256, 64), (300, 1000, 192), (1024, 2048, 1024), (4096, 4096, 1024)])
def test_both_block_shapes_against_float64_product(gemm, threads, M, N, K):
    """`art_gemm_f16_tuned`: the 256 x 256 tile worked by 2 x 2 wavefronts (256 threads) or by 2 x 4 (512 threads) -
    the launch parameter `tune:N` searches; the library's own choice is 256 threads."""
    from ctypes import c_void_p
    from antares_amd.runtime import capi
    autort, _ = gemm
    print(f'[case] art_gemm_f16_tuned threads={threads} {M}x{N}x{K}', flush=True)
    g = torch.Generator().manual_seed(M + N + K + threads)
    a = (torch.randn(M, K, generator=g) * 0.02).half()
    b = (torch.randn(K, N, generator=g) * 0.02).half()
    dev = autort.device()
    capi.init(dev.index or 0)
    ad, bd = a.to(dev), b.to(dev)
    c = torch.empty(M, N, dtype=torch.float16, device=dev)
    capi.check(capi.lib().art_gemm_f16_tuned(c_void_p(ad.data_ptr()), c_void_p(bd.data_ptr()), c_void_p(c.data_ptr()), M, N, K, threads,
                                             c_void_p(torch.cuda.current_stream().cuda_stream)))
    want = torch.from_numpy(oracle_gemm(a.numpy(), b.numpy()))
    assert torch.allclose(c.cpu().float(), want.float(), **FP16_TOL)
    other = torch.empty_like(c)
    capi.check(capi.lib().art_gemm_f16_tuned(c_void_p(ad.data_ptr()), c_void_p(bd.data_ptr()), c_void_p(other.data_ptr()), M, N, K,
                                             768 - threads, c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert torch.equal(c, other)            # same k order per output: the two shapes agree bit for bit
    assert capi.lib().art_gemm_f16_tuned(c_void_p(ad.data_ptr()), c_void_p(bd.data_ptr()), c_void_p(c.data_ptr()), M, N, K, 128,
                                         c_void_p(0)) != 0


def test_shapes_the_kernel_does_not_take_use_the_generic_lowering(gemm):
    """K % 64 != 0 (or N % 8 != 0) is left to the generic reduce lowering."""
    autort, op = gemm
    print('[case] gemm 96x80x40 (generic lowering)', flush=True)
    g = torch.Generator().manual_seed(5)
    a = (torch.randn(96, 40, generator=g) * 0.1).half()
    b = (torch.randn(40, 80, generator=g) * 0.1).half()
    got = op(a.to(autort.device()), b.to(autort.device())).cpu().numpy()
    assert np.allclose(got.astype(np.float32), oracle_gemm(a.numpy(), b.numpy()).astype(np.float32), **FP16_TOL)


def test_8192_cubed_through_a_random_projection(gemm):
    """The larger benchmark size, checked by a property that needs O(n^2) work on the host:
    (A B) v = A (B v) for a random v, in float64 from the fp16 operands and the fp16 result."""
    autort, op = gemm
    n = 8192
    print(f'[case] gemm {n}^3 projection', flush=True)
    a, b = workloads.gemm_inputs(3, n)
    dev = autort.device()
    c = op(a.to(dev), b.to(dev)).cpu()
    g = torch.Generator().manual_seed(9)
    for _ in range(2):
        v = torch.randn(n, generator=g, dtype=torch.float64)
        want = a.double() @ (b.double() @ v)
        got = c.double() @ v
        # every element of C carries a relative rounding error of 2^-11; over a row of n random terms they add up to
        # about sqrt(n) * 2^-11 * |c| * |v| - three times that is the bound
        bound = 3 * (n ** 0.5) * 2.0 ** -11 * c.double().abs().mean() * v.abs().mean() * 1.3
        assert (got - want).abs().max() < bound, ((got - want).abs().max(), bound)
    # and the rows and columns are where they belong: two single-row / single-column spot checks in float64
    i, j = 1234, 4321
    assert abs(float(c[i, j]) - float(a[i].double() @ b[:, j].double())) < 1e-2 * max(1.0, abs(float(c[i, j])))
    assert abs(float(c[n - 1, 0]) - float(a[n - 1].double() @ b[:, 0].double())) < 1e-2 * max(1.0, abs(float(c[n - 1, 0])))


TILE_TYPES = {'float16': (0, 64), 'float32': (1, 32), 'int8': (2, 128)}      # dtype -> (kind, values of k in a chunk)


def _tile_operands(dtype, M, N, K, dev, offset):
    """Operands at an address that is aligned to nothing but the element (offset odd), and the float64 / int64 product with
    the sum of the products' magnitudes."""
    g = torch.Generator().manual_seed(M + N + K)
    if dtype == 'int8':
        a, b = torch.randint(-128, 128, (M, K), generator=g, dtype=torch.int8), torch.randint(-128, 128, (N, K), generator=g, dtype=torch.int8)
        want, size = a.double() @ b.double().t(), None
    else:
        t = getattr(torch, dtype)
        a, b = torch.randn(M, K, generator=g).to(t), torch.randn(K, N, generator=g).to(t)
        want, size = a.double() @ b.double(), a.double().abs() @ b.double().abs()

    def put(x):
        room = torch.empty(x.numel() + offset, dtype=x.dtype, device=dev)[offset:].view(x.shape)
        room.copy_(x)
        return room
    return put(a), put(b), want, size


@pytest.mark.parametrize('dtype', list(TILE_TYPES))
# one tile, a row / column / value of k more or less than a tile, the shortest k, the narrowest N, several chunks and slices
@pytest.mark.parametrize('M,N,chunks,rest', [(64, 64, 1, 0), (65, 63, 1, 1), (63, 129, 2, -1), (1, 17, 0, 16), (130, 129, 5, 3), (257, 66, 7, 0), (128, 128, 4, 17),
                                             (200, 1000, 3, 9)])
def test_tile_products_of_every_form(dtype, M, N, chunks, rest):
    """`art_gemm_tile`: every form and several numbers of slices against the 64-bit product.  Bounds: int8 exact; float32 sums of
    at most 32 + chunks + slices terms in a row, each addition off by 2^-24 of the magnitudes; float16 the same over all of K,
    and the result's own rounding (2^-11)."""
    import autort
    from ctypes import c_void_p
    from antares_amd.runtime import capi
    kind, per = TILE_TYPES[dtype]
    K = chunks * per + rest
    dev = autort.device()
    capi.init(dev.index or 0)
    lib = capi.lib()
    a, b, want, size = _tile_operands(dtype, M, N, K, dev, 1)
    total = (K + per - 1) // per
    for form in (1, 2, 3, 4):
        for slices in sorted({1, 2, 3, total}):
            if not lib.art_gemm_tile_form(kind, M, N, K, 0, form, slices):
                assert form == (3 if kind == 1 else 4) or slices > total
                continue
            print(f'[case] art_gemm_tile {dtype} {M}x{N}x{K} form {form} slices {slices}', flush=True)
            c = torch.zeros(M, N, dtype=torch.int32 if kind == 2 else getattr(torch, dtype), device=dev)
            partial = torch.full((slices * M * N,), -7, dtype=torch.int32, device=dev)      # NaN as float32: nothing is read before it is written
            capi.check(lib.art_gemm_tile(*(c_void_p(t.data_ptr()) for t in (a, b, c, partial)), kind, M, N, K, form, slices,
                                         c_void_p(torch.cuda.current_stream().cuda_stream)))
            got = c.cpu().double()
            if kind == 2:
                assert torch.equal(got, want)
            elif kind == 1:
                assert bool(((got - want).abs() <= (32 + total + slices) * 2.0 ** -24 * size).all())
            else:
                assert bool(((got - want).abs() <= (K + slices) * 2.0 ** -24 * size + 2.0 ** -11 * want.abs() + 2.0 ** -24).all())


# rows of tiles, as many columns as rows, columns whose eighths are and are not whole vectors; 16 tiles and numbers that are no multiple of eight
@pytest.mark.parametrize('M,N', [(1100, 67), (1027, 64), (250, 255), (65, 1000), (130, 644), (64, 1021), (70, 4096)])
@pytest.mark.parametrize('dtype', list(TILE_TYPES))
def test_sliced_tile_products_of_sixteen_tiles_and_more(dtype, M, N):
    """Slices that are numbered by tile and added by eighths of the rows or of the columns, as above: int8 exact, the others within their bounds."""
    from ctypes import c_void_p
    from antares_amd.runtime import capi
    capi.init(0)
    dev, lib = torch.device('cuda', 0), capi.lib()
    kind, per = TILE_TYPES[dtype]
    K = 7 * per + 16 // (2, 4, 1)[kind]
    a, b, want, size = _tile_operands(dtype, M, N, K, dev, 1)
    for form, slices in ((1, 2), (1, 8), (2, 3)):
        print(f'[case] art_gemm_tile {dtype} {M}x{N}x{K} form {form} slices {slices}', flush=True)
        c = torch.zeros(M, N, dtype=torch.int32 if kind == 2 else getattr(torch, dtype), device=dev)
        partial = torch.full((slices * M * N,), -7, dtype=torch.int32, device=dev)          # NaN as float32
        capi.check(lib.art_gemm_tile(*(c_void_p(t.data_ptr()) for t in (a, b, c, partial)), kind, M, N, K, form, slices,
                                     c_void_p(torch.cuda.current_stream().cuda_stream)))
        got = c.cpu().double()
        if kind == 2:
            assert torch.equal(got, want)
        elif kind == 1:
            assert bool(((got - want).abs() <= (32 + 8 + slices) * 2.0 ** -24 * size).all())
        else:
            assert bool(((got - want).abs() <= (K + slices) * 2.0 ** -24 * size + 2.0 ** -11 * want.abs() + 2.0 ** -24).all())


# on both sides of what an XCD's L2 holds (an eighth of the longer operand and the other: 4 MiB, float32 6), and of the widths whose columns are cut
@pytest.mark.parametrize('M,N,K', [('L2', 0, 0), ('L2', 0, 64), ('L2', 1, 0), ('L2', 1, 64), (64, 768, 704), (64, 784, 704), (64, 796, 700), (64, 800, 704), (130, 640, 715)])
@pytest.mark.parametrize('dtype', list(TILE_TYPES))
def test_sliced_tile_products_numbered_by_tile_and_by_slice(dtype, M, N, K):
    """As above: int8 exact, the others within their bounds."""
    from ctypes import c_void_p
    from antares_amd.runtime import capi
    capi.init(0)
    dev, lib = torch.device('cuda', 0), capi.lib()
    kind, per = TILE_TYPES[dtype]
    if M == 'L2':
        most, (M, N) = (4 << 20, 6 << 20, 4 << 20)[kind] // (2, 4, 1)[kind], ((576, 192), (192, 832))[N]
        K += most // (max(M, N) // 8 + min(M, N)) // 16 * 16
    a, b, want, size = _tile_operands(dtype, M, N, K, dev, 1)
    for form, slices in ((1, 2), (1, 5), (2, 3)):
        print(f'[case] art_gemm_tile {dtype} {M}x{N}x{K} form {form} slices {slices}', flush=True)
        c = torch.zeros(M, N, dtype=torch.int32 if kind == 2 else getattr(torch, dtype), device=dev)
        partial = torch.full((slices * M * N,), -7, dtype=torch.int32, device=dev)          # NaN as float32
        capi.check(lib.art_gemm_tile(*(c_void_p(t.data_ptr()) for t in (a, b, c, partial)), kind, M, N, K, form, slices,
                                     c_void_p(torch.cuda.current_stream().cuda_stream)))
        got = c.cpu().double()
        if kind == 2:
            assert torch.equal(got, want)
        elif kind == 1:
            assert bool(((got - want).abs() <= (32 + (K + 31) // 32 + slices) * 2.0 ** -24 * size).all())
        else:
            assert bool(((got - want).abs() <= (K + slices) * 2.0 ** -24 * size + 2.0 ** -11 * want.abs() + 2.0 ** -24).all())


@pytest.mark.parametrize('chunks,rest', [(1, 0), (2, 3), (3, 0), (4, -1), (7, 5)])
def test_tile_products_of_more_blocks_than_compute_units(chunks, rest):
    """float16 puts the next chunk into LDS in front of the products with up to 256 blocks, behind them with more: the same sums in
    the same order, so the rows that 16 x 16 and 18 x 16 tiles share are the same bit for bit, and within the bound of the other forms
    (every addition off by 2^-24 of the magnitudes, one rounding to float16)."""
    from ctypes import c_void_p
    from antares_amd.runtime import capi
    capi.init(0)
    dev, N, K = torch.device('cuda', 0), 1000, 64 * chunks + rest
    a, b, want, size = _tile_operands('float16', 1100, N, K, dev, 1)
    results = []
    for M in (1000, 1100):
        print(f'[case] art_gemm_tile float16 {M}x{N}x{K} form 1', flush=True)
        c = torch.full((M, N), float('nan'), dtype=torch.float16, device=dev)
        capi.check(capi.lib().art_gemm_tile(c_void_p(a.data_ptr()), c_void_p(b.data_ptr()), c_void_p(c.data_ptr()), None, 0, M, N, K, 1, 1,
                                            c_void_p(torch.cuda.current_stream().cuda_stream)))
        results.append(c.cpu())
    assert torch.equal(results[0], results[1][:1000])
    assert ((results[1].double() - want).abs() <= size * (K * 2.0 ** -24) + want.abs() * 2.0 ** -11 + 2.0 ** -24).all()


@pytest.mark.parametrize('dtype,M,N,K', [('float16', 78, 207, 582), ('float16', 448, 704, 2368), ('float16', 144, 160, 104), ('float32', 248, 120, 1616),
                                         ('float32', 192, 576, 192), ('float32', 70, 420, 268), ('int8', 232, 120, 1448), ('int8', 112, 3568, 72),
                                         # thin or short: the generic kernels sum on the vector units however many tiles there are
                                         ('float32', 16, 2048, 512), ('float32', 8, 4096, 256), ('float32', 3, 4096, 512), ('float32', 20000, 24, 130),
                                         ('float32', 900, 1200, 28),
                                         # large, with rows that are not whole vectors
                                         ('float16', 2100, 8001, 70), ('int8', 4097, 4099, 80)])
def test_small_products_take_the_tile_kernel_and_agree_with_the_generic_kernels(dtype, M, N, K):
    """The route of an exported program: the call goes to `art_gemm_tile`, agrees with the generic kernels (int8 bit for bit), and
    in float32 is no further from the 64-bit product than they are."""
    import autort
    from antares_amd.autort import patterns
    from antares_amd.runtime import capi
    dev = autort.device()
    print(f'[case] tile route {dtype} {M}x{N}x{K}', flush=True)
    ir, inputs = {'float16': (patterns.GEMM_F16_IR, patterns.GEMM_F16_INPUTS), 'float32': (patterns.GEMM_F32_IR, patterns.GEMM_F32_INPUTS),
                  'int8': ('o[N, M] +=! x[N, K].cast(`int32`) * y[M, K].cast(`int32`)', ['x=int8[N:64, K:64]', 'y=int8[M:64, K:64]'])}[dtype]
    a, b, want, _ = _tile_operands(dtype, M, N, K, dev, 0)
    kind = TILE_TYPES[dtype][0]
    assert capi.lib().art_gemm_tile_form(kind, M, N, K, 0, 0, 0)
    results = []
    for generic in (False, True):
        op = autort.export(ir=ir, inputs=inputs, name=f'tile_{dtype}_{int(generic)}')
        if generic:
            op.fast_path = None
        else:
            assert op.fast_path is not None
        results.append(op(a, b).cpu().double())
    got, old = results
    if kind == 2:
        assert torch.equal(got, old) and torch.equal(got, want)
    else:
        off = [float((r - want).norm() / want.norm()) for r in results]
        assert off[0] <= (1e-3 if kind == 0 else 1.05 * off[1]), off
