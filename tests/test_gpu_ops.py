"""GPU parity tests: every operator is called through the autort surface (which
goes through the C-ABI library) and compared with the CPU oracle on the same
seeded inputs.  Integer results must be bit-exact; fp32 within 1e-5, fp16
within rtol 1e-2 / atol 1e-2."""
import sys

import numpy as np
import pytest
import torch

from antares_amd import workloads

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures('oracle_built')]

FP32_TOL = dict(rtol=1e-5, atol=1e-5)
FP16_TOL = dict(rtol=1e-2, atol=1e-2)


@pytest.fixture(scope='module')
def autort():
    import autort as mod
    assert torch.cuda.is_available(), 'these tests need the GPU'
    return mod


def note(msg):
    print(f'[case] {msg}', flush=True)
    sys.stdout.flush()


SIGMOID_IR = 'sigmoid_f32[N] = 1 - 1 / (1 + data[N].call(strs.exp))'


def test_sigmoid_readme_example(autort):
    note('sigmoid N=10')
    f = autort.export(ir=SIGMOID_IR, inputs=['data=float32[N:4096000]'], config='tune:5')
    data = torch.arange(0, 10, dtype=torch.float32, device=autort.device())
    want = [0.5000, 0.7311, 0.8808, 0.9526, 0.9820, 0.9933, 0.9975, 0.9991, 0.9997, 0.9999]
    assert np.allclose(f(data).cpu().numpy(), want, atol=5e-5)
    assert np.allclose(autort.ops.sigmoid_f32(data).cpu().numpy(), want, atol=5e-5)


@pytest.mark.parametrize('n', [0, 1, 3, 4, 5, 1023, 4_096_000, 4_096_003])
def test_sigmoid_matches_oracle(autort, n):
    from oracle import hot_ops
    note(f'sigmoid N={n}')
    f = autort.export(ir=SIGMOID_IR, inputs=['data=float32[N:4096000]'])
    x = workloads.sigmoid_input(7, n)
    got = f(x.to(autort.device())).cpu().numpy()
    assert got.shape == (n,)
    assert np.allclose(got, hot_ops.sigmoid_f32(x.numpy()), **FP32_TOL)


def test_sigmoid_unaligned_view(autort):
    from oracle import hot_ops
    note('sigmoid on a view that is not 16-byte aligned')
    f = autort.export(ir=SIGMOID_IR, inputs=['data=float32[N:4096000]'])
    x = workloads.sigmoid_input(8, 10_001)
    xd = x.to(autort.device())
    out = torch.zeros(10_001, dtype=torch.float32, device=autort.device())
    f(xd[1:], out=out[1:])
    assert np.allclose(out[1:].cpu().numpy(), hot_ops.sigmoid_f32(x.numpy()[1:]), **FP32_TOL)
    assert float(out[0]) == 0.0


def run_sort_sample(autort, x: torch.Tensor) -> torch.Tensor:
    """samples/01_sort_even_first.py:16-27 verbatim in structure."""
    autort.export(ir='space[data[N] % 2, N] = 1', inputs=['data=int32[N]', 'space=int32[2, N]'],
                  config='~N~:[1,256,1]', name='my_classify_i32')
    autort.export(ir='output[ids[N] - 1] = (val[N % val.size(0)]).when(ids[N] > 0)',
                  inputs=['ids=int32[N]', 'val=int32[M]', 'output=int32[M]'], config='~N~:[1,256,1]', name='my_bucket_i32')
    y = torch.zeros([2, x.size(0)], dtype=torch.int32, device=x.device)
    autort.ops.my_classify_i32(x, y)
    ids = torch.cumsum(y.view(-1), 0, dtype=y.dtype) * y.view(-1)
    output = torch.zeros_like(x)
    autort.ops.my_bucket_i32(ids, x, output)
    return output


def test_sort_sample_known_answer(autort):
    note('sort sample, README input')
    x = torch.tensor([101, 102, 208, 99, 1, 127, 62, 8, 336, 336], dtype=torch.int32, device=autort.device())
    assert run_sort_sample(autort, x).cpu().tolist() == [102, 208, 62, 8, 336, 336, 101, 99, 1, 127]
    assert autort.ops.partition_even_first_i32(x).cpu().tolist() == [102, 208, 62, 8, 336, 336, 101, 99, 1, 127]


@pytest.mark.parametrize('n', [1, 2, 63, 64, 65, 4095, 4096, 4097, 8191, 8192, 100_003, 1_048_576])
def test_partition_bit_exact(autort, n):
    from oracle import hot_ops
    note(f'partition N={n}')
    x = workloads.partition_input(100 + n, n)
    want = hot_ops.sort_even_first_i32(x.numpy())
    xd = x.to(autort.device())
    assert np.array_equal(autort.ops.partition_even_first_i32(xd).cpu().numpy(), want)
    assert np.array_equal(run_sort_sample(autort, xd).cpu().numpy(), want)


def test_partition_empty_and_degenerate(autort):
    note('partition edge cases')
    dev = autort.device()
    assert autort.ops.partition_even_first_i32(torch.empty(0, dtype=torch.int32, device=dev)).numel() == 0
    ev = torch.arange(0, 20000, 2, dtype=torch.int32, device=dev)
    assert torch.equal(autort.ops.partition_even_first_i32(ev), ev)
    assert torch.equal(autort.ops.partition_even_first_i32(ev + 1), ev + 1)
    # the output may start anywhere on a 4-byte boundary (its 16-byte stores find their own alignment) and nothing
    # outside it is written
    for shift in (1, 2, 3):
        x = workloads.partition_input(shift, 10_007).to(dev)
        backing = torch.full((10_007 + 8,), -7, dtype=torch.int32, device=dev)
        out = backing[shift:shift + 10_007]
        autort.ops.partition_even_first_i32(x, out)
        xc = x.cpu()
        assert torch.equal(out.cpu(), torch.cat([xc[xc % 2 == 0], xc[xc % 2 == 1]]))
        assert (backing[:shift] == -7).all() and (backing[shift + 10_007:] == -7).all()


# one launch up to 65536 values: edges of a wavefront's vectors, of tiles, of the eight tiles that are read at a time, of the range
@pytest.mark.parametrize('n', [1, 2, 5, 255, 257, 4095, 4096, 4097, 32767, 32769, 65533, 65536, 65537])
@pytest.mark.parametrize('shift', [0, 1])
def test_partition_of_few_values_in_one_launch_and_in_two(autort, n, shift):
    from ctypes import c_void_p
    from antares_amd.runtime import capi
    note(f'partition N={n} shift={shift}')
    dev = autort.device()
    autort.ops.partition_even_first_i32(torch.zeros(8, dtype=torch.int32, device=dev))
    x = torch.randint(-2 ** 31, 2 ** 31, (n,), generator=torch.Generator().manual_seed(n), dtype=torch.int64).to(torch.int32)
    xd = x.to(dev)
    for values in (xd, xd & ~1, xd | 1):
        want = torch.cat([values[(values & 1) == 0], values[(values & 1) == 1]]).cpu()
        for blocks in (0, 1024):                 # the library's choice; two launches
            out = torch.full((n + 8,), 7, dtype=torch.int32, device=dev)
            capi.check(capi.lib().art_partition_even_first_i32_tuned(c_void_p(values.data_ptr()), c_void_p(out.data_ptr() + 4 * shift), n, blocks,
                                                                     c_void_p(torch.cuda.current_stream().cuda_stream)))
            got = out.cpu()
            assert torch.equal(got[shift:shift + n], want) and (got[:shift] == 7).all() and (got[shift + n:] == 7).all()


def test_partition_full_size_properties(autort):
    note('partition N=16777216 (size-independent properties)')
    x = workloads.partition_input(2, 16_777_216).to(autort.device())
    out = autort.ops.partition_even_first_i32(x)
    want = torch.cat([x[x % 2 == 0], x[x % 2 == 1]])
    assert torch.equal(out, want)
    # idempotent
    assert torch.equal(autort.ops.partition_even_first_i32(out), out)
    # two calls in a row give the same bits (ticket words are restored)
    assert torch.equal(autort.ops.partition_even_first_i32(x), out)


# ------------------------------------------------------------------ int4 GEMV
def w4_op(autort):
    from antares_amd.autort import patterns
    return autort.export(ir=patterns.W4A16_IR, inputs=patterns.W4A16_INPUTS, name='gemv_w4a16')


@pytest.mark.parametrize('M,K,N', [(1, 128, 16), (1, 256, 64), (2, 384, 144), (3, 1024, 1040), (4, 4096, 512), (8, 512, 256),
                                   (1, 4096, 4096), (1, 4096, 11008), (1, 11008, 4096), (1, 4096, 32000)])
def test_w4a16_gemv_matches_oracle(autort, M, K, N):
    from oracle import hot_ops
    note(f'w4a16 M={M} K={K} N={N}')
    p = workloads.w4_problem(K + N + M, M, K, N)
    f = w4_op(autort)
    assert f.fast_path is not None
    dev = autort.device()
    y = f(p['x'].to(dev), p['qweight'].to(dev), p['scales'].to(dev), p['qzeros'].to(dev))
    torch.cuda.synchronize()
    want = hot_ops.gemm_w4a16(p['x'].numpy(), p['qweight'].numpy(), p['scales'].numpy(), p['qzeros'].numpy())
    assert np.allclose(y.cpu().numpy().astype(np.float32), want.astype(np.float32), **FP16_TOL)
    # second call must see clean ticket words
    y2 = f(p['x'].to(dev), p['qweight'].to(dev), p['scales'].to(dev), p['qzeros'].to(dev))
    assert torch.equal(y, y2)


@pytest.mark.parametrize('M,K,N', [(9, 128, 16), (17, 256, 144), (32, 384, 1040), (33, 1024, 512), (64, 2048, 272),
                                   (100, 512, 4096), (200, 4096, 512),
                                   (64, 4096, 4096), (64, 4096, 11008), (64, 11008, 4096), (64, 4096, 32000)])
def test_w4a16_gemm_matches_oracle(autort, M, K, N):
    """Batches of four rows and more run on the matrix cores (one pass over the weights per 64 rows)."""
    from oracle import hot_ops
    note(f'w4a16 gemm M={M} K={K} N={N}')
    p = workloads.w4_problem(K + N + M, M, K, N)
    f = w4_op(autort)
    assert f.fast_path is not None
    dev = autort.device()
    args = [p[k].to(dev) for k in ('x', 'qweight', 'scales', 'qzeros')]
    y = f(*args)
    torch.cuda.synchronize()
    want = hot_ops.gemm_w4a16(p['x'].numpy(), p['qweight'].numpy(), p['scales'].numpy(), p['qzeros'].numpy())
    assert np.allclose(y.cpu().numpy().astype(np.float32), want.astype(np.float32), **FP16_TOL)
    # K-splits are combined in a fixed order: a second call gives the same bits
    assert torch.equal(y, f(*args))
    # row m of the batch agrees with the same row sent alone through the GEMV kernel
    m = M - 1
    y1 = f(args[0][m:m + 1].contiguous(), *args[1:])
    assert np.allclose(y1.cpu().numpy().astype(np.float32), want[m:m + 1].astype(np.float32), **FP16_TOL)
    # (the GEMM rounds s * (q - z) to fp16 as the oracle does, the GEMV applies s in fp32: both are inside the oracle
    # tolerance, and within half of it of each other)
    assert np.allclose(y1.float().cpu().numpy(), y[m:m + 1].float().cpu().numpy(), rtol=5e-3, atol=5e-3)


@pytest.mark.parametrize('M,K,N', [(4, 512, 256), (5, 1024, 144), (6, 4096, 512), (7, 384, 1040), (8, 4096, 4096)])
def test_w4a16_gemv_entry_point_up_to_eight_rows(autort, M, K, N):
    """`art_gemv_w4a16` takes up to 8 rows (the weights are streamed once per pair of rows); autort.export sends
    4 rows and more to the matrix-core kernel, so the entry point is called directly here."""
    from ctypes import c_void_p
    from antares_amd.runtime import capi
    from oracle import hot_ops
    note(f'art_gemv_w4a16 direct M={M} K={K} N={N}')
    p = workloads.w4_problem(K + N + M, M, K, N)
    dev = autort.device()
    capi.init(dev.index or 0)
    x, q, s_, z = (p[k].to(dev) for k in ('x', 'qweight', 'scales', 'qzeros'))
    y = torch.empty(M, N, dtype=torch.float16, device=dev)
    stream = torch.cuda.current_stream().cuda_stream
    capi.check(capi.lib().art_gemv_w4a16(c_void_p(x.data_ptr()), c_void_p(q.data_ptr()), c_void_p(s_.data_ptr()),
                                         c_void_p(z.data_ptr()), c_void_p(y.data_ptr()), M, K, N, c_void_p(stream)))
    torch.cuda.synchronize()
    want = hot_ops.gemm_w4a16(p['x'].numpy(), p['qweight'].numpy(), p['scales'].numpy(), p['qzeros'].numpy())
    assert np.allclose(y.cpu().numpy().astype(np.float32), want.astype(np.float32), **FP16_TOL)


@pytest.mark.parametrize('poison', [float('nan'), float('inf'), 60000.0])
def test_gemv_with_non_finite_rows_stays_clean(autort, poison):
    """A NaN, an infinity or values that overflow the sum in x must come out as non-finite results (the reference's
    float sums propagate them) and must not leave anything behind in the split-K slots: the same operator called
    on ordinary data right afterwards gives the ordinary answer."""
    from antares_amd.autort import patterns
    from oracle import hot_ops
    note(f'w4a16 / gptq gemv with x poisoned by {poison}')
    dev = autort.device()
    K, N = 4096, 1024
    p = workloads.w4_problem(77, 1, K, N)
    f = w4_op(autort)
    args = [p[k].to(dev) for k in ('x', 'qweight', 'scales', 'qzeros')]
    good = f(*args)
    bad_x = args[0].clone()
    if poison == 60000.0:
        bad_x[:] = poison                        # finite, but every partial sum is far outside fp16
    else:
        bad_x[0, 1000] = poison
    bad = f(bad_x, *args[1:])
    if poison != 60000.0:
        assert not torch.isfinite(bad).any()
    again = f(*args)
    assert torch.equal(again, good)
    want = hot_ops.gemm_w4a16(p['x'].numpy(), p['qweight'].numpy(), p['scales'].numpy(), p['qzeros'].numpy())
    assert np.allclose(again.cpu().numpy().astype(np.float32), want.astype(np.float32), **FP16_TOL)
    # the sample's own program (fp32, GPTQ words)
    g = torch.Generator().manual_seed(5)
    q = torch.randint(0, 16, (K, N), generator=g)
    s = torch.rand(K // 128, N, generator=g) * 0.019 + 0.001
    x = torch.randn(K, generator=g)
    h = autort.export(ir=patterns.GPTQ_GEMV_IR, inputs=patterns._gptq_inputs('float32', 'float32'))
    qw = workloads.pack_gptq(q).to(dev)
    good = h(x.to(dev), qw, s.to(dev)).clone()
    bad_x = x.clone()
    if poison == 60000.0:
        bad_x[:] = 1e30                          # the sums are beyond what a split-K slot carries: reported as NaN
    else:
        bad_x[17] = poison
    bad = h(bad_x.to(dev), qw, s.to(dev))
    assert not torch.isfinite(bad).any()
    assert torch.equal(h(x.to(dev), qw, s.to(dev)), good)


def test_w4a16_generic_lowering_agrees(autort):
    """The same program through the generic reduce lowering (no hand kernel)."""
    from oracle import hot_ops
    note('w4a16 through the generic lowering')
    p = workloads.w4_problem(9, 2, 256, 64)
    f = w4_op(autort)
    dev = autort.device()
    bound = {'x': p['x'].to(dev), 'qweight': p['qweight'].to(dev), 'scales': p['scales'].to(dev), 'qzeros': p['qzeros'].to(dev)}
    saved, f.fast_path = f.fast_path, None
    try:
        y = f(bound['x'], bound['qweight'], bound['scales'], bound['qzeros'])
    finally:
        f.fast_path = saved
    want = hot_ops.gemm_w4a16(p['x'].numpy(), p['qweight'].numpy(), p['scales'].numpy(), p['qzeros'].numpy())
    assert np.allclose(y.cpu().numpy().astype(np.float32), want.astype(np.float32), **FP16_TOL)


@pytest.mark.parametrize('K,N,sdt', [(4096, 12288, 'float32'), (4096, 4096, 'float16'), (11008, 4096, 'float32'), (256, 36, 'float32')])
def test_gptq_gemv_sample_program(autort, K, N, sdt):
    from antares_amd.autort import patterns
    from oracle import hot_ops
    note(f'gptq gemv K={K} N={N} scales={sdt}')
    g = torch.Generator().manual_seed(K + N)
    q = torch.randint(0, 16, (K, N), generator=g)
    s = (torch.rand(K // 128, N, generator=g) * 0.019 + 0.001).to(torch.float32 if sdt == 'float32' else torch.float16)
    x = torch.randn(K, generator=g)
    qw = workloads.pack_gptq(q)
    f = autort.export(ir=patterns.GPTQ_GEMV_IR, inputs=patterns._gptq_inputs('float32', sdt), config='~N~:[256,8,32],~S~:[64,8]')
    dev = autort.device()
    out = torch.empty(N, dtype=torch.float32, device=dev)
    y = f(x.to(dev), qw.to(dev), s.to(dev), out=out)
    assert y.data_ptr() == out.data_ptr()
    want = hot_ops.gemv_gptq_f32(x.numpy(), qw.numpy(), s.numpy())
    exact = x.numpy().astype(np.float64) @ ((q.numpy().astype(np.float64) - 8) * np.repeat(s.numpy().astype(np.float64), 128, axis=0))
    got = y.cpu().numpy()
    # fp32 sums of K terms: the oracle's own distance from the exact value sets the scale of the tolerance
    tol = max(1e-5, 4 * float(np.abs(want - exact).max()))
    assert np.abs(got - exact).max() <= tol, (np.abs(got - exact).max(), tol)
    assert np.allclose(got, want, rtol=1e-4, atol=1e-4)


# ------------------------------------------------------------------ generic lowering
def test_generic_reduce_variants(autort):
    from antares_amd.ir import parse_program
    from oracle.cpu_backend import CpuModule
    note('generic reduce: softmax program')
    ir = ('temp0[N] >=! input0[N, C]; temp1[N] +=! (input0[N, C] - temp0[N]).call(`exp`); '
          'output0[N, C] = (input0[N, C] - temp0[N]).call(`exp`) / temp1[N]')
    dev = autort.device()
    for shape in [(32, 1024), (3, 5000), (300, 7)]:
        inp = {'input0': {'dtype': 'float32', 'shape': list(shape)}}
        x = torch.randn(*shape, generator=torch.Generator().manual_seed(1))
        f = autort.export(ir=ir, inputs=['input0=float32[%d, %d]' % shape])
        got = f(x.to(dev)).cpu().numpy()
        want = CpuModule(parse_program(ir, inp))(input0=x.numpy())['output0']
        assert np.allclose(got, want, **FP32_TOL)


def test_generic_matmul_and_scatter(autort):
    note('generic matmul + scatter-add')
    dev = autort.device()
    g = torch.Generator().manual_seed(3)
    a, b = torch.randn(70, 50, generator=g), torch.randn(50, 33, generator=g)
    f = autort.export(ir='output0[N, M] +=! input0[N, K] * input1[K, M]', inputs=['input0=float32[N:70, K:50]', 'input1=float32[K:50, M:33]'])
    assert np.allclose(f(a.to(dev), b.to(dev)).cpu().numpy(), (a.double() @ b.double()).numpy(), rtol=1e-4, atol=1e-4)
    idx = torch.randint(0, 16, (1000,), generator=g, dtype=torch.int64).to(torch.int32)
    upd = torch.randint(0, 100, (1000,), generator=g, dtype=torch.int64).to(torch.int32)
    hist = torch.zeros(16, dtype=torch.int32, device=dev)
    h = autort.export(ir='hist[idx[B]] +=. upd[B]', inputs=['hist=int32[H]', 'idx=int32[B]', 'upd=int32[B]'], name='scatter_add_i32')
    h(hist, idx.to(dev), upd.to(dev))
    want = torch.zeros(16, dtype=torch.int64).index_add_(0, idx.long(), upd.long())
    assert hist.cpu().long().tolist() == want.tolist()


def test_code_object_file_loads_and_runs(autort, tmp_path):
    """art_module_load_file: a code object written to disk (what `hipcc --genco` leaves) is loaded and launched."""
    import ctypes
    from antares_amd.runtime import capi
    note('art_module_load_file')
    capi.init(0)
    image = capi.compile_hip('extern "C" __global__ void twice(float* a, int n) { int i = blockIdx.x * 64 + threadIdx.x; if (i < n) a[i] *= 2.f; }')
    path = tmp_path / 'twice.hsaco'
    path.write_bytes(image)
    h, f = ctypes.c_void_p(), ctypes.c_void_p()
    capi.check(capi.lib().art_module_load_file(str(path).encode(), ctypes.byref(h)))
    capi.check(capi.lib().art_get_function(h, b'twice', ctypes.byref(f)))
    a = torch.arange(100, dtype=torch.float32, device=autort.device())
    capi.launch(f, (2, 1, 1), (64, 1, 1), torch.cuda.current_stream().cuda_stream, [a.data_ptr(), 100])
    torch.cuda.synchronize()
    assert torch.equal(a.cpu(), torch.arange(100, dtype=torch.float32) * 2)


@pytest.mark.parametrize('ir,inputs,shapes', [
    ('output0[] +=! input0[N]', ['input0=float32[N:1048576]'], [(1048576,), (1000003,), (262144,)]),
    ('output0[C] +=! input0[N, C]', ['input0=float32[N:2048, C:512]'], [(2048, 512), (4096, 96)]),
    ('output0[N] >=! input0[N, C]', ['input0=float32[N:8, C:65536]'], [(8, 65536), (3, 40000)]),
    ('output0[N] <=! input0[N, C]', ['input0=float32[8, 32768]'], [(8, 32768)]),
    ('output0[N, M] +=! input0[N, K] * input1[K, M]', ['input0=float32[N:4, K:8192]', 'input1=float32[K:8192, M:16]'], [(4, 8192, 16)]),
    ('output0[] +=! input0[N]', ['input0=int32[N:2097152]'], [(2097152,)]),
])
def test_wide_reductions_are_sliced_and_still_right(autort, ir, inputs, shapes):
    """Reductions with too few outputs to fill the chip run as two statements (slices, then the slices); programs with
    named dimensions get kernels per set of values, and sizes that do not divide fall back to the one-statement form."""
    note(f'wide reduction {ir}')
    dev = autort.device()
    op = autort.export(ir=ir, inputs=inputs, name='wide_' + str(abs(hash((ir, tuple(inputs)))) % 10 ** 8))
    g = torch.Generator().manual_seed(11)
    for shape in shapes:
        if 'input1' in ir:
            n, k, m = shape
            a, b = torch.randn(n, k, generator=g), torch.randn(k, m, generator=g)
            got = op(a.to(dev), b.to(dev)).cpu()
            assert torch.allclose(got, (a.double() @ b.double()).float(), rtol=1e-4, atol=1e-3)
            continue
        if 'int32' in inputs[0]:
            x = torch.randint(-1000, 1000, shape, generator=g, dtype=torch.int32)
            assert int(op(x.to(dev)).cpu()) == int(x.sum())
            continue
        x = torch.randn(shape, generator=g)
        got = op(x.to(dev)).cpu()
        if '>=!' in ir:
            assert torch.equal(got, x.max(dim=1).values)
        elif '<=!' in ir:
            assert torch.equal(got, x.min(dim=1).values)
        elif ir.startswith('output0[C]'):
            assert torch.allclose(got, x.double().sum(0).float(), rtol=1e-4, atol=1e-3)
        else:
            assert abs(float(got) - float(x.double().sum())) < 0.05


@pytest.mark.parametrize('ir,spec,shape,perm', [
    ('output0[C, N] = input0[N, C]', 'input0=float32[N:1000, C:777]', (1000, 777), (1, 0)),
    ('output0[N, H, W, C] = input0[N, C, H, W]', 'input0=float16[N:3, C:70, H:5, W:129]', (3, 70, 5, 129), (0, 2, 3, 1)),
    ('output0[B, C, N] = input0[N, B, C] * 2', 'input0=float32[N:65, B:2, C:64]', (65, 2, 64), (1, 2, 0)),
    ('output0[C, N] = input0[N, C]', 'input0=int32[N:16, C:4096]', (16, 4096), (1, 0)),
])
def test_permutation_copies_go_through_lds_tiles(autort, ir, spec, shape, perm):
    """A copy whose store walks memory along another axis than its load is lowered to 64 x 64 tiles through LDS."""
    note(f'tiled permutation {ir} {shape}')
    dev = autort.device()
    op = autort.export(ir=ir, inputs=[spec], name='perm_' + str(abs(hash((ir, spec))) % 10 ** 8))
    assert 'tile' in op.plans[0].variants
    g = torch.Generator().manual_seed(4)
    if 'int32' in spec:
        x = torch.randint(-10 ** 6, 10 ** 6, shape, generator=g, dtype=torch.int32)
    else:
        x = torch.randn(shape, generator=g).to(torch.float16 if 'float16' in spec else torch.float32)
    want = x.permute(*perm).contiguous()
    if '* 2' in ir:
        want = want * 2
    assert torch.equal(op(x.to(dev)).cpu(), want)


@pytest.mark.parametrize('ir,spec,shape,perm', [
    ('output0[C, N] = input0[N, C]', 'input0=float32[N:1024, C:448]', (1024, 448), (1, 0)),
    ('output0[N, H, W, C] = input0[N, C, H, W]', 'input0=float16[N:2, C:128, H:3, W:64]', (2, 128, 3, 64), (0, 2, 3, 1)),
    ('output0[B, C, N] = input0[N, B, C] * 2', 'input0=float32[N:192, B:3, C:64]', (192, 3, 64), (1, 2, 0)),
    ('output0[C, N] = input0[N, C].cast(`float32`)', 'input0=int32[N:64, C:4096]', (64, 4096), (1, 0)),
])
def test_permutation_copies_of_whole_tiles_move_16_byte_vectors(autort, ir, spec, shape, perm):
    """With whole 64 x 64 tiles and aligned tensors the transposing variant reads and writes 16-byte vectors; a view
    that is not 16-byte aligned takes the scalar tiles, with the same result."""
    note(f'vector-tiled permutation {ir} {shape}')
    dev = autort.device()
    op = autort.export(ir=ir, inputs=[spec], name='permv_' + str(abs(hash((ir, spec))) % 10 ** 8))
    plan = op.plans[0]
    assert 'tilevec' in plan.variants
    g = torch.Generator().manual_seed(5)
    if 'int32' in spec:
        x = torch.randint(-10 ** 6, 10 ** 6, shape, generator=g, dtype=torch.int32)
    else:
        x = torch.randn(shape, generator=g).to(torch.float16 if 'float16' in spec else torch.float32)
    want = x.permute(*perm).contiguous()
    if '* 2' in ir:
        want = want * 2
    if 'cast' in ir:
        want = want.float()
    xd = x.to(dev)
    env = {k: v for k, v in zip([d.split(':')[0] for d in spec[spec.index('[') + 1:-1].split(', ')], shape)}
    out = torch.empty(want.shape, dtype=want.dtype, device=dev)
    assert plan.choose(env, {'input0': xd.data_ptr(), 'output0': out.data_ptr()})[0] == plan.variants['tilevec']
    assert torch.equal(op(xd).cpu(), want)
    # the same values 4 bytes further on: not aligned for vectors
    flat = torch.empty(x.numel() + 4, dtype=x.dtype, device=dev)
    skip = 4 // x.element_size()
    shifted = flat[skip:skip + x.numel()].view(shape)
    shifted.copy_(xd)
    assert plan.choose(env, {'input0': shifted.data_ptr(), 'output0': out.data_ptr()})[0] == plan.variants['tile']
    assert torch.equal(op(shifted).cpu(), want)


def test_split_k_launches_on_two_streams_do_not_disturb_each_other(autort):
    """Every stream has a workspace of its own: GEMVs with K-splits enqueued on two streams at the same time give
    the bits they give alone, and an aliasing y is refused."""
    from ctypes import c_void_p
    from antares_amd.runtime import capi
    note('split-K GEMVs on two streams')
    dev = autort.device()
    f = w4_op(autort)
    pa, pb = workloads.w4_problem(31, 1, 11008, 4096), workloads.w4_problem(32, 1, 11008, 4096)
    a = [pa[k].to(dev) for k in ('x', 'qweight', 'scales', 'qzeros')]
    b = [pb[k].to(dev) for k in ('x', 'qweight', 'scales', 'qzeros')]
    alone_a, alone_b = f(*a).clone(), f(*b).clone()
    torch.cuda.synchronize()
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    outs_a = [torch.empty_like(alone_a) for _ in range(20)]
    outs_b = [torch.empty_like(alone_b) for _ in range(20)]
    for i in range(20):
        with torch.cuda.stream(s1):
            f(*a, out=outs_a[i])
        with torch.cuda.stream(s2):
            f(*b, out=outs_b[i])
    torch.cuda.synchronize()
    for i in range(20):
        assert torch.equal(outs_a[i], alone_a) and torch.equal(outs_b[i], alone_b), i
    # y overlapping x is refused by the entry points (only the residual may alias y)
    x = a[0]
    rc = capi.lib().art_gemv_w4a16(c_void_p(x.data_ptr()), c_void_p(a[1].data_ptr()), c_void_p(a[2].data_ptr()),
                                   c_void_p(a[3].data_ptr()), c_void_p(x.data_ptr() + 64), 1, 11008, 4096, None)
    assert rc != 0 and b'overlap' in capi.lib().art_last_error()
    rc = capi.lib().art_gemv_w4a16_fused(c_void_p(x.data_ptr()), c_void_p(a[1].data_ptr()), c_void_p(a[2].data_ptr()),
                                         c_void_p(a[3].data_ptr()), c_void_p(x.data_ptr()), 11008, 4096, None, 1e-5, None, 0, None)
    assert rc != 0 and b'overlap' in capi.lib().art_last_error()


def test_fp16_reductions_where_tree_order_leaves_the_sequential_oracle(autort):
    """A reduction written in fp16 accumulates in fp16 on both sides (the reference's rule), but the GPU adds in tree
    order and the oracle in index order.  For 64 to 1024 terms of N(0,1) data the GPU stays within the fp16 tolerance
    of the float64 sum; the sequential oracle itself drifts from it (0.03 at 64 terms, 0.4 at 1024, where 1e-2 of the
    result's size is 0.3), so the two are compared with the oracle's own drift added to the tolerance.  Far beyond
    that they part for good: 16384 positive terms stall a sequential fp16 sum (at 2048 an addend below 1 is rounded
    away), while the tree keeps adding numbers of similar size - there the GPU result must be the one closer to the
    float64 sum, and within the fp16 tolerance of it."""
    from antares_amd.ir import parse_program
    from oracle.cpu_backend import CpuModule
    dev = autort.device()
    ir = 'output0[N] +=! input0[N, C]'
    for C in (64, 256, 1024):
        note(f'fp16 row sums, C={C}')
        x = torch.randn(48, C, generator=torch.Generator().manual_seed(C)).half()
        f = autort.export(ir=ir, inputs=[f'input0=float16[48, {C}]'], name=f'rowsum_f16_{C}')
        got = f(x.to(dev)).float().cpu().numpy()
        want = CpuModule(parse_program(ir, {'input0': {'dtype': 'float16', 'shape': [48, C]}}), fast_math=False)(input0=x.numpy())['output0']
        exact = x.double().sum(1).numpy()
        # sums of C terms of unit variance: sqrt(C) in size; fp16 keeps 2^-11 of that per addition
        tol = 1e-2 * max(1.0, C ** 0.5)
        assert np.abs(got - exact).max() <= tol, (C, np.abs(got - exact).max())
        drift = np.abs(want.astype(np.float64) - exact).max()
        assert np.abs(got - want.astype(np.float32)).max() <= tol + drift, (C, np.abs(got - want.astype(np.float32)).max(), drift)
    C = 16384
    note(f'fp16 row sums of positive data, C={C}')
    x = torch.rand(8, C, generator=torch.Generator().manual_seed(7)).half()
    f = autort.export(ir=ir, inputs=[f'input0=float16[8, {C}]'], name=f'rowsum_f16_{C}')
    got = f(x.to(dev)).float().cpu().numpy()
    want = CpuModule(parse_program(ir, {'input0': {'dtype': 'float16', 'shape': [8, C]}}), fast_math=False)(input0=x.numpy())['output0'].astype(np.float32)
    exact = x.double().sum(1).numpy()                      # about 8192
    assert np.all(want < 0.5 * exact)                      # the sequential fp16 sum has stalled (near 2048)
    assert np.allclose(got, exact, rtol=1e-2)              # the tree-ordered one has not
    assert np.all(np.abs(got - exact) < np.abs(want - exact))


@pytest.mark.parametrize('M,K,N', [(5, 512, 272), (64, 4096, 4096), (128, 1024, 1040), (200, 4096, 512)])
def test_w4a16_gemm_with_the_residual_folded_in(autort, M, K, N):
    """gemm_w4a16_residual: y = fp16(fp16(x @ W) + residual), in place on the residual, with and without K-splits."""
    from oracle import hot_ops
    note(f'w4a16 gemm + residual M={M} K={K} N={N}')
    dev = autort.device()
    p = workloads.w4_problem(K + N + M, M, K, N)
    res = torch.randn(M, N, generator=torch.Generator().manual_seed(M)).half()
    prod = hot_ops.gemm_w4a16(p['x'].numpy(), p['qweight'].numpy(), p['scales'].numpy(), p['qzeros'].numpy())
    want = (prod.astype(np.float32) + res.numpy().astype(np.float32)).astype(np.float16).astype(np.float32)
    d = [p[k].to(dev) for k in ('x', 'qweight', 'scales', 'qzeros')]
    acc = res.to(dev).clone()
    autort.ops.gemm_w4a16_residual(*d, acc, residual=acc)
    assert np.allclose(acc.float().cpu().numpy(), want, **FP16_TOL)
    out = torch.empty_like(acc)
    autort.ops.gemm_w4a16_residual(*d, out, residual=res.to(dev))
    assert torch.equal(out, acc)
    plain = torch.empty_like(acc)
    autort.ops.gemm_w4a16_residual(*d, plain)
    assert np.allclose(plain.float().cpu().numpy(), prod.astype(np.float32), **FP16_TOL)


# one group and many; one row past and one short of a block; the last column tile a chunk of 16; more K-splits than groups
@pytest.mark.parametrize('M,K,N', [(1, 128, 16), (33, 640, 144), (65, 128, 16), (128, 256, 272), (129, 384, 528), (255, 1024, 240), (257, 640, 256), (300, 2048, 1040)])
def test_w4a16_gemm_in_every_form(autort, M, K, N):
    from ctypes import c_void_p
    from antares_amd.runtime import capi
    from oracle import hot_ops
    dev = autort.device()
    p = workloads.w4_problem(K + N + M, M, K, N)
    res = torch.randn(M, N, generator=torch.Generator().manual_seed(M)).half()
    prod = hot_ops.gemm_w4a16(p['x'].numpy(), p['qweight'].numpy(), p['scales'].numpy(), p['qzeros'].numpy()).astype(np.float32)
    d = [p[k].to(dev) for k in ('x', 'qweight', 'scales', 'qzeros')] + [torch.empty(M, N, dtype=torch.float16, device=dev), res.to(dev)]
    ptr = [c_void_p(t.data_ptr()) for t in d]
    for form in (1, 2, 5, 4, 8):          # 32, 64 and 128 rows over 128 columns, 128 and 256 rows over 256 columns
        for splits in (1, 2, 3, 16):
            note(f'w4a16 gemm M={M} K={K} N={N} form {form}, {splits} splits')
            code = form * 256 + splits
            for residual, want in ((c_void_p(0), prod), (ptr[5], (prod + res.numpy().astype(np.float32)))):
                d[4].fill_(float('nan'))
                capi.check(capi.lib().art_gemm_w4a16_residual(*ptr[:5], residual, M, K, N, code, c_void_p(torch.cuda.current_stream().cuda_stream)))
                torch.cuda.synchronize()
                assert np.allclose(d[4].float().cpu().numpy(), want, **FP16_TOL)


# both kernels, with and without K-splits (code 0: the library's choice); halves of 16 columns and past a tile of 128
@pytest.mark.parametrize('M,K,F', [(5, 128, 16), (33, 512, 144), (64, 1024, 112), (65, 256, 128), (130, 2048, 272), (257, 640, 400)])
def test_w4a16_gemm_with_swiglu_behind_it(autort, M, K, F):
    from ctypes import c_void_p
    from antares_amd.runtime import capi
    from oracle import hot_ops
    dev = autort.device()
    p = workloads.w4_problem(K + F + M, M, K, 2 * F)
    p['scales'] = p['scales'] * 0.1
    prod = hot_ops.gemm_w4a16(p['x'].numpy(), p['qweight'].numpy(), p['scales'].numpy(), p['qzeros'].numpy()).astype(np.float32)
    gate, up = prod[:, :F], prod[:, F:]
    want = gate / (1 + np.exp(-gate)) * up
    d = [p[k].to(dev) for k in ('x', 'qweight', 'scales', 'qzeros')]
    for code in (0, 256 + 1, 256 + 2, 512 + 1, 512 + 3, 1280 + 1, 1280 + 2, 1024 + 1, 1024 + 4, 2048 + 1, 2048 + 2):
        note(f'w4a16 gemm + swiglu M={M} K={K} F={F} code {code}')
        out = torch.full((M, F), float('nan'), dtype=torch.float16, device=dev)
        capi.check(capi.lib().art_gemm_w4a16_swiglu(*(c_void_p(t.data_ptr()) for t in d), c_void_p(out.data_ptr()), M, K, 2 * F, code,
                                                    c_void_p(torch.cuda.current_stream().cuda_stream)))
        torch.cuda.synchronize()
        assert np.allclose(out.float().cpu().numpy(), want, **FP16_TOL)
    got = autort.ops.gemm_w4a16_swiglu(*d)
    assert got.shape == (M, F) and np.allclose(got.float().cpu().numpy(), want, **FP16_TOL)


# column tiles whose number is no multiple of eight times one, a few and more row blocks than XCDs; K-splits of every count that the pass behind
# the product knows and one more
@pytest.mark.parametrize('M,K,N', [(20, 384, 128 * 9), (300, 256, 128 * 15 + 16), (33 * 8 + 1, 128, 256 * 9 + 48), (70, 1280, 256 * 3)])
def test_w4a16_gemm_blocks_that_are_dealt_to_all_xcds(autort, M, K, N):
    from ctypes import c_void_p
    from antares_amd.runtime import capi
    from oracle import hot_ops
    dev = autort.device()
    capi.init(0)
    p = workloads.w4_problem(K + N + M, M, K, N)
    want = hot_ops.gemm_w4a16(p['x'].numpy(), p['qweight'].numpy(), p['scales'].numpy(), p['qzeros'].numpy()).astype(np.float32)
    d = [p[k].to(dev) for k in ('x', 'qweight', 'scales', 'qzeros')]
    for form in (1, 2, 5, 4, 8):
        for splits in range(1, min(K // 128, 9) + 1):
            note(f'w4a16 gemm M={M} K={K} N={N} form {form}, {splits} splits')
            y = torch.full((M + 1, N), 7.0, dtype=torch.float16, device=dev)
            capi.check(capi.lib().art_gemm_w4a16_tuned(*(c_void_p(t.data_ptr()) for t in d), c_void_p(y.data_ptr()), M, K, N, form * 256 + splits,
                                                       c_void_p(torch.cuda.current_stream().cuda_stream)))
            got = y.float().cpu().numpy()
            assert np.allclose(got[:M], want, **FP16_TOL) and (got[M] == 7.0).all()


# Every fp16 gate: one weight of a gate column is 1 (infinite gates: 2), one of its up column too.  The gate itself is exact; silu in float32
# is less than 2^-22 off, the product with up and its rounding 2^-24 and 2^-11, or half of 2^-24 among the subnormal numbers.
@pytest.mark.parametrize('code', [256 + 1, 512 + 1, 1280 + 1, 1024 + 1, 2048 + 1])
def test_w4a16_gemm_with_swiglu_over_every_fp16_gate(autort, code):
    from ctypes import c_void_p
    from antares_amd.runtime import capi
    dev = autort.device()
    capi.init(0)
    g = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.float16)
    g = torch.cat([g[torch.isfinite(g)], torch.tensor([40000.0, -40000.0, 60000.0, -60000.0], dtype=torch.float16)])
    F, M = 16, g.numel()
    x = torch.zeros(M, 128, dtype=torch.float16)
    x[:, 0], x[:, 1] = g, torch.tensor([1.0, -3.5, 1000.0], dtype=torch.float16).repeat(M // 3 + 1)[:M]
    q = torch.full((128, 2 * F), 8, dtype=torch.uint8)
    q[0, :F] = 9
    q[1, F:] = 9
    scales = torch.ones(1, 2 * F, dtype=torch.float16)
    scales[0, 1] = 2.0                    # gate column 1: twice the value, infinite beyond 32752
    d = [t.to(dev) for t in (x, q[0::2] | (q[1::2] << 4), scales, torch.full((1, F), 0x88, dtype=torch.uint8))]
    out = torch.empty(M, F, dtype=torch.float16, device=dev)
    note(f'every gate, code {code}')
    capi.check(capi.lib().art_gemm_w4a16_swiglu(*(c_void_p(t.data_ptr()) for t in d), c_void_p(out.data_ptr()), M, 128, 2 * F, code,
                                                c_void_p(torch.cuda.current_stream().cuda_stream)))
    got = out.cpu()
    for column, gate in ((0, g), (1, g * 2), (F - 1, g)):
        exact = gate.double()
        want = torch.where(exact < -700, -0.0, exact / (1 + torch.exp(-exact.clamp(min=-700)))) * x[:, 1].double()
        want[exact == -float('inf')] = float('nan')
        y, fits = got[:, column].double(), want.abs() < 65504
        assert torch.equal(torch.isnan(y), torch.isnan(want))
        bound = want[fits].abs() * (2.0 ** -11 + 2.0 ** -21) + 2.0 ** -25
        assert bool(((y[fits] - want[fits]).abs() <= bound).all())
        assert torch.equal(y[want.abs() > 65520], torch.sign(want[want.abs() > 65520]) * float('inf'))


ROW_VECTOR_CASES = [
    # program, inputs, shapes of the inputs, does the row-vector variant apply to these extents
    ('output0[N, C] = input0[N, C] + input1[C]', ['input0=float32[N:300, C:1024]', 'input1=float32[C:1024]'], [(300, 1024), (1024,)], True),
    ('output0[N, C] = input0[input1[N], C]', ['input0=float32[V:500, C:256]', 'input1=int32[N:1000]'], [(500, 256), (1000,)], True),
    ('emb[T, D] = table[tok[T], D]', ['table=float16[V:320, D:4096]', 'tok=int32[T:37]'], [(320, 4096), (37,)], True),
    ('output0[B, N, C] = (input0[B, N, C].to(`float32`) * input1[B, C] + input2[N]).to(`float16`)',
     ['input0=float16[B:3, N:50, C:72]', 'input1=float32[B:3, C:72]', 'input2=float32[N:50]'], [(3, 50, 72), (3, 72), (50,)], True),
    ('output0[N, C] = input0[N, C] * C + input1[N]', ['input0=int32[N:33, C:64]', 'input1=int32[N:33]'], [(33, 64), (33,)], True),
    # a last extent that is no multiple of the vector: the scalar kernel runs
    ('output0[N, C] = input0[N, C] + input1[C]', ['input0=float32[N:30, C:1023]', 'input1=float32[C:1023]'], [(30, 1023), (1023,)], False),
]


@pytest.mark.parametrize('ir,inputs,shapes,applies', ROW_VECTOR_CASES)
def test_row_vector_maps_match_the_oracle(autort, ir, inputs, shapes, applies):
    """Maps whose loads are runs along the last axis or constant along it (bias rows, gathered rows) move 16-byte
    vectors per lane; results are the oracle's, and the scalar kernel takes over where the extents do not fit."""
    from antares_amd.ir import parse_program
    from oracle.cpu_backend import CpuModule
    note(f'row-vector map {ir} {shapes}')
    dev = autort.device()
    op = autort.export(ir=ir, inputs=inputs, name='rowvec_' + str(abs(hash((ir, tuple(inputs)))) % 10 ** 8))
    plan = op.plans[0]
    assert 'rowvec' in plan.variants and 'vec' not in plan.variants
    g = torch.Generator().manual_seed(len(ir))
    tensors, names = [], []
    for spec, shape in zip(inputs, shapes):
        name, rest = spec.split('=')
        names.append(name)
        if rest.startswith('int32'):
            hi = 320 if 'tok' in name else (500 if name == 'input1' and 'input0[input1' in ir else 1000)
            tensors.append(torch.randint(0, hi, shape, generator=g, dtype=torch.int32))
        else:
            tensors.append(torch.randn(shape, generator=g).to(torch.float16 if rest.startswith('float16') else torch.float32))
    env = {}
    for spec, shape in zip(inputs, shapes):
        dims = spec.split('[', 1)[1].rstrip(']').split(',')
        for d, v in zip(dims, shape):
            env[d.split(':')[0].strip()] = v
    ptrs = {n: 0 for n in plan.args}
    assert (plan.choose(env, ptrs)[0] == plan.variants['rowvec']) == applies
    got = op(*[t.to(dev) for t in tensors]).cpu().numpy()
    out_name = ir.split('[', 1)[0].strip()
    want = CpuModule(parse_program(ir, inputs), fast_math=False)(**{n: t.numpy() for n, t in zip(names, tensors)})[out_name]
    if got.dtype.kind == 'i':
        assert np.array_equal(got, want)
    else:
        assert np.allclose(got.astype(np.float32), want.astype(np.float32), rtol=1e-2 if got.dtype == np.float16 else 1e-5,
                           atol=1e-2 if got.dtype == np.float16 else 1e-5)
    # an operand that is not 16-byte aligned falls back to the scalar kernel, same result
    if applies and tensors[0].dtype != torch.int32:
        base = torch.empty(tensors[0].numel() + 1, dtype=tensors[0].dtype, device=dev)
        view = base[1:].view(tensors[0].shape)
        view.copy_(tensors[0])
        got2 = op(view, *[t.to(dev) for t in tensors[1:]]).cpu().numpy()
        assert np.array_equal(got2, got)


def dims_of(inputs, shapes):
    """{named dimension: value} of tensors of these shapes for input specs like `input0=float32[N:8, C:16]`."""
    env = {}
    for spec, shape in zip(inputs, shapes):
        for d, v in zip(spec.split('[', 1)[1].rstrip(']').split(','), shape):
            if ':' in d:
                env[d.split(':')[0].strip()] = v
    return env


PATCH_CASES = [
    ('output0[N, M] +=! input0[N, K] * input1[K, M]', ['input0=float32[N:64, K:96]', 'input1=float32[K:96, M:128]'], [(64, 96), (96, 128)]),
    ('output0[B, N, M] +=! input0[B, N, K] * input1[B, K, M]', ['input0=float32[B:3, N:32, K:40]', 'input1=float32[B:3, K:40, M:64]'],
     [(3, 32, 40), (3, 40, 64)]),
    ('output0[N, M] +=! input0[N, K] * input1[M, K]', ['input0=float16[N:32, K:64]', 'input1=float16[M:48, K:64]'], [(32, 64), (48, 64)]),
    ('output0[N, F, HO, WO] +=! input0[N, C, HO + KH, WO + KW] * input1[F, C, KH, KW] where HO in 10, WO in 12',
     ['input0=float32[N:2, C:5, H:12, W:14]', 'input1=float32[F:8, C:5, KH:3, KW:3]'], [(2, 5, 12, 14), (8, 5, 3, 3)]),
    ('output0[N, M] >=! input0[N, K] + input1[K, M]', ['input0=int32[N:16, K:33]', 'input1=int32[K:33, M:20]'], [(16, 33), (33, 20)]),
    # a depthwise filter whose size comes as named dimensions: the kernels of this call have 3 x 3 written into them
    ('output0[N, C, HO, WO] +=! input0[N, C, HO + KH, WO + KW] * input1[C, KH, KW] where HO in 12, WO in 16',
     ['input0=float32[N:3, C:7, H:14, W:18]', 'input1=float32[C:7, KH:3, KW:3]'], [(3, 7, 14, 18), (7, 3, 3)]),
]


@pytest.mark.parametrize('ir,inputs,shapes', PATCH_CASES)
def test_register_tiled_contractions_match_the_oracle(autort, ir, inputs, shapes, monkeypatch):
    """The reduce variant in which a thread owns 4 x 4 neighbouring outputs (what large contractions get) gives the
    oracle's results, and the bits of the one-output-per-thread variant, whose order of accumulation it keeps."""
    from antares_amd.ir import parse_program
    from oracle.cpu_backend import CpuModule
    note(f'register-tiled reduce {ir} {shapes}')
    dev = autort.device()
    op = autort.export(ir=ir, inputs=inputs, name='patch_' + str(abs(hash((ir, tuple(inputs)))) % 10 ** 8))
    plan = op.plans_for(dims_of(inputs, shapes))[0]
    assert 'patch' in plan.variants
    g = torch.Generator().manual_seed(len(ir))
    names = [spec.split('=')[0] for spec in inputs]
    tensors = [torch.randint(-1000, 1000, shp, generator=g, dtype=torch.int32) if 'int32' in spec else
               (torch.randn(shp, generator=g) * 0.5).to(torch.float16 if 'float16' in spec else torch.float32)
               for spec, shp in zip(inputs, shapes)]
    total = op(*[t.to(dev) for t in tensors]).numel()
    results = {}
    for tag in ('patch', 'thread'):
        work = total // 16 if tag == 'patch' else total
        monkeypatch.setattr(plan, 'choose', lambda env, ptrs, tag=tag, work=work: (plan.variants[tag], (work + 255) // 256, 256))
        results[tag] = op(*[t.to(dev) for t in tensors]).cpu()
    assert torch.equal(results['patch'], results['thread'])
    out_name = ir.split('[', 1)[0].strip()
    want = CpuModule(parse_program(ir, inputs), fast_math=False)(**{n: t.numpy() for n, t in zip(names, tensors)})[out_name]
    got = results['patch'].numpy()
    if got.dtype.kind == 'i':
        assert np.array_equal(got, want)
    else:
        tol = 1e-2 if got.dtype == np.float16 else 1e-4
        assert np.allclose(got.astype(np.float32), want.astype(np.float32), rtol=tol, atol=tol)


def test_large_contractions_take_the_register_tiled_variant(autort):
    """Without the matrix-instruction variant a 2048 x 2048 x 256 fp32 matrix product is large enough for the
    register-tiled one (a 1024 x 1024 one is not); the result is the float64 product's."""
    note('register-tiled reduce picked for a 2048x2048x256 fp32 matmul')
    dev = autort.device()
    op = autort.export(ir='output0[N, M] +=! input0[N, K] * input1[K, M]', inputs=['input0=float32[N:2048, K:256]', 'input1=float32[K:256, M:2048]'],
                       name='patch_matmul_2048')
    op.fast_path = None               # the generic lowering is what is tested here
    plan = op.plans[0]
    zero = {n: 0 for n in plan.args}
    assert plan.choose({'N': 2048, 'K': 256, 'M': 2048}, zero)[0] == plan.variants['matrixv']
    for tag in [t for t in plan.variants if t.startswith('matrix')]:
        del plan.variants[tag]
    assert plan.choose({'N': 2048, 'K': 256, 'M': 2048}, zero)[0] == plan.variants['patch']
    assert plan.choose({'N': 2046, 'K': 256, 'M': 2048}, zero)[0] != plan.variants['patch']
    assert plan.choose({'N': 1024, 'K': 256, 'M': 1024}, zero)[0] != plan.variants['patch']
    g = torch.Generator().manual_seed(2)
    a, b = torch.randn(2048, 256, generator=g), torch.randn(256, 2048, generator=g)
    got = op(a.to(dev), b.to(dev)).cpu()
    want = (a.double() @ b.double()).float()
    assert torch.allclose(got, want, rtol=1e-4, atol=1e-3)


MATRIX_CASES = [
    # a convolution; the same with stride 2; a batched product with ragged tiles and k = 5 x 16; fp16 operands cast to
    # float32 with B stored [N, K]; elementwise work on one factor (AntaresIR.md:247 over all of K); a product whose
    # output axes are stored columns first
    ('output0[N, F, HO, WO] +=! input0[N, C, HO + KH, WO + KW] * input1[F, C, KH, KW] where HO in 32, WO in 32',
     ['input0=float32[N:8, C:16, H:34, W:34]', 'input1=float32[F:64, C:16, KH:3, KW:3]'], [(8, 16, 34, 34), (64, 16, 3, 3)]),
    ('output0[N, F, HO, WO] +=! input0[N, C, HO * 2 + KH, WO * 2 + KW] * input1[F, C, KH, KW] where HO in 32, WO in 32',
     ['input0=float32[N:8, C:16, H:66, W:66]', 'input1=float32[F:70, C:16, KH:3, KW:3]'], [(8, 16, 66, 66), (70, 16, 3, 3)]),
    ('output0[B, N, M] +=! input0[B, N, K] * input1[B, K, M]', ['input0=float32[B:3, N:700, K:80]', 'input1=float32[B:3, K:80, M:520]'],
     [(3, 700, 80), (3, 80, 520)]),
    ('output0[N, M] +=! input0[N, K].to(`float32`) * input1[M, K].to(`float32`)', ['input0=float16[N:1024, K:64]', 'input1=float16[M:1000, K:64]'],
     [(1024, 64), (1000, 64)]),
    ('temp0[K, N] = input0[N, K] + 100; output0[N, M] +=! temp0[K, N] * input1[K, M]',
     ['input0=float32[N:1024, K:512]', 'input1=float32[K:512, M:1024]'], [(1024, 512), (512, 1024)]),
    ('output0[M, N] +=! input0[N, K] * input1[K, M]', ['input0=float32[N:1030, K:64]', 'input1=float32[K:64, M:1024]'], [(1030, 64), (64, 1024)]),
    # k that is no multiple of the tile: a first-layer convolution (3 channels, 7 x 7, stride 2: k = 147), a product with k = 250
    ('output0[N, F, HO, WO] +=! input0[N, C, HO * 2 + KH, WO * 2 + KW] * input1[F, C, KH, KW] where HO in 29, WO in 29',
     ['input0=float32[N:10, C:3, H:64, W:64]', 'input1=float32[F:64, C:3, KH:7, KW:7]'], [(10, 3, 64, 64), (64, 3, 7, 7)]),
    ('output0[N, M] +=! input0[N, K] * input1[M, K]', ['input0=float32[N:1024, K:250]', 'input1=float32[M:1024, K:250]'], [(1024, 250), (1024, 250)]),
    # fp16 operands that are only cast up stay fp16 in the tiles (v_mfma_f32_32x32x16_f16): B stored [K, M], k = 2.5 tiles;
    # a batched product of fp16 operands
    ('output0[N, M] +=! input0[N, K].to(`float32`) * input1[K, M].to(`float32`)', ['input0=float16[N:1100, K:80]', 'input1=float16[K:80, M:1024]'],
     [(1100, 80), (80, 1024)]),
    ('output0[B, N, M] +=! input0[B, N, K].to(`float32`) * input1[B, M, K].to(`float32`)',
     ['input0=float16[B:4, N:520, K:96]', 'input1=float16[B:4, M:500, K:96]'], [(4, 520, 96), (4, 500, 96)]),
    # guarded factors: a convolution that pads by one with zeros (AntaresIR.md:166), in float32 and with fp16 tiles; a
    # product whose first operand is shifted along k and cut where it runs out, lanes along k
    ('output0[N, F, HO, WO] +=! input0[N, C, HO + KH - 1, WO + KW - 1].when([HO + KH - 1 >= 0, HO + KH - 1 < 32, WO + KW - 1 >= 0, '
     'WO + KW - 1 < 32], 0.0) * input1[F, C, KH, KW] where HO in 32, WO in 32',
     ['input0=float32[N:6, C:16, H:32, W:32]', 'input1=float32[F:64, C:16, KH:3, KW:3]'], [(6, 16, 32, 32), (64, 16, 3, 3)]),
    ('output0[N, F, HO, WO] +=! input0[N, C, HO + KH - 1, WO + KW - 1].to(`float32`).when([HO + KH - 1 >= 0, HO + KH - 1 < 30, '
     'WO + KW - 1 >= 0, WO + KW - 1 < 30], 0.0) * input1[F, C, KH, KW].to(`float32`) where HO in 30, WO in 30',
     ['input0=float16[N:5, C:20, H:30, W:30]', 'input1=float16[F:72, C:20, KH:3, KW:3]'], [(5, 20, 30, 30), (72, 20, 3, 3)]),
    ('output0[N, M] +=! input0[N, K + 5].when([K + 5 < 80], 0.0) * input1[K, M] where K in 80',
     ['input0=float32[N:1024, J:80]', 'input1=float32[K:80, M:1024]'], [(1024, 80), (80, 1024)]),
    # channels last (image `[N, H, W, C]`, filter `[KH, KW, C, F]`): the image in 16-byte vectors of channels, the filter staged as it
    # lies; the same with fp16 operands and 24 channels (k = 216: 6.75 tiles)
    ('output0[N, HO, WO, F] +=! input0[N, HO + KH, WO + KW, C] * input1[KH, KW, C, F] where HO in 20, WO in 20',
     ['input0=float32[N:5, H:22, W:22, C:16]', 'input1=float32[KH:3, KW:3, C:16, F:72]'], [(5, 22, 22, 16), (3, 3, 16, 72)]),
    ('output0[N, HO, WO, F] +=! input0[N, HO + KH, WO + KW, C].to(`float32`) * input1[KH, KW, C, F].to(`float32`) where HO in 20, WO in 20',
     ['input0=float16[N:5, H:22, W:22, C:24]', 'input1=float16[KH:3, KW:3, C:24, F:72]'], [(5, 22, 22, 24), (3, 3, 24, 72)]),
    # the guarded factor second: the filter's output channels are the rows, the padded image's positions the columns
    ('output0[F, N, HO, WO] +=! input1[F, C, KH, KW] * input0[N, C, HO + KH - 2, WO + KW - 2].when([HO + KH - 2 >= 0, HO + KH - 2 < 20, '
     'WO + KW - 2 >= 0, WO + KW - 2 < 24], 0.0) where HO in 20, WO in 24',
     ['input0=float32[N:4, C:12, H:20, W:24]', 'input1=float32[F:96, C:12, KH:5, KW:5]'], [(4, 12, 20, 24), (96, 12, 5, 5)]),
]


@pytest.mark.parametrize('ir,inputs,shapes,how', [c + (None,) for c in MATRIX_CASES] +
                         [c + ('guards in the kernel',) for c in MATRIX_CASES if '.when(' in c[0]])
def test_contractions_on_the_matrix_instructions_match_the_oracle(autort, monkeypatch, ir, inputs, shapes, how):
    """Sums of products of two loads whose indices split into a row (or column) part and a k part run on
    v_mfma_f32_32x32x2_f32 when k is a multiple of 16 and there are enough tiles; results are the oracle's to the
    rounding of a float32 sum in another order, and the register-tiled variant gives the same to that rounding.
    A zero-padded factor is normally copied into a padded tensor first (one more statement in front); the cases marked
    'guards in the kernel' switch that off, so that the contraction itself evaluates the conditions - what a program
    gets whose conditions the rewrite does not take."""
    from antares_amd.ir import parse_program
    from oracle.cpu_backend import CpuModule
    note(f'matrix-instruction contraction {ir[:60]} {shapes} {how or ""}')
    dev = autort.device()
    if how:
        monkeypatch.setattr('antares_amd.autort.op.pad_guarded_factors', lambda graph, env=None: graph)
    op = autort.export(ir=ir, inputs=inputs, name='mfma_' + str(abs(hash((ir, tuple(inputs), how))) % 10 ** 8))
    op.fast_path = None
    env = dims_of(inputs, shapes)
    plan = op.plans_for(env)[-1]                  # a filter of a few named elements gets kernels of its own
    if '.when(' in ir:
        padded = any(n.endswith('__pad') for n in plan.args)
        assert padded == (how is None) and len(op.plans_for(env)) == (2 if padded else 1)
    assert plan.choose(env, {n: 0 for n in plan.args})[0] in [v for t, v in plan.variants.items() if t.startswith('matrix')]
    assert plan.row_group is None                 # nothing else takes the statement
    g = torch.Generator().manual_seed(len(ir))
    tensors = [torch.randn(shape, generator=g).to(torch.float16 if 'float16' in spec else torch.float32) for spec, shape in zip(inputs, shapes)]
    names = [spec.split('=')[0] for spec in inputs]
    want = CpuModule(parse_program(ir, inputs), fast_math=False)(**{n: t.numpy() for n, t in zip(names, tensors)})['output0']
    K = 1
    for ax, e in plan.reduce_axes:
        K *= e if isinstance(e, int) else env[e]
    scale = 100.0 if '+ 100' in ir else 1.0
    tol = 2e-5 * scale * K ** 0.5 * 4
    M, N, B = (int(np.prod([e if isinstance(e, int) else env[e] for e in plan.matrix[k]])) for k in ('m', 'n', 'batch'))
    rule = plan.choose
    sizes = [('matrix', 128), ('matrix64', 64)]                # blocks of 128 x 128 and of 64 x 64 outputs
    if 'matrixv' in plan.variants and (plan._matrix_choice(env, {n: 0 for n in plan.args})[0] or '').endswith('v'):
        sizes += [('matrixv', 128), ('matrix64v', 64)]          # ... and their forms that fetch rows of k in 16-byte vectors
        ptrs = {n: 0 for n in plan.args}
        assert plan.choose(env, ptrs)[0] in (plan.variants['matrixv'], plan.variants['matrix64v'])
        ptrs[plan.matrix['vec_tensors'][0]] = 8                 # a tensor that is not 16-byte aligned: scalar fetches
        assert plan.choose(env, ptrs)[0] in (plan.variants['matrix'], plan.variants['matrix64'])
    for tag, side in sizes:
        blocks = ((M + side - 1) // side) * ((N + side - 1) // side) * B
        plan.choose = lambda env_, ptrs, tag=tag, blocks=blocks: (plan.variants[tag], blocks, 256)
        got = op(*[t.to(dev) for t in tensors]).cpu().numpy()
        assert got.shape == want.shape
        assert np.allclose(got, want, rtol=1e-4, atol=tol), (tag, np.abs(got - want).max())
    # the same statement through the register-tiled variant
    plan.choose = rule
    for tag in [t for t in plan.variants if t.startswith('matrix')]:
        del plan.variants[tag]
    apart = op(*[t.to(dev) for t in tensors]).cpu().numpy()
    assert np.allclose(got, apart, rtol=1e-4, atol=tol)


@pytest.mark.parametrize('ir,inputs,shapes', [
    ('output0[N, M] +=! input0[N, K] * input1[K, M]', ['input0=float16[N:1024, K:512]', 'input1=float16[K:512, M:1000]'], [(1024, 512), (512, 1000)]),
    ('output0[B, N, M] +=! input0[B, N, K] * input1[B, M, K]', ['input0=float16[B:3, N:300, K:200]', 'input1=float16[B:3, M:260, K:200]'],
     [(3, 300, 200), (3, 260, 200)]),
])
def test_fp16_contractions_sum_in_float32_on_the_matrix_instructions(autort, ir, inputs, shapes):
    """A float16 sum of products of two float16 loads (AntaresIR.md:115 with float16 tensors) runs on
    v_mfma_f32_32x32x16_f16: exact products, a float32 sum, one rounding at the end.  The reference rounds every product
    and every partial sum to float16 (the oracle does the same); the GPU result must be within one float16 rounding
    of the float64 result, never further from it than the oracle's, and within the oracle's own drift of the oracle."""
    from antares_amd.ir import parse_program
    from oracle.cpu_backend import CpuModule
    note(f'fp16 contraction on the matrix instructions {ir} {shapes}')
    dev = autort.device()
    op = autort.export(ir=ir, inputs=inputs, name='mfma_f16_' + str(abs(hash((ir, tuple(inputs)))) % 10 ** 8))
    op.fast_path = None
    env = dims_of(inputs, shapes)
    plan = op.plans_for(env)[-1]
    g = torch.Generator().manual_seed(len(ir))
    a, b = [(torch.randn(shape, generator=g) * 0.5).half() for shape in shapes]
    want = CpuModule(parse_program(ir, inputs), fast_math=False)(input0=a.numpy(), input1=b.numpy())['output0'].astype(np.float64)
    exact = torch.einsum('...nk,...km->...nm', a.double(), b.double() if ir.endswith('[K, M]') else b.double().transpose(-1, -2)).numpy()
    drift = np.abs(want - exact).max()
    M, N, B = (int(np.prod([e if isinstance(e, int) else env[e] for e in plan.matrix[k]])) for k in ('m', 'n', 'batch'))
    assert plan.choose(env, {n: 0 for n in plan.args})[0] in (plan.variants['matrixv'], plan.variants['matrix64v'])
    for tag, side in (('matrix', 128), ('matrix64', 64), ('matrixv', 128), ('matrix64v', 64)):
        blocks = ((M + side - 1) // side) * ((N + side - 1) // side) * B
        plan.choose = lambda env_, ptrs, tag=tag, blocks=blocks: (plan.variants[tag], blocks, 256)
        out = op(a.to(dev), b.to(dev))
        assert out.dtype == torch.float16 and tuple(out.shape) == exact.shape
        got = out.cpu().numpy().astype(np.float64)
        # one float16 rounding of the result, plus what a float32 sum of K terms of this size may be off by
        assert np.all(np.abs(got - exact) <= 2.0 ** -10 * np.abs(exact) + 2e-4), (tag, np.abs(got - exact).max())
        assert np.abs(got - exact).max() <= drift and np.abs(got - want).max() <= 2 * drift + 1e-3, (tag, drift)


@pytest.mark.parametrize('ir,inputs,shapes,vectors', [
    ('output0[N, F, HO, WO] +=! input0[N, C, HO + KH, WO + KW] * input1[F, C, KH, KW] where HO in 7, WO in 7',
     ['input0=float32[N:4, C:512, H:9, W:9]', 'input1=float32[F:256, C:512, KH:3, KW:3]'], [(4, 512, 9, 9), (256, 512, 3, 3)], True),
    ('output0[N, M] +=! input0[N, K] * input1[M, K]', ['input0=float32[N:320, K:4096]', 'input1=float32[M:512, K:4096]'], [(320, 4096), (512, 4096)], True),
    ('output0[B, N, M] +=! input0[B, N, K] * input1[B, K, M]', ['input0=float32[B:2, N:256, K:2048]', 'input1=float32[B:2, K:2048, M:200]'],
     [(2, 256, 2048), (2, 2048, 200)], True),
    ('output0[N, M] +=! input0[N, K].to(`float32`) * input1[M, K].to(`float32`)', ['input0=float16[1024, 2048]', 'input1=float16[512, 2048]'],
     [(1024, 2048), (512, 2048)], True),
])
def test_contractions_with_few_output_tiles_are_cut_into_slices_of_k(autort, ir, inputs, shapes, vectors):
    """A contraction whose 64 x 64 output tiles number fewer than two per compute unit, over at least 1024 values of k,
    runs as a batch of slices of k on the matrix instructions plus a sum over the slices; an operand that lies as rows
    of k keeps its 16-byte fetches inside a slice.  Results against the oracle, to the rounding of a float32 sum in
    another order."""
    from antares_amd.ir import parse_program
    from oracle.cpu_backend import CpuModule
    note(f'sliced contraction {ir[:60]} {shapes}')
    dev = autort.device()
    op = autort.export(ir=ir, inputs=inputs, name='sliced_' + str(abs(hash((ir, tuple(inputs)))) % 10 ** 8))
    op.fast_path = None
    env = dims_of(inputs, shapes)
    plans = op.plans_for(env)
    assert len(plans) == 2 and plans[0].matrix is not None and plans[1].matrix is None
    sym, blocks, _ = plans[0].choose(env, {n: 0 for n in plans[0].args})
    assert blocks >= 512 or plans[0].matrix['batch'][0] == 8          # the slices fill the chip, or there are 8 of them
    assert sym in [v for t, v in plans[0].variants.items() if t.startswith('matrix') and t.endswith('v') == vectors]
    g = torch.Generator().manual_seed(len(ir))
    tensors = [torch.randn(shape, generator=g).to(torch.float16 if 'float16' in spec else torch.float32) for spec, shape in zip(inputs, shapes)]
    names = [spec.split('=')[0] for spec in inputs]
    want = CpuModule(parse_program(ir, inputs), fast_math=False)(**{n: t.numpy() for n, t in zip(names, tensors)})['output0']
    K = int(np.prod([e if isinstance(e, int) else env[e] for _, e in parse_program(ir, inputs).statements[0].reduce_axes]))
    got = op(*[t.to(dev) for t in tensors]).cpu().numpy()
    assert got.shape == want.shape and np.allclose(got, want, rtol=1e-4, atol=2e-5 * K ** 0.5 * 4), np.abs(got - want).max()


@pytest.mark.parametrize('ir,inputs,shapes', [
    # both operands stored along rows; the second one only, batched (the V of an attention), ragged tiles, k = 2.5 tiles
    ('output0[N, M] +=! input0[K, N].to(`float32`) * input1[K, M].to(`float32`)', ['input0=float16[K:96, N:1000]', 'input1=float16[K:96, M:520]'],
     [(96, 1000), (96, 520)]),
    ('output0[B, S, D] +=! input0[B, S, T].to(`float32`) * input1[B, T, D].to(`float32`)', ['input0=float16[B:3, S:300, T:80]', 'input1=float16[B:3, T:80, D:128]'],
     [(3, 300, 80), (3, 80, 128)]),
    # float32: both operands along rows; the second one only, batched, k = 2.5 tiles of the big blocks
    ('output0[N, M] +=! input0[K, N] * input1[K, M]', ['input0=float32[K:72, N:1000]', 'input1=float32[K:72, M:516]'], [(72, 1000), (72, 516)]),
    ('output0[B, S, D] +=! input0[B, S, T] * input1[B, T, D]', ['input0=float32[B:3, S:300, T:40]', 'input1=float32[B:3, T:40, D:128]'],
     [(3, 300, 40), (3, 40, 128)]),
])
def test_operands_stored_along_rows_are_staged_as_they_lie(autort, ir, inputs, shapes):
    """An operand whose neighbouring rows (columns) are neighbours in memory - `input1[K, M]` - is fetched in 16-byte
    vectors of rows and staged in LDS as [k][row]; fp16 tiles are transposed on their way to the matrix instruction by
    ds_read_b64_tr_b16, float32 ones are read element by element.  The result is that of the kernels that stage it row
    by row, bit for bit, and the oracle's."""
    from antares_amd.ir import parse_program
    from oracle.cpu_backend import CpuModule
    note(f'fp16 operands staged as they lie {ir} {shapes}')
    dev = autort.device()
    op = autort.export(ir=ir, inputs=inputs, name='mfma_tr_' + str(abs(hash((ir, tuple(inputs)))) % 10 ** 8))
    op.fast_path = None
    env = dims_of(inputs, shapes)
    plan = op.plans_for(env)[-1]
    zero = {n: 0 for n in plan.args}
    assert plan.choose(env, zero)[0] in (plan.variants['matrixv'], plan.variants['matrix64v'])
    odd = {k: (v + 2 if k in ('M', 'D') else v) for k, v in env.items()}          # a row length that is no whole number of vectors
    assert plan.choose(odd, zero)[0] in (plan.variants['matrix'], plan.variants['matrix64'])
    g = torch.Generator().manual_seed(len(ir))
    a, b = [(torch.randn(shape, generator=g) * 0.5).to(torch.float16 if 'float16' in inputs[0] else torch.float32) for shape in shapes]
    want = CpuModule(parse_program(ir, inputs), fast_math=False)(input0=a.numpy(), input1=b.numpy())['output0']
    M, N, B = (int(np.prod([e if isinstance(e, int) else env[e] for e in plan.matrix[k]])) for k in ('m', 'n', 'batch'))
    got = {}
    for tag, side in (('matrix', 128), ('matrix64', 64), ('matrixv', 128), ('matrix64v', 64)):
        blocks = ((M + side - 1) // side) * ((N + side - 1) // side) * B
        plan.choose = lambda env_, ptrs, tag=tag, blocks=blocks: (plan.variants[tag], blocks, 256)
        got[tag] = op(a.to(dev), b.to(dev)).cpu().numpy()
        assert np.allclose(got[tag], want, rtol=1e-4, atol=1e-3), (tag, np.abs(got[tag] - want).max())
    # the same products in the same order of k inside a tile: the bits agree between the two ways of staging
    assert np.array_equal(got['matrix'], got['matrixv']) and np.array_equal(got['matrix64'], got['matrix64v'])


@pytest.mark.parametrize('ir,inputs,shapes', [
    ('output0[N, M] +=! input0[N, K].cast(`int32`) * input1[M, K].cast(`int32`)', ['input0=int8[N:1000, K:528]', 'input1=int8[M:1024, K:528]'],
     [(1000, 528), (1024, 528)]),
    ('output0[N, M] +=! input0[N, K].cast(`int32`) * input1[K, M].cast(`int32`)', ['input0=int8[N:300, K:200]', 'input1=int8[K:200, M:260]'],
     [(300, 200), (200, 260)]),
    ('output0[B, N, M] +=! input0[B, N, K].cast(`int32`) * input1[B, M, K].cast(`int32`)', ['input0=int8[B:2, N:256, K:4096]', 'input1=int8[B:2, M:192, K:4096]'],
     [(2, 256, 4096), (2, 192, 4096)]),
    # the second operand stored along its columns, whole vectors of them: staged as it lies, transposed by ds_read_b64_tr_b8
    ('output0[N, M] +=! input0[N, K].cast(`int32`) * input1[K, M].cast(`int32`)', ['input0=int8[N:200, K:160]', 'input1=int8[K:160, M:272]'],
     [(200, 160), (160, 272)]),
])
def test_int8_contractions_are_bit_exact_on_the_matrix_instructions(autort, ir, inputs, shapes):
    """An int32 sum of products of two int8 loads cast to int32 runs on v_mfma_i32_32x32x32_i8: exact products, exact
    sums, and integer sums do not depend on their order - every kernel gives the integers of a 64-bit product (and the
    oracle's), bit for bit; the third case is also cut into slices of k."""
    from antares_amd.ir import parse_program
    from oracle.cpu_backend import CpuModule
    note(f'int8 contraction on the matrix instructions {ir} {shapes}')
    dev = autort.device()
    op = autort.export(ir=ir, inputs=inputs, name='mfma_i8_' + str(abs(hash((ir, tuple(inputs)))) % 10 ** 8))
    op.fast_path = None
    env = dims_of(inputs, shapes)
    plan = op.plans_for(env)[0]
    assert plan.matrix is not None and len(op.plans_for(env)) == (2 if 'B:2' in inputs[0] else 1)
    g = torch.Generator().manual_seed(len(ir))
    a, b = [torch.randint(-128, 128, shape, generator=g, dtype=torch.int8) for shape in shapes]
    exact = torch.einsum('...nk,...km->...nm', a.long(), b.long() if ir.split('input1')[1].startswith('[K, M]') else b.long().transpose(-1, -2)).to(torch.int32).numpy()
    if a.numel() <= 1 << 20:
        want = CpuModule(parse_program(ir, inputs), fast_math=False)(input0=a.numpy(), input1=b.numpy())['output0']
        assert np.array_equal(want, exact)
    M, N, B = (int(np.prod([e if isinstance(e, int) else env[e] for e in plan.matrix[k]])) for k in ('m', 'n', 'batch'))
    for tag, side in (('matrix', 128), ('matrix64', 64), ('matrixv', 128), ('matrix64v', 64)):
        if tag not in plan.variants or (tag.endswith('v') and not (plan._matrix_choice(env, {n: 0 for n in plan.args})[0] or '').endswith('v')):
            continue                # the vector kernels are launched for whole vectors only
        blocks = ((M + side - 1) // side) * ((N + side - 1) // side) * B
        plan.choose = lambda env_, ptrs, tag=tag, blocks=blocks: (plan.variants[tag], blocks, 256)
        got = op(a.to(dev), b.to(dev))
        assert got.dtype == torch.int32 and np.array_equal(got.cpu().numpy(), exact), tag


@pytest.mark.parametrize('in_kernel', [False, True])
def test_int8_padded_convolution_is_bit_exact(autort, monkeypatch, in_kernel):
    """A zero-padded 3 x 3 convolution of int8 images and filters into int32 on v_mfma_i32_32x32x32_i8, with the image
    copied into a padded tensor first and with the conditions evaluated in the contraction: torch's integers both ways."""
    note(f'int8 padded convolution, guards {"in the kernel" if in_kernel else "in a padded copy"}')
    dev = autort.device()
    if in_kernel:
        monkeypatch.setattr('antares_amd.autort.op.pad_guarded_factors', lambda graph, env=None: graph)
    ir = ('output0[N, F, HO, WO] +=! input0[N, C, HO + KH - 1, WO + KW - 1].cast(`int32`).when([HO + KH - 1 >= 0, HO + KH - 1 < 20, '
          'WO + KW - 1 >= 0, WO + KW - 1 < 20], 0) * input1[F, C, KH, KW].cast(`int32`) where HO in 20, WO in 20')
    op = autort.export(ir=ir, inputs=['input0=int8[N:3, C:24, H:20, W:20]', 'input1=int8[F:72, C:24, KH:3, KW:3]'], name=f'conv_i8_{int(in_kernel)}')
    env = {'N': 3, 'C': 24, 'H': 20, 'W': 20, 'F': 72, 'KH': 3, 'KW': 3}
    plans = op.plans_for(env)
    assert len(plans) == (1 if in_kernel else 2) and plans[-1].matrix is not None and plans[-1].matrix['half_tiles']
    g = torch.Generator().manual_seed(9)
    x, w = torch.randint(-128, 128, (3, 24, 20, 20), generator=g, dtype=torch.int8), torch.randint(-128, 128, (72, 24, 3, 3), generator=g, dtype=torch.int8)
    want = torch.nn.functional.conv2d(x.double(), w.double(), padding=1).to(torch.int32)        # sums below 2^53: exact
    got = op(x.to(dev), w.to(dev)).cpu()
    assert got.dtype == torch.int32 and torch.equal(got, want)


TAIL_CASES = [
    # AntaresIR.md:248-250 (ConvBiasRelu tail fusion); a product with a scaled result, a per-column and a per-element
    # term under a tanh; a float16 result of a float32 sum; a column-wise maximum with a conditional store behind it
    ('conv_out[N, F, HO, WO] +=! input0[N, C, HO + KH, WO + KW] * input1[KH, KW, C, F] where HO in 30, WO in 30; '
     'conv_bias[N, F, HO, WO] = conv_out[N, F, HO, WO] + input2[0, 0, 0, F]; '
     'output0[N, F, HO, WO] = conv_bias[N, F, HO, WO].when(conv_bias[N, F, HO, WO] > 0.0, 0.0)',
     ['input0=float32[N:4, C:16, H:32, W:32]', 'input1=float32[KH:3, KW:3, C:16, F:64]', 'input2=float32[1, 1, 1, F:64]'],
     [(4, 16, 32, 32), (3, 3, 16, 64), (1, 1, 1, 64)], True),
    ('acc[N, M] +=! input0[N, K] * input1[M, K]; output0[N, M] = (acc[N, M] * 0.5 + input2[M] + input3[N, M]).call(`tanh`)',
     ['input0=float32[N:300, K:256]', 'input1=float32[M:200, K:256]', 'input2=float32[M:200]', 'input3=float32[N:300, M:200]'],
     [(300, 256), (200, 256), (200,), (300, 200)], True),
    ('acc[B, N, M] +=! input0[B, N, K].to(`float32`) * input1[B, K, M].to(`float32`); output0[B, N, M] = (acc[B, N, M] + input2[B, M]).to(`float16`)',
     ['input0=float16[B:3, N:128, K:64]', 'input1=float16[B:3, K:64, M:160]', 'input2=float32[B:3, M:160]'], [(3, 128, 64), (3, 64, 160), (3, 160)], True),
    ('top[C] >=! input0[N, C]; output0[C] = top[C].when(top[C] > input1[C])', ['input0=float32[N:40, C:20000]', 'input1=float32[C:20000]', 'output0=float32[C:20000]'],
     [(40, 20000), (20000,), (20000,)], False),
]


@pytest.mark.parametrize('ir,inputs,shapes,matrix', TAIL_CASES)
def test_a_map_behind_a_reduction_is_applied_at_its_stores(autort, ir, inputs, shapes, matrix):
    """Tail fusion (AntaresIR.md:248-250): the kernels of the reduction store f(result, other tensors) straight into the
    map's output; the reduction's own output is never written and the map's kernels are not launched.  Every variant of
    the fused kernels against the oracle, which runs the statements one by one."""
    from antares_amd.ir import parse_program
    from oracle.cpu_backend import CpuModule
    note(f'tail fusion {ir[:60]} {shapes}')
    dev = autort.device()
    op = autort.export(ir=ir, inputs=inputs, name='tail_' + str(abs(hash((ir, tuple(inputs)))) % 10 ** 8))
    op.fast_path = None
    env = dims_of(inputs, shapes)
    plans = op.plans_for(env)
    assert len(plans) == 2 and plans[0].covers == 2 and plans[0].output == 'output0' and plans[0].args[-1] == 'output0'
    assert not any(a in plans[0].args for a in ('acc', 'conv_out', 'top'))
    assert ('matrix' in plans[0].variants) == matrix
    g = torch.Generator().manual_seed(len(ir))
    tensors = [(torch.randn(shape, generator=g) * 0.5).to(torch.float16 if 'float16' in spec else torch.float32) for spec, shape in zip(inputs, shapes)]
    names = [spec.split('=')[0] for spec in inputs]
    want = CpuModule(parse_program(ir, inputs), fast_math=False)(**{n: t.numpy().copy() for n, t in zip(names, tensors)})['output0'].astype(np.float32)
    plan, total = plans[0], int(np.prod(want.shape))
    launches = [('thread', (total + 255) // 256), ('wave', (total + 3) // 4), ('block', total)]
    if 'patch' in plan.variants and plan._patches(env, total):
        launches.append(('patch', (plan._patches(env, total) + 255) // 256))
    if matrix:
        M, N, B = (int(np.prod([e if isinstance(e, int) else env[e] for e in plan.matrix[k]])) for k in ('m', 'n', 'batch'))
        launches += [(tag, ((M + side - 1) // side) * ((N + side - 1) // side) * B) for tag, side in (('matrix', 128), ('matrix64', 64)) if tag in plan.variants]
        if (plan._matrix_choice(env, {n: 0 for n in plan.args})[0] or '').endswith('v'):       # whole vectors everywhere they are fetched
            launches += [(tag, ((M + side - 1) // side) * ((N + side - 1) // side) * B) for tag, side in (('matrixv', 128), ('matrix64v', 64))]
    tol = 1e-2 if want.dtype == np.float16 or 'float16' in ir else 2e-4
    for tag, grid in launches:
        plan.choose = lambda env_, ptrs, tag=tag, grid=grid: (plan.variants[tag], min(grid, 65536), 256)
        got = op(*[t.clone().to(dev) for t in tensors]).float().cpu().numpy()
        assert got.shape == want.shape and np.allclose(got, want, rtol=tol, atol=tol), (tag, np.abs(got - want).max())


def test_one_operator_called_at_several_sizes_gets_the_rewrites_of_each(autort):
    """A padded convolution with bias and ReLU exported once with named dimensions and called with three batch sizes and
    two filter sizes: every call finds (or builds) the kernels of its own dimension values - filter size written in,
    operand padded by a statement in front, tail applied at the stores - and gives torch's result."""
    note('padded conv + bias + relu at several sizes through one operator')
    dev = autort.device()
    ir = ('conv[N, F, HO, WO] +=! input0[N, C, HO + KH - KH.val() / 2, WO + KW - KW.val() / 2].when([HO + KH - KH.val() / 2 >= 0, '
          'HO + KH - KH.val() / 2 < 24, WO + KW - KW.val() / 2 >= 0, WO + KW - KW.val() / 2 < 24], 0.0) * input1[F, C, KH, KW] where HO in 24, WO in 24; '
          'output0[N, F, HO, WO] = (conv[N, F, HO, WO] + input2[F]).call(`max`, [0.0])')
    op = autort.export(ir=ir, inputs=['input0=float32[N:4, C:16, H:24, W:24]', 'input1=float32[F:64, C:16, KH:3, KW:3]', 'input2=float32[F:64]'],
                       name='conv_bias_relu_sizes')
    g = torch.Generator().manual_seed(5)
    seen = set()
    for n, k in ((4, 3), (2, 3), (7, 5), (4, 3)):
        x, w, b = torch.randn(n, 16, 24, 24, generator=g), torch.randn(64, 16, k, k, generator=g) * 0.1, torch.randn(64, generator=g)
        got = op(x.to(dev), w.to(dev), b.to(dev)).cpu()
        want = torch.relu(torch.nn.functional.conv2d(x.double(), w.double(), b.double(), padding=k // 2)).float()
        assert got.shape == want.shape and torch.allclose(got, want, rtol=1e-4, atol=1e-3), (n, k, (got - want).abs().max())
        seen.add((n, k))
        assert len(op._variants) == len(seen)
    env = {'N': 7, 'C': 16, 'H': 24, 'W': 24, 'F': 64, 'KH': 5, 'KW': 5}
    plans = op.plans_for(env)
    # the copy padded by two on each side, then the contraction with the tail at its stores (the map's own plan is not launched)
    assert [p.output for p in plans] == ['input0__pad', 'output0', 'output0'] and plans[1].covers == 2 and plans[1].matrix is not None
    assert dict(plans[1].reduce_axes)['KH'] == 5


ROW_GROUP_CASES = [
    # program, inputs, shapes, does the row kernel run at these extents
    ('temp0[N] >=! input0[N, C]; temp1[N] +=! (input0[N, C] - temp0[N]).call(`exp`); '
     'output0[N, C] = (input0[N, C] - temp0[N]).call(`exp`) / temp1[N]', ['input0=float32[N:37, C:1000]'], [(37, 1000)], True),
    ('temp0[N] +=! input0[N, C]; temp1[N] +=! input0[N, C] * input0[N, C]; '
     'output0[N, C] = (input0[N, C] * C.val() - temp0[N]) * (temp1[N] * C.val() - temp0[N] * temp0[N] + 1e-5).call(`rsqrt`)',
     ['input0=float32[N:32, C:1024]'], [(32, 1024)], True),
    # rows of a 3-D tensor, a per-column weight and a per-row shift besides the row itself, fp16 storage
    ('ss[B, N] +=! x[B, N, C].to(`float32`) * x[B, N, C].to(`float32`); '
     'y[B, N, C] = (x[B, N, C].to(`float32`) * (ss[B, N] / C.val() + 1e-5).call(`rsqrt`) * w[C].to(`float32`) + shift[B, N]).to(`float16`)',
     ['x=float16[B:3, N:17, C:520]', 'w=float16[C:520]', 'shift=float32[B:3, N:17]'], [(3, 17, 520), (520,), (3, 17)], True),
    # integer rows: maximum and count of the maxima, exact
    ('top[N] >=! v[N, C]; hits[N] +=! (v[N, C] == top[N]).to(`int32`); out[N, C] = (top[N] - v[N, C]) * hits[N]',
     ['v=int32[N:50, C:300]'], [(50, 300)], True),
    # many short rows (a wavefront per row), fp16 vectors of 8; a long row that is walked; a row of 16 vectors per lane
    ('ss[N] +=! x[N, C].to(`float32`) * x[N, C].to(`float32`); '
     'y[N, C] = (x[N, C].to(`float32`) * (ss[N] / C.val() + 1e-5).call(`rsqrt`) * w[C].to(`float32`)).to(`float16`)',
     ['x=float16[N:9001, C:264]', 'w=float16[C:264]'], [(9001, 264), (264,)], True),
    ('temp0[N] +=! input0[N, C]; temp1[N] +=! input0[N, C] * input0[N, C]; '
     'output0[N, C] = (input0[N, C] * C.val() - temp0[N]) * (temp1[N] * C.val() - temp0[N] * temp0[N] + 1e-5).call(`rsqrt`)',
     ['input0=float32[N:5, C:20001]'], [(5, 20001)], True),
    ('temp0[N] +=! input0[N, C]; temp1[N] +=! input0[N, C] * input0[N, C]; '
     'output0[N, C] = (input0[N, C] * C.val() - temp0[N]) * (temp1[N] * C.val() - temp0[N] * temp0[N] + 1e-5).call(`rsqrt`)',
     ['input0=float32[N:9, C:12000]'], [(9, 12000)], True),
    # reductions with no map behind them: row sums, an integer row maximum of products with a weight row
    ('output0[N] +=! input0[N, C]', ['input0=float32[N:600, C:1000]'], [(600, 1000)], True),
    ('top[B, N] >=! v[B, N, C] * w[C]', ['v=int32[B:2, N:300, C:300]', 'w=int32[C:300]'], [(2, 300, 300), (300,)], True),
    # short rows: the per-statement kernels run, same result
    ('temp0[N] >=! input0[N, C]; temp1[N] +=! (input0[N, C] - temp0[N]).call(`exp`); '
     'output0[N, C] = (input0[N, C] - temp0[N]).call(`exp`) / temp1[N]', ['input0=float32[N:300, C:64]'], [(300, 64)], False),
]


@pytest.mark.parametrize('ir,inputs,shapes,applies', ROW_GROUP_CASES)
def test_row_reductions_and_their_map_run_as_one_kernel(autort, ir, inputs, shapes, applies):
    """Reductions over the last axis followed by the map that uses them (softmax, layer normalisation,
    AntaresIR.md:226-232) are computed by one kernel, a block per row; results are the oracle's, and they equal
    what the per-statement kernels give to the rounding of the reductions."""
    from antares_amd.ir import parse_program
    from oracle.cpu_backend import CpuModule
    note(f'row group {ir[:40]} {shapes}')
    dev = autort.device()
    op = autort.export(ir=ir, inputs=inputs, name='rows_' + str(abs(hash((ir, tuple(inputs)))) % 10 ** 8))
    group = op.plans[0].row_group
    assert group is not None and group.count == len(op.plans) == ir.count(';') + 1
    env = {}
    for spec, shape in zip(inputs, shapes):
        for d, v in zip(spec.split('[', 1)[1].rstrip(']').split(','), shape):
            env[d.split(':')[0].strip()] = v
    assert (group.choose(env, {n: 0 for n in group.args})[1] > 0) == applies
    g = torch.Generator().manual_seed(len(ir))
    tensors, names = [], []
    for spec, shape in zip(inputs, shapes):
        name, rest = spec.split('=')
        names.append(name)
        if rest.startswith('int32'):
            tensors.append(torch.randint(-40, 40, shape, generator=g, dtype=torch.int32))
        else:
            tensors.append(torch.randn(shape, generator=g).to(torch.float16 if rest.startswith('float16') else torch.float32))
    got = op(*[t.to(dev) for t in tensors]).cpu().numpy()
    out_name = ir.rsplit(';', 1)[-1].split('[', 1)[0].strip()
    want = CpuModule(parse_program(ir, inputs), fast_math=False)(**{n: t.numpy() for n, t in zip(names, tensors)})[out_name]
    if got.dtype.kind == 'i':
        assert np.array_equal(got, want)
    else:
        tol = 2e-2 if got.dtype == np.float16 else 2e-5
        assert np.allclose(got.astype(np.float64), want.astype(np.float64), rtol=tol, atol=tol), np.abs(got.astype(np.float64) - want).max()
    # statement by statement (the row kernel switched off): same values up to the order of the sums
    for p in op.plans:
        p.row_group = None
    apart = op(*[t.to(dev) for t in tensors]).cpu().numpy()
    if got.dtype.kind == 'i':
        assert np.array_equal(got, apart)
    else:
        assert np.allclose(got.astype(np.float64), apart.astype(np.float64), rtol=tol, atol=tol)


SHORT_ROWS = {
    'softmax': ('temp0[N] >=! input0[N, C]; temp1[N] +=! (input0[N, C] - temp0[N]).call(`exp`); '
                'output0[N, C] = (input0[N, C] - temp0[N]).call(`exp`) / temp1[N]'),
    'sum': 'temp0[N] +=! input0[N, C]; output0[N, C] = input0[N, C] - temp0[N] * C.val()',
}


# a row in 16 lanes: lanes with one element and with eight, the last length of every form and the first of the next, rows that end inside a
# block, vectors from the first length that gives every lane one; addresses and lengths that take vectors away
@pytest.mark.parametrize('program,dtype', [('softmax', 'float32'), ('softmax', 'float16'), ('softmax', 'float64'), ('sum', 'int32'), ('sum', 'int8')])
@pytest.mark.parametrize('rows,n,offset', [(1, 16, 0), (15, 17, 0), (17, 32, 0), (33, 33, 0), (1000, 63, 0), (16, 64, 0), (47, 64, 1), (31, 65, 0), (50, 124, 0), (8200 * 16 + 3, 127, 0)])
def test_rows_of_fewer_than_two_wavefronts(autort, program, dtype, rows, n, offset):
    """One kernel, four rows to a wavefront, and the statements one by one: exact for whole numbers, else both within (n + 8) roundings of the
    sums, the exponentials and the quotient of the float64 result.  Infinities, NaN and rows of the type's lowest value included."""
    if dtype == 'int8' and n > 100 or dtype == 'float64' and rows > 100000:
        pytest.skip('sums past int8, or a large case once more')
    note(f'short rows {program} {dtype} {rows} x {n} at {offset}')
    dev, t = autort.device(), getattr(torch, dtype)
    op = autort.export(ir=SHORT_ROWS[program], inputs=[f'input0={dtype}[N:64, C:100]'], name=f'short_{program}_{dtype}')
    g = torch.Generator().manual_seed(rows + n)
    x = torch.randint(-1, 2, (rows, n), generator=g).to(t) if program == 'sum' else torch.randn(rows, n, generator=g).to(t)
    special = program == 'softmax' and rows > 8
    if special:
        x[1, 3], x[2], x[3, 0], x[4], x[5, n - 1] = float('-inf'), float('-inf'), float('nan'), torch.finfo(t).min, float('inf')
    xd = torch.zeros(rows * n + offset, dtype=t, device=dev)[offset:].view(rows, n).copy_(x)
    group = op.plans[0].row_group
    pointers = {a: (4 if offset else 0) for a in group.args}
    assert group.choose({'N': rows, 'C': n}, pointers)[1] == 0 and group.choose_short({'N': rows, 'C': n}, pointers)[1] > 0
    assert group.choose_short({'N': rows, 'C': 15}, pointers)[1] == 0
    together = op(xd).cpu()
    try:
        for p in op.plans:
            p.row_group = None
        apart = op(xd).cpu()
    finally:
        op.plans[0].row_group = group
    if program == 'sum':
        assert torch.equal(together, apart) and torch.equal(together.long(), x.long() - x.long().sum(1, keepdim=True) * n)
        return
    want = torch.softmax(x.double(), 1)
    eps = torch.finfo(t).eps
    for got in (together, apart):
        assert torch.equal(got.isnan(), want.isnan())
        fine = ~want.isnan()
        # an exponent is off by the rounding of its difference, at most 40 here but for the lowest values, which are all equal
        assert bool(((got.double() - want)[fine].abs() <= want[fine] * (n + 60) * eps + torch.finfo(t).tiny).all())


# vectors that start anywhere: the first and the last length of every form, rows of whole vectors at odd addresses, rows that end inside a block
@pytest.mark.parametrize('program,dtype', [('softmax', 'float32'), ('sum', 'int32')])
@pytest.mark.parametrize('rows,n,offset', [(3, 128, 0), (7, 129, 0), (5, 253, 1), (1001, 256, 0), (515, 257, 0), (514, 511, 0), (513, 512, 1), (8195, 513, 0), (8193, 1023, 0), (8193, 1024, 3),
                                           (2, 1025, 0), (1, 2047, 2), (3, 4097, 0), (2, 8191, 0), (1025, 8192, 0)])
def test_rows_in_vectors_that_start_anywhere(autort, program, dtype, rows, n, offset):
    """One kernel, and the statements one by one: exact for whole numbers, else both within (n + 8) roundings of the sums, the exponentials and the
    quotient of the float64 result.  Infinities, NaN and rows of the type's lowest value included."""
    note(f'ragged rows {program} {dtype} {rows} x {n} at {offset}')
    dev, t = autort.device(), getattr(torch, dtype)
    op = autort.export(ir=SHORT_ROWS[program], inputs=[f'input0={dtype}[N:64, C:100]'], name=f'ragged_{program}_{dtype}')
    g = torch.Generator().manual_seed(rows + n)
    x = torch.randint(-1, 2, (rows, n), generator=g).to(t) if program == 'sum' else torch.randn(rows, n, generator=g)
    if program == 'softmax' and rows > 8:
        x[1, 3], x[2], x[3, 0], x[4], x[5, n - 1], x[6, n - 2] = float('-inf'), float('-inf'), float('nan'), torch.finfo(t).min, float('inf'), float('-inf')
    xd = torch.zeros(rows * n + offset, dtype=t, device=dev)[offset:].view(rows, n).copy_(x)
    group = op.plans[0].row_group
    assert group.choose_ragged({'N': rows, 'C': n}, {a: (4 * offset if a == 'input0' else 0) for a in group.args})[1] > 0
    together = op(xd).cpu()
    try:
        for p in op.plans:
            p.row_group = None
        apart = op(xd).cpu()
    finally:
        op.plans[0].row_group = group
    if program == 'sum':
        assert torch.equal(together, apart) and torch.equal(together.long(), x.long() - x.long().sum(1, keepdim=True) * n)
        return
    want = torch.softmax(x.double(), 1)
    eps = torch.finfo(t).eps
    for got in (together, apart):
        assert torch.equal(got.isnan(), want.isnan())
        fine = ~want.isnan()
        assert bool(((got.double() - want)[fine].abs() <= want[fine] * (n + 60) * eps + torch.finfo(t).tiny).all())


@pytest.mark.parametrize('rows,n,form', [(65537, 67, 'q8'), (8193, 255 + 1, 'w4v4'), (8193, 257, 'rw2'), (8193, 601, 'rw4'), (2049, 1024, 'b4v4'), (2101, 1025, 'rb2'), (1100, 4100, 'rb8'), (257, 8196, 'b16v4'), (129, 16391, '')])
def test_large_results_of_rows_past_the_caches(autort, rows, n, form):
    """A kernel that stores past the caches gives the bits of the one that does not."""
    note(f'rows past the caches {rows} x {n}')
    op = autort.export(ir=SHORT_ROWS['softmax'], inputs=['input0=float32[N:64, C:100]'], name='past_softmax')
    x = torch.randn(rows, n, generator=torch.Generator().manual_seed(n)).to(autort.device())
    group, taken = op.plans[0].row_group, []
    choose = group.choose_stores
    try:
        group.choose_stores = lambda sym, env: taken.append(choose(sym, env)) or taken[-1]
        past = op(x).clone()
        group.choose_stores = lambda sym, env: sym
        through = op(x)
    finally:
        del group.choose_stores
    assert taken == [f'{group.symbol}{"_" + form if form else ""}_past']
    assert torch.equal(past, through) and torch.allclose(past, torch.softmax(x, 1), rtol=1e-4, atol=1e-7)


@pytest.mark.parametrize('reduce', ['>', '<'])
@pytest.mark.parametrize('rows,n,offset', [(36, 129, 0), (38, 254, 0), (37, 255, 1), (514, 511, 0), (8195, 601, 0), (36, 1026, 0), (41, 4099, 0), (1025, 4100, 0)])       # a form of these kernels each
def test_extremes_of_rows_in_vectors_that_start_anywhere_skip_a_nan(autort, reduce, rows, n, offset):
    """A NaN at each place of the first, an inner and the last vector of a row (which overlaps the one before), beside the row's extreme at each
    other place: as the statements one by one, the row minus the extreme of its other values, to the bit."""
    note(f'ragged rows {reduce} with NaN {rows} x {n} at {offset}')
    dev, sign = autort.device(), 1.0 if reduce == '>' else -1.0
    op = autort.export(ir=f't[N] {reduce}=! x[N, C]; y[N, C] = x[N, C] - t[N]', inputs=['x=float32[N:64, C:200]'], name=f'extreme_{"max" if sign > 0 else "min"}')
    x = torch.randn(rows, n, generator=torch.Generator().manual_seed(n)) * sign
    places = [(first, a, b) for first in (0, 64, n - 4) for a in range(4) for b in range(4) if a != b]
    for row, (first, a, b) in enumerate(places):
        x[row, first + a], x[row, first + b] = float('nan'), sign * (100 + row)
    xd = torch.zeros(rows * n + offset, device=dev)[offset:].view(rows, n).copy_(x)
    group = op.plans[0].row_group
    assert group.choose_ragged({'N': rows, 'C': n}, {v: (4 * offset if v == 'x' else 0) for v in group.args})[1] > 0
    together = op(xd).cpu()
    try:
        for p in op.plans:
            p.row_group = None
        apart = op(xd).cpu()
    finally:
        op.plans[0].row_group = group
    want = x - x.nan_to_num(nan=-sign * 1e30).mul(sign).max(1, keepdim=True).values * sign
    for got in (together, apart):
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(), want.nan_to_num())


@pytest.mark.parametrize('ir,ta,tb,M,N,K', [
    ('out[M, N] +=! x[K, M] * w[K, N]', True, False, 1028, 512, 96),
    ('out[M, N] +=! x[M, K] * w[N, K]', False, True, 1000, 1030, 64),       # a linear layer: N need not be a multiple of 4
    ('out[M, N] +=! x[K, M] * w[N, K]', True, True, 2048, 129, 160),
    ('out[M, N] +=! x[M, K] * w[N, K]', False, True, 4096, 4096, 1024),
])
def test_fp32_gemm_with_operands_stored_the_other_way_round(autort, ir, ta, tb, M, N, K):
    """`A^T B`, `A B^T` and `A^T B^T` in float32 go to art_gemm_f32_ex; results are the float64 products' to fp32
    accuracy, and a one-hot operand pins which axis of each operand is k."""
    note(f'gemm_f32 layouts {ir} {M}x{N}x{K}')
    dev = autort.device()
    sa, sb = (f'x=float32[K:{K}, M:{M}]' if ta else f'x=float32[M:{M}, K:{K}]'), (f'w=float32[N:{N}, K:{K}]' if tb else f'w=float32[K:{K}, N:{N}]')
    op = autort.export(ir=ir, inputs=[sa, sb], name=f'gemm_f32_l{int(ta)}{int(tb)}_{M}_{N}_{K}')
    assert op.fast_path is not None
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.randn((K, M) if ta else (M, K), generator=g)
    b = torch.randn((N, K) if tb else (K, N), generator=g)
    got = op(a.to(dev), b.to(dev)).cpu()
    am, bm = (a.t() if ta else a).double(), (b.t() if tb else b).double()
    want = am @ bm
    assert torch.allclose(got.double(), want, rtol=1e-5, atol=1e-5 * max(1.0, K ** 0.5)), (got.double() - want).abs().max()
    if M <= 2048:
        sel = torch.zeros(M, K)
        sel[torch.arange(M), torch.arange(M) % K] = 1.0              # row m of the result = row m % K of B
        sel_in = sel.t().contiguous() if ta else sel
        assert torch.equal(op(sel_in.to(dev), b.to(dev)).cpu(), (b.t() if tb else b)[torch.arange(M) % K].contiguous())


def conv_program(dtype, hw, out, pads, guard=True):
    """A 3 x 3 convolution over hw = (H, W) with pads = (ph, pw) and results of out = (HO, WO)."""
    cast = '.to(`float32`)' if dtype == 'float16' else ''
    idx = [f'{a}O + K{a} - {p}' if p > 0 else f'{a}O + K{a} + {-p}' for a, p in zip('HW', pads)]
    when = f'.when([{idx[0]} >= 0, {idx[0]} < {hw[0]}, {idx[1]} >= 0, {idx[1]} < {hw[1]}], 0.0)' if guard else ''
    return (f'output0[N, F, HO, WO] +=! input0[N, C, {idx[0]}, {idx[1]}]{cast}{when} * input1[F, C, KH, KW]{cast} '
            f'where HO in {out[0]}, WO in {out[1]}')


CONV_CASES = [  # N, C, (H, W), F, (ph, pw), (HO, WO), guarded
    (2, 16, (9, 9), 33, (1, 1), (9, 9), True),             # a block spans several images, one more feature than a tile
    (3, 33, (13, 17), 64, (1, 1), (13, 17), True),         # channels one past a chunk, a wide image
    (1, 70, (40, 3), 130, (1, 1), (40, 3), True),          # rows of three points, a block of two features
    (5, 24, (8, 8), 48, (0, 0), (6, 6), False),            # no padding: no guards
    (2, 20, (12, 10), 40, (2, 0), (14, 7), True),          # padded on one axis by two, results short of the other's end
    (1, 16, (1, 1), 32, (1, 1), (1, 1), True),             # one point
    (4, 8, (30, 31), 20, (-1, 1), (27, 31), True),         # taps that start inside
]
CONV_WIDE = (2, 33, (5, 200), 21, (1, 1), (5, 200), True)  # gathered by a block that has a compute unit's LDS to itself (float16 64 x 64)


@pytest.mark.parametrize('dtype,form,case', [(d, f, c) for c in CONV_CASES for f in (1, 2, 3) for d in ('float16', 'float32')] + [('float16', 1, CONV_WIDE)])
def test_convolution_blocks_match_float64(autort, dtype, form, case):
    """Each block shape of the convolution kernel against the same sum in 64 bits: products of float16 are exact in
    float32, so the error is that of float32 sums of 9 C terms in any order."""
    from ctypes import c_void_p
    from antares_amd.runtime import capi
    N, C, (H, W), F, (ph, pw), (HO, WO), _ = case
    note(f'convolution {dtype} form {form} {case}')
    g = torch.Generator().manual_seed(N * 1000 + C)
    x = torch.randn(N, C, H, W, generator=g).to(getattr(torch, dtype))
    w = torch.randn(F, C, 3, 3, generator=g).to(getattr(torch, dtype))
    f16 = int(dtype == 'float16')
    shape = (f16, N, C, H, W, F, HO, WO, ph, pw)
    lib = capi.lib()
    assert lib.art_conv2d_form(*shape, form) == form
    dev = autort.device()
    xd, wd = x.to(dev), w.to(dev)
    y = torch.full((N, F, HO, WO), 7.0, device=dev)
    packed = torch.empty(lib.art_conv2d_packed_bytes(f16, C, F), dtype=torch.uint8, device=dev)
    capi.check(lib.art_conv2d(*(c_void_p(t.data_ptr()) for t in (xd, wd, packed, y)), *shape, form, c_void_p(torch.cuda.current_stream().cuda_stream)))
    pad = max(ph, pw, 0) + 2
    big = torch.nn.functional.conv2d(torch.nn.functional.pad(x.double(), (pad, pad + 2, pad, pad + 2)), w.double())
    want = big[:, :, pad - ph:pad - ph + HO, pad - pw:pad - pw + WO]
    bound = 2.0 ** -23 * 9 * C * torch.nn.functional.conv2d(
        torch.nn.functional.pad(x.double().abs(), (pad, pad + 2, pad, pad + 2)), w.double().abs())[:, :, pad - ph:pad - ph + HO, pad - pw:pad - pw + WO]
    assert ((y.cpu().double() - want).abs() <= bound + 1e-30).all()


@pytest.mark.parametrize('dtype,form,case', [(d, f, c) for c in (
    (3, 40, (20, 1), 40, (1, 1), (20, 1), True),           # a point to a row: gathered one by one
    (2, 24, (33, 2), 40, (1, 1), (33, 2), True),           # both points of a pair, and one of each of two
    (2, 33, (7, 9), 70, (0, 0), (5, 7), False),            # odd rows without padding: no point outside between two rows
    (1, 16, (6, 11), 33, (1, 3), (7, 13), True),           # pairs that begin two points outside
) for f in (1, 2, 3) for d in ('float16', 'float32')])
def test_convolutions_gathered_two_points_at_a_time_match_float64(autort, dtype, form, case):
    test_convolution_blocks_match_float64(autort, dtype, form, case)


@pytest.mark.parametrize('dtype', ['float16', 'float32'])
@pytest.mark.parametrize('case', CONV_CASES + [(1, 100, (11, 57), 70, (1, 1), (11, 57), True),      # several chunks, a row longer than a block of 64
                                               (2, 40, (120, 5), 200, (1, 1), (120, 5), True)])     # many rows to a block
def test_staged_convolution_blocks_match_float64(autort, dtype, case):
    """Every form over the staged image, whole and in slices of the channels, with scratch that holds NaN: nothing is read that
    was not written.  The bound is that of the gathering forms, one addition per slice more; the short sums (form 7) are held
    to 2^-24 for each of a chain of 7 and two roundings."""
    from ctypes import c_void_p
    from antares_amd.runtime import capi
    N, C, (H, W), F, (ph, pw), (HO, WO), _ = case
    note(f'staged convolution {dtype} {case}')
    g = torch.Generator().manual_seed(N * 1000 + C + W)
    x, w = torch.randn(N, C, H, W, generator=g).to(getattr(torch, dtype)), torch.randn(F, C, 3, 3, generator=g).to(getattr(torch, dtype))
    f16 = int(dtype == 'float16')
    shape = (f16, N, C, H, W, F, HO, WO, ph, pw)
    lib, dev = capi.lib(), autort.device()
    xd, wd = x.to(dev), w.to(dev)
    pad = max(ph, pw, 0) + 2

    def reference(a, b):
        return torch.nn.functional.conv2d(torch.nn.functional.pad(a, (pad, pad + 2, pad, pad + 2)), b)[:, :, pad - ph:pad - ph + HO, pad - pw:pad - pw + WO]
    want, size = reference(x.double(), w.double()), reference(x.double().abs(), w.double().abs())
    chunks = -(-C // (32 if f16 else 16))
    for kind in (4, 5, 6) if f16 else (4, 5, 6, 7):
        for slices in sorted({1, 2, 3, chunks}):
            form = kind + 256 * slices
            if slices > chunks:
                assert lib.art_conv2d_form(*shape, form) == 0
                continue
            assert lib.art_conv2d_form(*shape, form) == form
            y = torch.full((N, F, HO, WO), 7.0, device=dev)
            scratch = torch.full((lib.art_conv2d_scratch_bytes(*shape, form),), 255, dtype=torch.uint8, device=dev)
            capi.check(lib.art_conv2d(*(c_void_p(t.data_ptr()) for t in (xd, wd, scratch, y)), *shape, form, c_void_p(torch.cuda.current_stream().cuda_stream)))
            bound = (9 * 2.0 ** -24 if kind == 7 else 2.0 ** -23 * 9 * C + slices * 2.0 ** -24) * size
            assert bool(((y.cpu().double() - want).abs() <= bound + 1e-30).all()), (kind, slices)


@pytest.mark.parametrize('dtype', ['float16', 'float32'])
@pytest.mark.parametrize('case', [
    (2, 16, (9, 9), 33, (1, 1), (9, 9)),             # a block spans several images, one more feature than two tiles
    (3, 8, (13, 17), 16, (1, 1), (13, 17)),          # one unit of channels (float16: half of one)
    (1, 72, (40, 3), 130, (1, 1), (40, 3)),          # rows of three points
    (5, 24, (8, 8), 48, (0, 0), (6, 6)),             # no padding
    (2, 24, (12, 10), 40, (2, 0), (14, 7)),          # padded on one axis by two, results short of the other's end
    (1, 16, (1, 1), 32, (1, 1), (1, 1)),             # one point
    (4, 8, (30, 31), 20, (-1, 1), (27, 31)),         # taps that start inside, blocks that stay inside an image
    (3, 264, (6, 30), 15, (1, 1), (6, 30)),          # wavefronts in several rounds, four points per lane
    (1, 408, (24, 40), 17, (1, 1), (24, 40)),        # ... and more of them than the registers allow at once
])
@pytest.mark.parametrize('offset', [0, 1])           # values by which the filter misses a 16-byte boundary
def test_one_launch_convolutions_match_float64(autort, dtype, case, offset):
    """Sums in float64 of float32 sums of 8 products three times over (float16: of 48 products): a chain of 6 (48) roundings of 2^-24 and
    the one of the result."""
    from ctypes import c_void_p
    from antares_amd.runtime import capi
    N, C, (H, W), F, (ph, pw), (HO, WO) = case
    note(f'one-launch convolution {dtype} {case} offset {offset}')
    g = torch.Generator().manual_seed(N * 1000 + C + W)
    x, w = torch.randn(N, C, H, W, generator=g).to(getattr(torch, dtype)), torch.randn(F, C, 3, 3, generator=g).to(getattr(torch, dtype))
    f16 = int(dtype == 'float16')
    shape = (f16, N, C, H, W, F, HO, WO, ph, pw)
    lib, dev = capi.lib(), autort.device()
    xd, memory = x.to(dev), torch.empty(w.numel() + 1, dtype=w.dtype, device=dev)
    wd = memory[offset:offset + w.numel()].view(w.shape).copy_(w)
    pad = max(ph, pw, 0) + 2

    def reference(a, b):
        return torch.nn.functional.conv2d(torch.nn.functional.pad(a, (pad, pad + 2, pad, pad + 2)), b)[:, :, pad - ph:pad - ph + HO, pad - pw:pad - pw + WO]
    want, size = reference(x.double(), w.double()), reference(x.double().abs(), w.double().abs())
    for form in (8, 9, 10):
        assert lib.art_conv2d_form(*shape, form) == form and lib.art_conv2d_scratch_bytes(*shape, form) == 0
        y = torch.full((N, F, HO, WO), 7.0, device=dev)
        capi.check(lib.art_conv2d(c_void_p(xd.data_ptr()), c_void_p(wd.data_ptr()), None, c_void_p(y.data_ptr()), *shape, form,
                                  c_void_p(torch.cuda.current_stream().cuda_stream)))
        assert bool(((y.cpu().double() - want).abs() <= (49 if f16 else 7) * 2.0 ** -24 * size + 1e-30).all()), form


@pytest.mark.parametrize('dtype,n,c,f,hw', [('float32', 4, 40, 104, 8), ('float32', 1, 24, 24, 39), ('float32', 62, 8, 7, 22), ('float32', 16, 48, 16, 20), ('float16', 1, 104, 176, 9),
                                            ('float16', 3, 56, 232, 7)])
def test_one_launch_convolutions_are_no_further_from_float64_than_those_with_copies(autort, dtype, n, c, f, hw):
    from ctypes import c_void_p
    from antares_amd.runtime import capi
    note(f'one-launch convolution against copies {dtype} {n}x{c}x{hw}x{hw} -> {f}')
    lib, dev, f16 = capi.lib(), autort.device(), int(dtype == 'float16')
    shape = (f16, n, c, hw, hw, f, hw, hw, 1, 1)
    forms = [lib.art_conv2d_direct(*shape), lib.art_conv2d_choose(*shape)]
    assert forms[0] >= 8 and 0 < forms[1] & 255 < 8
    g = torch.Generator().manual_seed(c)
    x, w = torch.randn(n, c, hw, hw, generator=g).to(getattr(torch, dtype)), torch.randn(f, c, 3, 3, generator=g).to(getattr(torch, dtype))
    want = torch.nn.functional.conv2d(x.double(), w.double(), padding=1)
    xd, wd, off = x.to(dev), w.to(dev), []
    for form in forms:
        y, scratch = torch.empty(n, f, hw, hw, device=dev), torch.empty(lib.art_conv2d_scratch_bytes(*shape, form) + 16, dtype=torch.uint8, device=dev)
        capi.check(lib.art_conv2d(*(c_void_p(t.data_ptr()) for t in (xd, wd, scratch, y)), *shape, form, c_void_p(torch.cuda.current_stream().cuda_stream)))
        off.append(float((y.cpu().double() - want).norm() / want.norm()))
    assert off[0] <= 1.02 * off[1], off          # (2 %: what single inputs scatter)


@pytest.mark.parametrize('dtype,n,c,f,hw', [('float16', 1, 216, 48, 35), ('float32', 2, 72, 56, 20), ('float32', 9, 216, 64, 17), ('float32', 12, 24, 24, 46),
                                            ('float16', 6, 88, 40, 8), ('float16', 4, 48, 16, 20)])
def test_staged_convolutions_are_no_further_from_float64_than_the_generic_kernels(autort, dtype, n, c, f, hw):
    from antares_amd.runtime import capi
    note(f'staged convolution operator {dtype} {n}x{c}x{hw}x{hw} -> {f}')
    dev, dt = autort.device(), getattr(torch, dtype)
    assert capi.lib().art_conv2d_choose(int(dtype == 'float16'), n, c, hw, hw, f, hw, hw, 1, 1) & 255 > 3
    x, w = torch.randn(n, c, hw, hw, device=dev).to(dt), torch.randn(f, c, 3, 3, device=dev).to(dt)
    want = torch.nn.functional.conv2d(x.cpu().double(), w.cpu().double(), padding=1)
    off = []
    for generic in (False, True):
        op = autort.export(ir=conv_program(dtype, (hw, hw), (hw, hw), (1, 1)),
                           inputs=[f'input0={dtype}[N:{n}, C:{c}, H:{hw}, W:{hw}]', f'input1={dtype}[F:{f}, C:{c}, KH:3, KW:3]'], name=f'conv_st_{dtype}_{n}_{c}_{int(generic)}')
        if generic:
            op.fast_path = None
        off.append(float((op(x, w).cpu().double() - want).norm() / want.norm()))
    assert off[0] <= 1.05 * off[1], off


@pytest.mark.parametrize('dtype,n,c,f,h,w', [('float32', 3, 17, 8, 3000, 160), ('float16', 5, 40, 33, 2100, 150)])      # two (three) images to a pass, one (two) left
def test_staged_convolutions_of_large_batches_in_passes(autort, dtype, n, c, f, h, w):
    """A copy of 128 MiB at the most: the images go in passes.  The bounds are those of one pass."""
    from ctypes import c_void_p
    from antares_amd.runtime import capi
    note(f'staged convolution in passes {dtype} {n}x{c}x{h}x{w} -> {f}')
    g = torch.Generator().manual_seed(h)
    x, wt = torch.randn(n, c, h, w, generator=g).to(getattr(torch, dtype)), torch.randn(f, c, 3, 3, generator=g).to(getattr(torch, dtype))
    f16 = int(dtype == 'float16')
    shape = (f16, n, c, h, w, f, h, w, 1, 1)
    lib, dev = capi.lib(), autort.device()
    xd, wd = x.to(dev), wt.to(dev)
    # rows at both ends of every image and in its middle
    rows = [0, 1, h // 2, h // 2 + 1, h - 2, h - 1]
    pads = torch.nn.functional.pad(x.double(), (1, 1, 1, 1))
    want, size = (torch.cat([torch.nn.functional.conv2d(a[:, :, r:r + 3], b) for r in rows], 2) for a, b in ((pads, wt.double()), (pads.abs(), wt.double().abs())))
    for form in (4, 5, 4 + 512) if f16 else (4, 5, 7, 4 + 512):
        y = torch.full((n, f, h, w), 7.0, device=dev)
        scratch = torch.full((lib.art_conv2d_scratch_bytes(*shape, form),), 255, dtype=torch.uint8, device=dev)
        assert 0 < scratch.numel() < (130 << 20) + (2 * 3 * f * h * w * 4 if form > 255 else 0)
        capi.check(lib.art_conv2d(*(c_void_p(t.data_ptr()) for t in (xd, wd, scratch, y)), *shape, form, c_void_p(torch.cuda.current_stream().cuda_stream)))
        assert bool(((y[:, :, rows].cpu().double() - want).abs() <= 2.0 ** -23 * 9 * c * size + 1e-30).all()), form


@pytest.mark.parametrize('dtype,n,c,f,hw', [('float16', 9, 9, 200, 49), ('float16', 16, 25, 25, 40), ('float16', 4, 33, 17, 56), ('float16', 17, 25, 88, 29), ('float16', 4, 4, 96, 40), ('float32', 5, 24, 2424, 2),
                                            ('float32', 1, 208, 1160, 4), ('float32', 8, 3, 64, 40)])
def test_convolutions_of_few_channels_or_points_are_no_further_from_float64_than_the_generic_kernels(autort, dtype, n, c, f, hw):
    """Whichever kernel takes them: the generic sums are short here, on the vector units or over less than a chunk of channels."""
    note(f'convolution of few channels or points {dtype} {n}x{c}x{hw}x{hw} -> {f}')
    dev, dt = autort.device(), getattr(torch, dtype)
    g = torch.Generator().manual_seed(n * c + f)
    x, w = torch.randn(n, c, hw, hw, generator=g).to(dt), torch.randn(f, c, 3, 3, generator=g).to(dt)
    want = torch.nn.functional.conv2d(x.double(), w.double(), padding=1)
    off = []
    for generic in (False, True):
        op = autort.export(ir=conv_program(dtype, (hw, hw), (hw, hw), (1, 1)),
                           inputs=[f'input0={dtype}[N:{n}, C:{c}, H:{hw}, W:{hw}]', f'input1={dtype}[F:{f}, C:{c}, KH:3, KW:3]'], name=f'conv_few_{dtype}_{n}_{c}_{int(generic)}')
        if generic:
            op.fast_path = None
        off.append(float((op(x.to(dev), w.to(dev)).cpu().double() - want).norm() / want.norm()))
    assert off[0] <= 1.02 * off[1], off


@pytest.mark.parametrize('dtype,n,c,f,hw', [('float16', 4, 40, 72, 20), ('float16', 2, 64, 24, 23), ('float32', 5, 20, 72, 21), ('float16', 30, 16, 256, 28)])
def test_convolution_operator_takes_the_kernel_and_agrees_with_the_generic_one(autort, dtype, n, c, f, hw):
    note(f'convolution operator {dtype} {n}x{c}x{hw}x{hw} -> {f}')
    dev = autort.device()
    dt = getattr(torch, dtype)
    op = autort.export(ir=conv_program(dtype, (hw, hw), (hw, hw), (1, 1)),
                       inputs=[f'input0={dtype}[N:{n}, C:{c}, H:{hw}, W:{hw}]', f'input1={dtype}[F:{f}, C:{c}, KH:3, KW:3]'], name=f'conv_hand_{dtype}_{n}_{c}')
    x, w = torch.randn(n, c, hw, hw, device=dev).to(dt), torch.randn(f, c, 3, 3, device=dev).to(dt)
    x[0, 0, 0, 0], x[0, 0, hw - 1, hw - 1] = float('inf'), float('nan')
    taken = []
    handler = op.fast_path
    op.fast_path = lambda *a: taken.append(handler(*a)) or taken[-1]
    got, again = op(x, w), op(x, w)
    assert taken and all(taken) and torch.equal(got.isnan(), again.isnan()) and torch.equal(got.nan_to_num(), again.nan_to_num())
    op = autort.export(ir=op.ir, inputs=op.input_specs, name=f'conv_generic_{dtype}_{n}_{c}')
    op.fast_path = None
    want = op(x, w)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    fin = want.isfinite()
    assert ((got - want)[fin].norm() / want[fin].norm()).item() < 2.0 ** -23 * 9 * c       # float32 sums of 9 c terms, another order


# one, two and four chunks of 8 per thread, at the ends of each, and a length that is not whole chunks
@pytest.mark.parametrize('dtype', ['float16', 'float32'])
@pytest.mark.parametrize('n', [8, 2048, 2056, 4096, 4104, 8192, 1001])
def test_rmsnorm_rows_of_every_length(autort, dtype, n):
    """art_rmsnorm against float64: a float32 sum of n squares in some order (n 2^-24 of it at most, half of that in the root), three
    roundings to float32 and one to the result's type; nothing behind the rows is written."""
    from ctypes import c_void_p
    from antares_amd.runtime import capi
    dev, t = autort.device(), getattr(torch, dtype)
    capi.init(0)
    g = torch.Generator().manual_seed(n)
    x, w = torch.randn(3, n, generator=g).to(t), torch.randn(n, generator=g).to(t)
    xd, wd, out = x.to(dev), w.to(dev), torch.full((4, n), 7.0, dtype=t, device=dev)
    kind = int(dtype == 'float16')
    note(f'rmsnorm {dtype} 3 rows of {n}')
    capi.check(capi.lib().art_rmsnorm(c_void_p(xd.data_ptr()), None, c_void_p(wd.data_ptr()), c_void_p(out.data_ptr()), 3, n, 1.0 / n, 1e-5, kind, kind, kind,
                                      c_void_p(torch.cuda.current_stream().cuda_stream)))
    y = x.double()
    exact = y / torch.sqrt((y * y).mean(1, keepdim=True) + 1e-5) * w.double()
    got = out.cpu().double()
    assert ((got[:3] - exact).abs() <= exact.abs() * ((n / 2 + 8) * 2.0 ** -24 + (2.0 ** -11 if kind else 0)) + 2.0 ** -24).all()
    assert (got[3] == 7.0).all()


# with and without K-splits, one and two turns of a block, a row that is not whole 16-byte pieces of 8 (two launches)
@pytest.mark.parametrize('M,K,N', [(1, 256, 16), (5, 512, 272), (33, 1024, 4096), (130, 640, 8192), (20, 512, 8208), (300, 256, 144)])
def test_w4a16_gemm_with_residual_and_rmsnorm_behind_it(autort, M, K, N):
    """gemm_w4a16_residual_norm gives gemm_w4a16_residual's result bit for bit, and its RMSNorm: the square root's argument is
    a float32 sum in another order (N 2^-24 at most), the result is rounded to float16 (2^-11)."""
    from ctypes import c_void_p
    from antares_amd.runtime import capi
    dev = autort.device()
    capi.init(0)
    p = workloads.w4_problem(K + N + M, M, K, N)
    d = [p[k].to(dev) for k in ('x', 'qweight', 'scales', 'qzeros')]
    g = torch.Generator().manual_seed(M)
    res, weight = torch.randn(M, N, generator=g).half().to(dev), (torch.randn(N, generator=g) * 0.1 + 1).half().to(dev)
    stream = c_void_p(torch.cuda.current_stream().cuda_stream)
    for code in (0, 256 + 1, 256 + 2, 512 + 3, 1024 + 2, 2048 + 1):
        for residual in (None, res):
            note(f'w4a16 gemm + residual + norm M={M} K={K} N={N} code {code} {"with" if residual is not None else "no"} residual')
            want, got, norm = (torch.full((M, N), float('nan'), dtype=torch.float16, device=dev) for _ in range(3))
            ptr = [c_void_p(t.data_ptr()) for t in d]
            r = c_void_p(residual.data_ptr() if residual is not None else 0)
            capi.check(capi.lib().art_gemm_w4a16_residual(*ptr, c_void_p(want.data_ptr()), r, M, K, N, code, stream))
            capi.check(capi.lib().art_gemm_w4a16_residual_norm(*ptr, c_void_p(got.data_ptr()), r, c_void_p(weight.data_ptr()), c_void_p(norm.data_ptr()),
                                                               M, K, N, 1e-5, code, stream))
            assert torch.equal(got, want)
            y = want.cpu().double()
            exact = y / torch.sqrt((y * y).mean(1, keepdim=True) + 1e-5) * weight.cpu().double()
            assert ((norm.cpu().double() - exact).abs() <= exact.abs() * (2.0 ** -11 + N * 2.0 ** -24) + 2.0 ** -24).all()
    acc = res.clone()
    out = autort.ops.gemm_w4a16_residual_norm(*d, acc, weight, residual=acc)
    plain = res.clone()
    autort.ops.gemm_w4a16_residual(*d, plain, residual=plain)
    assert torch.equal(acc, plain) and torch.equal(out, autort.ops.gemm_w4a16_residual_norm(*d, res.clone(), weight, residual=res))
    assert capi.lib().art_gemm_w4a16_residual_norm(*ptr, c_void_p(acc.data_ptr()), None, c_void_p(weight.data_ptr()), c_void_p(acc.data_ptr()),
                                                   M, K, N, 1e-5, 0, stream) != 0


@pytest.mark.parametrize('dtype', ['float16', 'float32'])
def test_convolution_into_part_of_a_larger_result(autort, dtype):
    """A declared result that is larger than what the program computes: only its part is written, in its place."""
    note(f'convolution {dtype} into part of a larger result')
    dev = autort.device()
    n, c, f, hw = 4, 64, 64, 28
    op = autort.export(ir=conv_program(dtype, (hw, hw), (hw, hw), (1, 1)), name=f'conv_part_{dtype}',
                       inputs=[f'input0={dtype}[N:{n}, C:{c}, H:{hw}, W:{hw}]', f'input1={dtype}[F:{f}, C:{c}, KH:3, KW:3]', 'output0=float32[N, F, A:32, B:30]'])
    g = torch.Generator().manual_seed(hw)
    x, w = torch.randn(n, c, hw, hw, generator=g).to(getattr(torch, dtype)), torch.randn(f, c, 3, 3, generator=g).to(getattr(torch, dtype))
    want, bound = (torch.nn.functional.conv2d(a, b, padding=1) for a, b in ((x.double(), w.double()), (x.double().abs(), w.double().abs())))
    for size in ((32, 30), (28, 28), (28, 30)):
        for _ in range(2):
            y = torch.full((n, f) + size, 7.0, device=dev)
            op(x.to(dev), w.to(dev), y)
            got = y.cpu().double()
            assert ((got[:, :, :hw, :hw] - want).abs() <= 2.0 ** -23 * 9 * c * bound).all()
            assert (got[:, :, hw:] == 7.0).all() and (got[:, :, :, hw:] == 7.0).all()


# more rows than one launch of any form takes (and one row more); 32-row blocks asked for; more columns than the narrow forms
# number, also where one of them is asked for, and a K-split that does not fit
@pytest.mark.parametrize('M,K,N,code', [(262145, 128, 16, 0), (1048576 + 40, 128, 16, 0), (262144 + 33, 256, 48, 256 + 1), (524288 + 1, 128, 32, 2048 + 1),
                                        (5, 128, 16384 * 513, 0), (40, 256, 16384 * 513, 512 + 2), (5, 256, 16384 * 300, 256 + 2)])
def test_w4a16_gemm_of_very_many_rows_or_columns(autort, M, K, N, code):
    """Rows and columns repeat with a period: the result is that of one period, the oracle's."""
    from ctypes import c_void_p
    from antares_amd.runtime import capi
    from oracle import hot_ops
    note(f'w4a16 gemm M={M} K={K} N={N} code={code}')
    dev = autort.device()
    capi.init(0)
    m, n, step = min(M, 999), min(N, 16384), 1 << 17
    p = workloads.w4_problem(M % 1000, m, K, n)
    x, q, s, z = (p[k] for k in ('x', 'qweight', 'scales', 'qzeros'))
    want = torch.from_numpy(hot_ops.gemm_w4a16(x.numpy(), q.numpy(), s.numpy(), z.numpy())).to(dev).float()
    rows = torch.arange(M, device=dev) % m
    operands = [x.to(dev)[rows]] + [t.to(dev).repeat(1, N // n) for t in (q, s, z)]
    lib, stream = capi.lib(), c_void_p(torch.cuda.current_stream().cuda_stream)

    def new(columns):
        return torch.full((M, columns), float('nan'), dtype=torch.float16, device=dev)

    def ptr(*tensors):
        return [c_void_p(t.data_ptr()) for t in tensors]

    def close(got, period, **tol):
        for r in range(0, M, step):
            part = got[r:r + step].float().view(-1, N // n, period.shape[1])
            assert torch.allclose(part, period[rows[r:r + step]].view(-1, 1, period.shape[1]).expand_as(part), **tol)
    y = new(N)
    capi.check(lib.art_gemm_w4a16_tuned(*ptr(*operands, y), M, K, N, code, stream))
    close(y, want, rtol=1e-2, atol=1e-2)
    if n < N:
        return
    if N % 32 == 0:
        hid = new(N // 2)
        capi.check(lib.art_gemm_w4a16_swiglu(*ptr(*operands, hid), M, K, N, code, stream))
        close(hid, torch.nn.functional.silu(want[:, :N // 2]) * want[:, N // 2:], rtol=2e-2, atol=2e-2)
    res, weight = torch.randn(m, N, device=dev).half()[rows], torch.rand(N, device=dev).half()
    acc, out = res.clone(), new(N)                           # the residual and the normalised rows move on with the rows
    capi.check(lib.art_gemm_w4a16_residual_norm(*ptr(*operands, acc, acc, weight, out), M, K, N, 1e-5, code, stream))
    assert torch.equal(acc, (y.float() + res.float()).half()) and torch.equal(out, autort.ops.rmsnorm_f16(acc, None, weight))
