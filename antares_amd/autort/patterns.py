"""Recognition of operator patterns that have a hand-written gfx950 kernel.

A program is recognised by the canonical text of its fused statements (tensor
and axis names replaced by order of appearance), so the user's spelling of
names does not matter.  The part each of the caller's tensors plays is taken
from that same order: ``match`` returns the handler together with a map from
the registered program's tensor names (the handler's vocabulary: ``x``,
``qweight`` ...) to the caller's names.  A handler returns True when it ran the
operator, or False to leave it to the generic lowering (shapes it does not
cover).
"""
from __future__ import annotations

from typing import Callable, Dict, Optional, Tuple

from ctypes import c_void_p

import torch

from ..ir import Graph, fuse_elementwise, parse_program
from ..runtime import capi
from ..runtime.calls import STREAM

_TABLE: Dict[str, Tuple[Callable, list]] = {}      # canonical key -> (handler, the registered program's tensor order)


def register(ir: str, inputs, handler: Callable):
    g = fuse_elementwise(parse_program(ir, inputs))
    key = g.canonical_key()
    _TABLE[key] = (handler, g.canonical_tensor_order())
    return key


def match(fused: Graph) -> Optional[Tuple[Callable, Dict[str, str]]]:
    """(handler, roles) for a recognised program, else None.  ``roles`` maps the registered program's tensor names
    to the names the caller's program uses for the tensors in the same places."""
    conv = _conv2d(fused)
    if conv is not None:
        return _conv2d_handler(fused.statements[0], *conv[3:]), dict(zip('xwy', conv[:3]))
    hit = _TABLE.get(fused.canonical_key())
    if hit is None or not _axes_span_their_dimensions(fused):
        return None
    handler, registered = hit
    return handler, dict(zip(registered, fused.canonical_tensor_order()))


def _axes_span_their_dimensions(fused: Graph) -> bool:
    """The canonical key drops extents, and the handlers take every size from the operands' shapes: a program that
    restricts an axis (`... where K in 100`, `... where M in 100`) spells the same statements but computes something
    else - a shorter sum, a smaller output.  Such a program is left to the generic lowering: a hand kernel is taken
    only when every axis that indexes a tensor dimension directly runs over exactly that dimension."""
    from ..ir.nodes import walk
    for st in fused.statements:
        extent = dict(st.data_axes + st.reduce_axes)
        uses = [(st.output, st.out_index)]
        uses += [(n.name, n.args) for n in walk(st.root) if n.kind == 'load']
        for name, index in uses:
            info = fused.tensors.get(name)
            if info is None:
                continue
            shape = list(info.shape)
            if len(index) != len(shape):
                continue                          # scalars (`[]` against `[1]`) carry no axis
            for ix, dim in zip(index, shape):
                if ix.kind == 'axis' and ix.name in extent and extent[ix.name] != dim:
                    return False
    return True


# ---------------------------------------------------------------------------
# int4 GEMV in the reference's weight format (samples/05_llama2_7b_int4.py:135-139)
# ---------------------------------------------------------------------------
GPTQ_GEMV_IR = """
  input1[S, N] = (qweight[S / 8, N] >> (S % 8 * 4)).call(strs.bitwise_and, 15) * input0[S].like(1)
  w[S, N] = scales[S / 128, N] * (input1[S, N] - 8)
  my_result[N] +=! input0[S] * w[S, N].to(input0.dtype())
"""


def _gptq_inputs(xdt: str, sdt: str):
    return [f'input0={xdt}[S:4096]', 'qweight=int32[L:512, N:12288]', f'scales={sdt}[K:32, N:12288]']


def _gptq_handler(op, bound, env, call) -> bool:
    r = op.fast_roles
    x, q, s, out = bound[r['input0']], bound[r['qweight']], bound[r['scales']], bound[r['my_result']]
    x_f16, s_f16 = int(x.dtype == torch.float16), int(s.dtype == torch.float16)
    K, N = x.shape[0], q.shape[1]
    if K % 128 or N % 4 or q.shape[0] * 8 != K or s.shape[0] * 128 != K or q.data_ptr() % 16:
        return False
    call.library(capi.lib().art_gemv_gptq, x, q, s, out, K, N, x_f16, s_f16, STREAM)
    return True


for _x in ('float32', 'float16'):
    for _s in ('float32', 'float16'):
        register(GPTQ_GEMV_IR, _gptq_inputs(_x, _s), _gptq_handler)


# ---------------------------------------------------------------------------
# int4 g128 GEMV / skinny GEMM with per-group zero points:
#   y[m,n] = sum_k x[m,k] * fp16( s[k/128,n] * (q[k,n] - z[k/128,n]) )     fp32 accumulate, fp16 out
# qweight uint8 [K/2,N] (low nibble = even k), qzeros uint8 [K/128,N/2] (low nibble = even n).
# ---------------------------------------------------------------------------
W4A16_IR = """
  acc[M, N] +=! x[M, K].to(`float32`) * (scales[K / 128, N] * (((qweight[K / 2, N] >> (K % 2 * 4)).call(strs.bitwise_and, 15) - (qzeros[K / 128, N / 2] >> (N % 2 * 4)).call(strs.bitwise_and, 15)) * scales[K / 128, N].like(1))).to(`float32`)
  y[M, N] = acc[M, N].to(`float16`)
"""
W4A16_INPUTS = ['x=float16[M:1, K:4096]', 'qweight=int8[KH:2048, N:11008]', 'scales=float16[G:32, N:11008]',
                'qzeros=int8[G:32, NH:5504]']


def scratch_memory(count: int, dtype, device):
    """Memory that a kernel works in, None when there is not that much: the handler then takes a form that needs less, or leaves the
    call to the generic kernels."""
    try:
        return torch.empty(count, dtype=dtype, device=device)
    except torch.OutOfMemoryError:
        return None


def tune_hand_kernel(op, key: str, candidates, run, trials: int, clones):
    """``config="tune:N"`` for a hand-written kernel: times up to N values of its launch parameter for the shape of
    this call (the reference's tuner walks the knob space of the schedule that runs, tuner/OpEvo/main.py:467-616; a
    hand kernel has one knob with a handful of values, so the walk is exhaustive up to N).  ``run(value, tensors)``
    enqueues one launch; ``clones`` yields sets of operand tensors - the timing rotates over several copies, since
    one buffer launched over and over would be served by the memory-side cache and favour the wrong choice - whose
    outputs are scratch, never the caller's.  The winner is kept in ``op.tuned[key]`` and in the module file."""
    sets = list(clones)
    stream = torch.cuda.current_stream().cuda_stream
    best = None
    for value in candidates[:max(1, trials)]:
        run(value, sets[0])                                   # warm-up (and the first use of a code path)
        start, stop = capi.Event(), capi.Event()
        start.record(stream)
        runs = max(6, 2 * len(sets))
        for i in range(runs):
            run(value, sets[i % len(sets)])
        stop.record(stream)
        us = start.elapsed_ms(stop) * 1e3 / runs
        if best is None or us < best['us']:
            best = {'value': int(value), 'us': round(us, 3)}
    op.tuned[key] = best
    op.persist()
    return best


def _w4a16_handler(op, bound, env, call) -> bool:
    r = op.fast_roles
    x, q, s, z, y = bound[r['x']], bound[r['qweight']], bound[r['scales']], bound[r['qzeros']], bound[r['y']]
    M, K = x.shape
    N = q.shape[1]
    if K % 128 or N % 16 or q.shape[0] * 2 != K or s.shape[0] * 128 != K or z.shape[1] * 2 != N \
            or q.data_ptr() % 16 or x.data_ptr() % 16 or z.data_ptr() % 8 or y.data_ptr() % 8:
        return False
    # the vector-unit kernel streams the weights once per four rows (7.5 / 11.1 / 13.0 / 15.3 us for 1..4 rows of
    # 4096 x 11008, 22 us for five), the matrix-core kernel once per 64 rows (16 us for 4..32 rows): four rows and
    # more go there
    lib = capi.lib()
    gemv = M <= 3

    # the entry point and its launch parameters (GEMV: 16 * rows per lane + wavefronts per block, 0: the library's choice)
    entry = lib.art_gemv_w4a16_knobs if gemv else lib.art_gemm_w4a16_tuned

    def knobs(value):
        return (int(value) >> 4, int(value) & 15) if gemv else (int(value),)

    def run(value, t):
        capi.check(entry(*(c_void_p(v.data_ptr()) for v in t), M, K, N, *knobs(value), c_void_p(torch.cuda.current_stream().cuda_stream)))

    # the launch parameters of the kernel that runs: (rows per lane, wavefronts per block) of the GEMV - two factors
    # searched as a product space, as the reference's tuner walks the factor spaces of a schedule's knobs
    # (tuner/OpEvo/main.py:154-293) -, (K-splits, rows per block) of the GEMM
    key = f"{'gemv_w4a16.rows_x16_plus_waves' if gemv else 'gemm_w4a16.k_splits'}|{M},{K},{N}"
    saved = op.tuned.get(key)
    trials = op.config.get('tune')
    if saved is None and isinstance(trials, int) and trials > 0 and not torch.cuda.is_current_stream_capturing():
        per_set = q.numel() + 2 * s.numel() + z.numel()
        copies = max(1, min(8, (256 << 20) // max(per_set, 1)))
        clones = [(x, q.clone(), s.clone(), z.clone(), torch.empty_like(y)) for _ in range(copies)]
        if gemv:
            cands = [16 * rows + waves for rows in (8, 4) for waves in ((4, 8) if M == 1 else (4,))]
        else:
            counts = [v for v in (1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 20, 24, 32) if v <= K // 128]
            # 512 + v: v K-splits over blocks of 64 rows; 256 + v: over blocks of 32 rows (twice the blocks);
            # 1280 + v: over blocks of 128 rows; 1024 + v, 2048 + v: of 128 and 256 rows and twice the columns
            cands = [0] + [512 + v for v in counts] + ([256 + v for v in counts] if M > 32 else [])
            cands += [rows + v for rows in (1280, 1024, 2048) for v in counts if v <= 16] if M > 64 else []
            # 2304, 2560 + v: blocks of 32 rows whose wavefronts divide K, over 32 and 64 columns; 2816 + v: of 64 rows over 32 columns
            cands += [form + v for form, rows in ((2304, 256), (2560, 256), (2816, 512)) for v in counts if v <= 16 and M <= rows]
        saved = tune_hand_kernel(op, key, cands, run, trials, clones)
        del clones
    call.library(entry, x, q, s, z, y, M, K, N, *knobs(saved['value'] if saved is not None else 0), STREAM)
    return True


register(W4A16_IR, W4A16_INPUTS, _w4a16_handler)


# ---------------------------------------------------------------------------
# Products of small and odd sizes (art_gemm_tile): float16 and float32 below, int8 A[M,K] @ B[N,K]^T
# ---------------------------------------------------------------------------
_TILE_SLICES = (1, 2, 3, 4, 6, 8, 12, 16, 24)
_TILE_SLICES_ROOM = 1 << 25                  # values that the slices of a product take at the most (the library's own bound)


def _tile_product(op, call, kind: int, a, b, c, M: int, N: int, K: int, large: bool, rival=None) -> bool:
    """Runs the product with ``art_gemm_tile`` if that is the faster kernel for these sizes.  ``rival``: what a tuning run keeps
    of the kernel for large products; the faster of the two runs, and one that was kept alone stays."""
    lib = capi.lib()
    if max(M, N, K) >= 1 << 31 or any(t.data_ptr() < c.data_ptr() + c.element_size() * c.numel() and c.data_ptr() < t.data_ptr() + t.element_size() * t.numel()
                                      for t in (a, b)):
        return False                              # a result over an operand: left to the kernels that always took it
    code = lib.art_gemm_tile_form(kind, M, N, K, int(large), 0, 0)
    key = f'gemm_tile.form|{kind},{M},{K},{N}'
    saved = op.tuned.get(key)
    trials = op.config.get('tune')
    if saved is None and rival is not None and not (isinstance(trials, int) and trials > 0):
        return False
    if not code and saved is None:
        return False

    def partial(value):
        return scratch_memory((value & 255) * M * N, torch.int32 if kind == 2 else torch.float32, a.device) if value & 255 > 1 else None

    if saved is None and isinstance(trials, int) and trials > 0 and not torch.cuda.is_current_stream_capturing():
        codes = [code] + [v for v in (lib.art_gemm_tile_form(kind, M, N, K, 0, form, s) for form in (1, 2, 3, 4) for s in _TILE_SLICES)
                          if v and v != code and (v >> 8 == 4) == (code >> 8 == 4) and ((v & 255) == 1 or (v & 255) * M * N <= _TILE_SLICES_ROOM)]
        codes = codes[:trials]
        scratch = partial(max(codes, key=lambda v: v & 255))
        if scratch is None:
            codes = [v for v in codes if v & 255 == 1] or [code >> 8 << 8 | 1]

        def run(value, t):
            capi.check(lib.art_gemm_tile(c_void_p(t[0].data_ptr()), c_void_p(t[1].data_ptr()), c_void_p(t[2].data_ptr()),
                                         c_void_p(scratch.data_ptr() if scratch is not None else 0), kind, M, N, K, value >> 8, value & 255,
                                         c_void_p(torch.cuda.current_stream().cuda_stream)))
        saved = tune_hand_kernel(op, key, codes, run, len(codes), [(a, b, torch.empty_like(c))])
    if saved is not None:
        if rival is not None and rival['us'] <= saved['us']:
            return False
        value = int(saved['value'])
        # kept by another version of the library, it may have longer sums than are taken now
        short_sums = lib.art_gemm_tile_form(kind, M, N, K, int(large), 0, 1) >> 8 == 4
        if lib.art_gemm_tile_form(kind, M, N, K, int(large), value >> 8, value & 255) == value and value >> 8 and (value >> 8 == 4) == short_sums \
                and (value & 255 == 1 or (value & 255) * M * N <= _TILE_SLICES_ROOM):
            code = value
    if not code:
        return False
    room = partial(code)
    if room is None and code & 255 > 1:
        code, call.replay = code >> 8 << 8 | 1, False
    call.library(lib.art_gemm_tile, a, b, c, room, kind, M, N, K, code >> 8, code & 255, STREAM)
    return True


def _gemm_i8_handler(op, bound, env, call) -> bool:
    a, b, c = (bound[op.fast_roles[n]] for n in 'abc')
    return _tile_product(op, call, 2, a, b, c, a.shape[0], b.shape[0], a.shape[1], False)


register('c[M, N] +=! a[M, K].cast(`int32`) * b[N, K].cast(`int32`)', ['a=int8[M:4096, K:4096]', 'b=int8[N:4096, K:4096]'], _gemm_i8_handler)


# ---------------------------------------------------------------------------
# fp16 GEMM with fp32 accumulation: C[M,N] = A[M,K] @ B[K,N] (AntaresIR.md:115 with the casts that
# make the accumulator fp32)
# ---------------------------------------------------------------------------
GEMM_F16_IR = """
  acc[M, N] +=! a[M, K].to(`float32`) * b[K, N].to(`float32`)
  c[M, N] = acc[M, N].to(`float16`)
"""
GEMM_F16_INPUTS = ['a=float16[M:4096, K:4096]', 'b=float16[K:4096, N:4096]']


def _gemm_f16_handler(op, bound, env, call) -> bool:
    r = op.fast_roles
    a, b, c = bound[r['a']], bound[r['b']], bound[r['c']]
    M, K = a.shape
    N = b.shape[1]
    if N % 8 or K % 64 or a.data_ptr() % 16 or b.data_ptr() % 16 or c.data_ptr() % 16:
        return _tile_product(op, call, 0, a, b, c, M, N, K, False)

    def run(value, t):
        capi.check(capi.lib().art_gemm_f16_tuned(c_void_p(t[0].data_ptr()), c_void_p(t[1].data_ptr()), c_void_p(t[2].data_ptr()), M, N, K,
                                                 int(value), c_void_p(torch.cuda.current_stream().cuda_stream)))
    # the launch parameter: threads per block (2 x 2 wavefronts of 128 x 128 outputs, or 2 x 4 of 128 x 64)
    key = f'gemm_f16.threads|{M},{K},{N}'
    saved = op.tuned.get(key)
    trials = op.config.get('tune')
    if saved is None and isinstance(trials, int) and trials > 0 and not torch.cuda.is_current_stream_capturing():
        saved = tune_hand_kernel(op, key, [256, 512], run, trials,
                                 [(a, b, torch.empty_like(c))])
    if _tile_product(op, call, 0, a, b, c, M, N, K, True, saved):
        return True
    call.library(capi.lib().art_gemm_f16_tuned, a, b, c, M, N, K, int(saved['value'] if saved is not None else 0), STREAM)
    return True


register(GEMM_F16_IR, GEMM_F16_INPUTS, _gemm_f16_handler)


# ---------------------------------------------------------------------------
# fp32 GEMM: C[M,N] = A[M,K] @ B[K,N] (AntaresIR.md:115 as written; the README's `gemm_f32`)
# ---------------------------------------------------------------------------
GEMM_F32_IR = 'c[M, N] +=! a[M, K] * b[K, N]'
GEMM_F32_INPUTS = ['a=float32[M:4096, K:4096]', 'b=float32[K:4096, N:4096]']


def _gemm_f32_handler(op, bound, env, call) -> bool:
    r = op.fast_roles
    a, b, c = bound[r['a']], bound[r['b']], bound[r['c']]
    M, K = a.shape
    N = b.shape[1]
    # a launch of the kernel for large products needs a few hundred tiles to pay
    if N % 4 or K % 32 or N < 4 or M * N < 128 * 128 * 32 or a.data_ptr() % 16 or b.data_ptr() % 16:
        return _tile_product(op, call, 1, a, b, c, M, N, K, False)

    def run(_, t):
        capi.check(capi.lib().art_gemm_f32(c_void_p(t[0].data_ptr()), c_void_p(t[1].data_ptr()), c_void_p(t[2].data_ptr()), M, N, K,
                                          c_void_p(torch.cuda.current_stream().cuda_stream)))
    # the kernel has no launch parameter to search; a tuning run records its time for the shape in the module file
    key = f'gemm_f32|{M},{K},{N}'
    trials = op.config.get('tune')
    if key not in op.tuned and isinstance(trials, int) and trials > 0 and not torch.cuda.is_current_stream_capturing():
        tune_hand_kernel(op, key, [0], run, 1, [(a, b, torch.empty_like(c))])
    if _tile_product(op, call, 1, a, b, c, M, N, K, True, op.tuned.get(key)):
        return True
    call.library(capi.lib().art_gemm_f32, a, b, c, M, N, K, STREAM)
    return True


register(GEMM_F32_IR, GEMM_F32_INPUTS, _gemm_f32_handler)


# ---------------------------------------------------------------------------
# batched fp32 GEMM: C[B,M,N] = A[B,M,K] @ B[B,K,N] (AntaresIR.md:121)
# ---------------------------------------------------------------------------
BATCH_GEMM_F32_IR = 'c[B, M, N] +=! a[B, M, K] * b[B, K, N]'
BATCH_GEMM_F32_INPUTS = ['a=float32[B:3, M:1024, K:512]', 'b=float32[B:3, K:512, N:512]']


def _batch_gemm_f32_handler(op, bound, env, call) -> bool:
    r = op.fast_roles
    a, b, c = bound[r['a']], bound[r['b']], bound[r['c']]
    batch, M, K = a.shape
    N = b.shape[2]
    # as for the single product: the tiled kernel needs a few hundred tiles to pay
    if N % 4 or K % 32 or N < 4 or batch > 65535 or batch * M * N < 128 * 128 * 32 or a.data_ptr() % 16 or b.data_ptr() % 16 \
            or (M * K) % 4 or (K * N) % 4:
        return False
    call.library(capi.lib().art_gemm_f32_batched, a, b, c, batch, M, N, K, STREAM)
    return True


register(BATCH_GEMM_F32_IR, BATCH_GEMM_F32_INPUTS, _batch_gemm_f32_handler)


# ---------------------------------------------------------------------------
# fp32 GEMM with an operand stored the other way round: A as [K, M], B as [N, K] (a linear layer's weight)
# ---------------------------------------------------------------------------
def _gemm_f32_layout_handler(trans_a: bool, trans_b: bool):
    def handler(op, bound, env, call) -> bool:
        r = op.fast_roles
        a, b, c = bound[r['a']], bound[r['b']], bound[r['c']]
        (K, M) = a.shape if trans_a else a.shape[::-1]
        N = b.shape[0] if trans_b else b.shape[1]
        if K % 32 or (not trans_b and N % 4) or (trans_a and M % 4) or M * N < 128 * 128 * 32 or a.data_ptr() % 16 or b.data_ptr() % 16:
            return False
        call.library(capi.lib().art_gemm_f32_ex, a, b, c, 1, M, N, K, int(trans_a), int(trans_b), STREAM)
        return True
    return handler


register('c[M, N] +=! a[K, M] * b[K, N]', ['a=float32[K:512, M:512]', 'b=float32[K:512, N:512]'], _gemm_f32_layout_handler(True, False))
register('c[M, N] +=! a[M, K] * b[N, K]', ['a=float32[M:512, K:512]', 'b=float32[N:512, K:512]'], _gemm_f32_layout_handler(False, True))
register('c[M, N] +=! a[K, M] * b[N, K]', ['a=float32[K:512, M:512]', 'b=float32[N:512, K:512]'], _gemm_f32_layout_handler(True, True))


# ---------------------------------------------------------------------------
# 2-D convolution, stride 1, zeros outside the image (AntaresIR.md:166): y[N, F, HO, WO] +=! x[N, C, HO + KH - ph,
# WO + KW - pw] * w[F, C, KH, KW], both factors float32 or float16 cast to float32.  Padding, extents and guards are part of
# the program's text, so it is recognised by its structure.
# ---------------------------------------------------------------------------
def _shifted_sum(ix):
    """``A + B - 3`` -> ([names of the axes added], constant); None for anything else."""
    if ix.kind == 'axis':
        return [ix.name], 0
    if ix.kind == 'const' and isinstance(ix.value, int):
        return [], ix.value
    if ix.kind == 'op' and ix.name in '+-' and len(ix.args) == 2:
        l, r = _shifted_sum(ix.args[0]), _shifted_sum(ix.args[1])
        if l is not None and r is not None and (ix.name == '+' or not r[0]):
            return sorted(l[0] + r[0]), l[1] + (r[1] if ix.name == '+' else -r[1])
    return None


def _guards(conds):
    """[lowest, past the highest] value that the conditions leave to each index expression, by its axes and constant;
    None when a condition is anything but an expression of that kind compared with an integer."""
    out = {}
    for c in conds:
        if c.kind != 'op' or c.name not in ('<', '<=', '>', '>=') or len(c.args) != 2:
            return None
        l, r = _shifted_sum(c.args[0]), _shifted_sum(c.args[1])
        if l is None or r is None or bool(l[0]) == bool(r[0]):
            return None
        op = c.name
        if r[0]:
            l, r, op = r, l, {'<': '>', '<=': '>=', '>': '<', '>=': '<='}[op]
        lo, hi = out.get((tuple(l[0]), l[1]), (None, None))
        value = r[1] + (op in ('<=', '>'))
        if op in ('<', '<='):
            hi = value if hi is None else min(hi, value)
        else:
            lo = value if lo is None else max(lo, value)
        out[(tuple(l[0]), l[1])] = (lo, hi)
    return out


def _conv2d(fused: Graph):
    """-> (x, w, y, axes by part, {index: (padding, lowest, past the highest)}) of a convolution, else None."""
    if len(fused.statements) != 1:
        return None
    st = fused.statements[0]
    if st.scatter or st.reduce != '+' or st.out_dtype != 'float32' or len(st.data_axes) != 4 or len(st.reduce_axes) != 3:
        return None
    n, f, ho, wo = (a for a, _ in st.data_axes)
    if [i.name if i.kind == 'axis' else None for i in st.out_index] != [n, f, ho, wo]:
        return None
    if st.root.kind != 'op' or st.root.name != '*' or len(st.root.args) != 2:
        return None
    factors = []
    for e in st.root.args:
        conds = []
        while e.kind in ('cast', 'when'):
            if e.kind == 'when':
                if len(e.args) != 2 or e.merge != 'all' or e.args[1].kind != 'const' or e.args[1].value != 0:
                    return None
                conds += list(e.conds)
            elif e.dtype != 'float32':
                return None
            e = e.args[0]
        if e.kind != 'load' or e.dtype not in ('float16', 'float32') or len(e.args) != 4 or e.name == st.output:
            return None
        factors.append((e, conds))
    if factors[0][0].args[0].kind == 'axis' and factors[0][0].args[0].name == f:
        factors.reverse()
    (x, conds), (w, w_conds) = factors
    if x.dtype != w.dtype or w_conds or not all(i.kind == 'axis' for i in w.args):
        return None
    wf, c, kh, kw = (i.name for i in w.args)
    if wf != f or sorted((c, kh, kw)) != sorted(a for a, _ in st.reduce_axes):
        return None
    if [i.name if i.kind == 'axis' else None for i in x.args[:2]] != [n, c]:
        return None
    guards, window = _guards(conds), {}
    if guards is None:
        return None
    for ix, axes, key in ((x.args[2], (ho, kh), 'h'), (x.args[3], (wo, kw), 'w')):
        s = _shifted_sum(ix)
        if s is None or s[0] != sorted(axes):
            return None
        window[key] = (-s[1],) + guards.pop((tuple(s[0]), s[1]), (None, None))
    if guards:                                    # a condition on something else than the two indices
        return None
    return x.name, w.name, st.output, {'n': n, 'f': f, 'c': c, 'kh': kh, 'kw': kw, 'ho': ho, 'wo': wo}, window


def _conv2d_handler(st, axes, window):
    extent = dict(st.data_axes + st.reduce_axes)

    def handler(op, bound, env, call) -> bool:
        x, w, y = (bound[op.fast_roles[r]] for r in 'xwy')
        e = {part: extent[a] if isinstance(extent[a], int) else env[extent[a]] for part, a in axes.items()}
        if x.dim() != 4 or w.dim() != 4 or (x.shape[0], x.shape[1]) != (e['n'], e['c']) or \
                tuple(w.shape) != (e['f'], e['c'], e['kh'], e['kw']) or \
                (e['kh'], e['kw']) != (3, 3) or not x.numel() or not y.numel():
            return False
        if op.fused.shape_of(op.fast_roles['y'], env) != [e[part] for part in ('n', 'f', 'ho', 'wo')]:
            return False                          # the kernel stores a dense result, not a part of a larger one
        # The kernel reads zeros outside the image and the image everywhere else: that has to be what the guards say, and
        # an index without a guard on one side must not reach past it.
        for key, size in (('h', x.shape[2]), ('w', x.shape[3])):
            pad, lo, hi = window[key]
            highest = e[key + 'o'] - 1 + e['k' + key] - 1 - pad
            if (lo != 0 if lo is not None else pad > 0) or (hi != size if hi is not None else highest >= size):
                return False
        size = x.element_size()
        if any(t.data_ptr() < y.data_ptr() + 4 * y.numel() and y.data_ptr() < t.data_ptr() + size * t.numel() for t in (x, w)):
            return False                          # a result over an operand: the generic kernels' order is kept
        lib = capi.lib()
        shape = (int(x.dtype == torch.float16), e['n'], e['c'], x.shape[2], x.shape[3], e['f'], e['ho'], e['wo'],
                 window['h'][0], window['w'][0])
        if max(abs(v) for v in shape) >= 1 << 31:
            return False
        form = lib.art_conv2d_direct(*shape) or lib.art_conv2d_choose(*shape)
        if not form:
            return False

        def scratch(forms):                       # 0: none is needed
            count = max(lib.art_conv2d_scratch_bytes(*shape, v) for v in forms)
            return scratch_memory(count, torch.uint8, x.device) if count else 0

        def run(value, t):
            capi.check(lib.art_conv2d(*(c_void_p(v.data_ptr() if isinstance(v, torch.Tensor) else v) for v in t), *shape, int(value), c_void_p(torch.cuda.current_stream().cuda_stream)))
        # the launch parameter: the shape of a block
        key = 'conv2d.form|' + ','.join(str(v) for v in shape)
        saved = op.tuned.get(key)
        trials = op.config.get('tune')
        if saved is None and isinstance(trials, int) and trials > 0 and not torch.cuda.is_current_stream_capturing():
            others = (1, 2, 3, 4, 5, 6, 8, 9, 10) + tuple(k + 256 * s for k in (4, 5, 6, 7) for s in (2, 3, 4, 6, 8))
            forms = [form] + [v for v in others if v != form and lib.art_conv2d_exact_enough(*shape, v)]
            forms = forms[:trials]
            room = scratch(forms)
            if room is not None:
                saved = tune_hand_kernel(op, key, forms, run, len(forms), [(x, w, room, torch.empty_like(y))])
        if saved is not None and lib.art_conv2d_exact_enough(*shape, int(saved['value'])):
            form = int(saved['value'])
        room = scratch([form])
        if room is None:                          # no copy of the image then: gathered, or left to the generic kernels
            call.replay = False
            form = lib.art_conv2d_form(*shape, 0)
            room = scratch([form]) if form else None
            if room is None:
                return False
        call.library(lib.art_conv2d, x, w, room, y, *shape, form, STREAM)
        return True
    return handler
