"""Performance cases: the work that users of this package have it do, through its public entry points.

``listed()`` names the cases, ``draw(rng)`` makes more of the same ranges; ``prepare`` builds what a program has in hand
before the call, ``run`` makes one pass, ``work`` and ``tolerance`` state what a pass cannot do without and how far
another correct implementation may be from it.  A case is a dict with a ``kind``:

map        an elementwise einstein_v2 program (the README's sigmoid in float32, SiLU(gate) * up in float16)
rows       a row-wise program of the IR document (softmax, layer normalisation)
partition  the even-first partition of samples/01_sort_even_first.py
w4         the packed int4 group-128 product y[M, N] = x[M, K] * W, one row (decode) to many (a batch, a prompt)
decode     steps of the int4 decoder as one recorded graph, a token at a time
prefill    a whole prompt through the same decoder
gemm       matrix products: float16 with float32 sums, float32, int8 with int32 sums
conv       3x3 convolutions with zero padding, float32 or float16 with float32 sums
sample     decoder layers called operator by operator, the way samples/05_llama2_7b_int4.py writes its forward pass
"""
from __future__ import annotations

import functools
import math

import torch

import autort
from antares_amd.autort import patterns
from antares_amd.llama import LlamaConfig, LlamaInt4Decoder
from antares_amd import workloads

HEAD = 128


def listed():
    return [
        # the README's first call at a size where only the call itself counts
        {'name': 'sigmoid_1k', 'kind': 'map', 'program': 'sigmoid', 'n': 1000},
        # the same program at the size it declares
        {'name': 'sigmoid_4m', 'kind': 'map', 'program': 'sigmoid', 'n': 4_096_000},
        # attention weights of a prompt whose length is no multiple of anything
        {'name': 'softmax_ragged', 'kind': 'rows', 'program': 'softmax', 'dtype': 'float32', 'rows': 32 * 1003, 'cols': 1003},
        # the sort sample at the benchmark's size
        {'name': 'partition_16m', 'kind': 'partition', 'n': 16_777_216},
        # one projection of one token: the headline workload, called as an operator
        {'name': 'w4_gemv', 'kind': 'w4', 'm': 1, 'k': 4096, 'n': 11008},
        # a batch of requests, not a round number of them
        {'name': 'w4_batch_50', 'kind': 'w4', 'm': 50, 'k': 11008, 'n': 4096},
        # token generation with the default model: all 32 layers, in the middle of a sequence
        {'name': 'decode', 'kind': 'decode', 'layers': 32, 'heads': 32, 'ffn': 11008, 'vocab': 32000, 'pos': 200, 'steps': 4},
        # the benchmark's prompt, and a long one of odd length
        {'name': 'prefill_128', 'kind': 'prefill', 'layers': 32, 'heads': 32, 'ffn': 11008, 'vocab': 32000, 'tokens': 128},
        {'name': 'prefill_1003', 'kind': 'prefill', 'layers': 32, 'heads': 32, 'ffn': 11008, 'vocab': 32000, 'tokens': 1003},
        # the benchmark's float16 product
        {'name': 'gemm_f16_4096', 'kind': 'gemm', 'dtype': 'float16', 'm': 4096, 'n': 4096, 'k': 4096},
        # a middle layer of a convolutional network in half precision
        {'name': 'conv_f16', 'kind': 'conv', 'dtype': 'float16', 'n': 32, 'c': 128, 'f': 128, 'hw': 28},
        # the llama sample as it is written: float32, one Python call per operator, no graph
        {'name': 'sample_layers', 'kind': 'sample', 'layers': 4, 'heads': 32, 'ffn': 11008, 'pos': 100},
    ]


def _log(rng, lo, hi, step=1):
    """An integer between lo and hi, even over the logarithm, a multiple of step."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(step, int(round(v / step)) * step)


def draw(rng):
    kind = rng.choice(['map', 'rows', 'partition', 'w4', 'w4', 'decode', 'prefill', 'gemm', 'conv', 'sample'])
    if kind == 'map':
        return {'kind': kind, 'program': rng.choice(['sigmoid', 'silu_mul']), 'n': _log(rng, 10, 32_000_000)}
    if kind == 'rows':
        cols = _log(rng, 16, 8192)
        return {'kind': kind, 'program': rng.choice(['softmax', 'layer_norm']), 'dtype': 'float32',
                'rows': _log(rng, 1, max(1, min(65536, (32 << 20) // cols))), 'cols': cols}
    if kind == 'partition':
        return {'kind': kind, 'n': _log(rng, 100, 16_777_216)}
    if kind == 'w4':
        return {'kind': kind, 'm': rng.choice([1, _log(rng, 1, 64), _log(rng, 1, 1024)]), 'k': _log(rng, 512, 11008, 128), 'n': _log(rng, 512, 12288, 16)}
    if kind in ('decode', 'prefill', 'sample'):
        heads = rng.choice([8, 16, 24, 32])
        model = {'kind': kind, 'layers': _log(rng, 1, 4 if kind == 'sample' else 32), 'heads': heads,
                 'ffn': 128 * round(heads * rng.uniform(2.5, 2.7))}
        if kind == 'sample':
            return dict(model, pos=_log(rng, 1, 500))
        if kind == 'prefill':
            return dict(model, vocab=32000, tokens=_log(rng, 8, 1000))
        return dict(model, vocab=32000, pos=_log(rng, 1, 4000), steps=4)
    if kind == 'gemm':
        dtype = rng.choice(['float16', 'float16', 'float32', 'int8'])
        step = rng.choice([1, 8, 64])
        return {'kind': kind, 'dtype': dtype, 'm': _log(rng, 64, 4096, step), 'n': _log(rng, 64, 4096, step), 'k': _log(rng, 64, 4096, step)}
    return {'kind': kind, 'dtype': rng.choice(['float32', 'float16']), 'n': _log(rng, 1, 32), 'c': _log(rng, 16, 256, 8), 'f': _log(rng, 16, 256, 8),
            'hw': _log(rng, 7, 56)}


# -- programs ---------------------------------------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _export(name, ir, inputs):
    """A program exports its operators once."""
    return autort.export(ir=ir, inputs=list(inputs), name='perf_' + name)


def _map_op(program):
    if program == 'sigmoid':
        return _export('sigmoid', 'sigmoid_f32[N] = 1 - 1 / (1 + data[N].call(strs.exp))', ('data=float32[N:4096000]',))
    return _export('silu_mul', 'hidden[N] = (gu[0, N].to(`float32`) / (1.0 + (0.0 - gu[0, N].to(`float32`)).call(strs.exp)) * gu[1, N].to(`float32`)).to(`float16`)',
                   ('gu=float16[2, N]',))


def _rows_op(program, dtype):
    if program == 'softmax':
        ir = ('temp0[N] >=! input0[N, C]; temp1[N] +=! (input0[N, C] - temp0[N]).call(`exp`); '
              'output0[N, C] = (input0[N, C] - temp0[N]).call(`exp`) / temp1[N]')
    else:
        ir = ('temp0[N] +=! input0[N, C]; temp1[N] +=! input0[N, C] * input0[N, C]; '
              'output0[N, C] = (input0[N, C] * C.val() - temp0[N]) * (temp1[N] * C.val() - temp0[N] * temp0[N] + 1e-5).call(`rsqrt`)')
    return _export(f'{program}_{dtype}', ir, (f'input0={dtype}[N:4096, C:1024]',))


def _gemm_op(dtype):
    if dtype == 'float16':
        return _export('gemm_f16', patterns.GEMM_F16_IR, tuple(patterns.GEMM_F16_INPUTS))
    if dtype == 'float32':
        return _export('gemm_f32', patterns.GEMM_F32_IR, tuple(patterns.GEMM_F32_INPUTS))
    return _export('gemm_i8', 'output0[N, M] +=! input0[N, K].cast(`int32`) * input1[M, K].cast(`int32`)', ('input0=int8[N:4096, K:4096]', 'input1=int8[M:4096, K:4096]'))


def _conv_op(dtype, n, c, f, hw):
    cast = '.to(`float32`)' if dtype == 'float16' else ''
    ir = (f'output0[N, F, HO, WO] +=! input0[N, C, HO + KH - 1, WO + KW - 1]{cast}.when([HO + KH - 1 >= 0, HO + KH - 1 < {hw}, '
          f'WO + KW - 1 >= 0, WO + KW - 1 < {hw}], 0.0) * input1[F, C, KH, KW]{cast} where HO in {hw}, WO in {hw}')
    return _export(f'conv_{dtype}_{n}_{c}_{f}_{hw}', ir, (f'input0={dtype}[N:{n}, C:{c}, H:{hw}, W:{hw}]', f'input1={dtype}[F:{f}, C:{c}, KH:3, KW:3]'))


def _gptq_op():
    return _export('gptq_linear', patterns.GPTQ_GEMV_IR, ('input0=float32[S:4096]', 'qweight=int32[L:512, N:12288]', 'scales=float32[K:32, N:12288]'))


# -- inputs -----------------------------------------------------------------------------------------------------------
class _Draws:
    """Seeded tensors made on the device."""

    def __init__(self, seed):
        self.dev = autort.device()
        self.gen = torch.Generator(device=self.dev).manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0, dtype=torch.float16):
        return (torch.randn(*shape, generator=self.gen, device=self.dev) * std + mean).to(dtype)

    def uniform(self, *shape, lo, hi, dtype=torch.float32):
        return (torch.rand(*shape, generator=self.gen, device=self.dev) * (hi - lo) + lo).to(dtype)

    def ints(self, *shape, lo, hi, dtype=torch.int32):
        return torch.randint(lo, hi, shape, generator=self.gen, device=self.dev, dtype=torch.int64 if hi > 2 ** 31 - 1 else dtype).to(dtype)

    def int4_linear(self, K, N, max_scale):
        """Packed weights: a uniform byte is two independent uniform nibbles."""
        return {'qweight': self.ints(K // 2, N, lo=0, hi=256, dtype=torch.uint8), 'qzeros': self.ints(K // 128, N // 2, lo=0, hi=256, dtype=torch.uint8),
                'scales': self.uniform(K // 128, N, lo=0.001, hi=max_scale, dtype=torch.float16)}

    def gptq_linear(self, K, N):
        return {'qweight': self.ints(K // 8, N, lo=-2 ** 31, hi=2 ** 31 - 1), 'scales': self.uniform(K // 128, N, lo=0.001, hi=0.005)}


# Scales up to this keep a layer's gain and its attention scores of the order of one, as a trained model's are: the
# rounding of one operator is then not amplified by the layers behind it.
MODEL_SCALE = 0.005


def _decoder(case, seed, max_seq):
    d = _Draws(seed)
    cfg = LlamaConfig(n_layers=case['layers'], dim=HEAD * case['heads'], n_heads=case['heads'], ffn=case['ffn'], vocab=case['vocab'], max_seq=max_seq)
    weights = {'embed': d.normal(cfg.vocab, cfg.dim, std=0.02), 'final_norm': d.normal(cfg.dim, std=0.1, mean=1.0),
               'lm_head': d.int4_linear(cfg.dim, cfg.vocab, MODEL_SCALE), 'layers': []}
    for _ in range(cfg.n_layers):
        weights['layers'].append({
            'att_norm': d.normal(cfg.dim, std=0.1, mean=1.0), 'ffn_norm': d.normal(cfg.dim, std=0.1, mean=1.0),
            'qkv': d.int4_linear(cfg.dim, 3 * cfg.dim, MODEL_SCALE), 'o': d.int4_linear(cfg.dim, cfg.dim, MODEL_SCALE),
            'gate_up': d.int4_linear(cfg.dim, 2 * cfg.ffn, MODEL_SCALE), 'down': d.int4_linear(cfg.ffn, cfg.dim, MODEL_SCALE)})
    return d, cfg, LlamaInt4Decoder(cfg, weights)


def prepare(case, seed):
    kind = case['kind']
    if kind == 'decode':
        pos, steps = case['pos'], case['steps']
        d, cfg, dec = _decoder(case, seed, max(384, pos + steps))
        prompt = d.ints(pos + steps + 1, lo=0, hi=cfg.vocab)
        dec.capture(greedy=True, prompt=prompt)
        dec.key_cache[:, :pos].normal_(generator=d.gen)
        dec.val_cache[:, :pos].normal_(generator=d.gen)
        return {'run': functools.partial(_run_decode, dec, int(prompt[pos]), pos, steps)}
    if kind == 'prefill':
        d, cfg, dec = _decoder(case, seed, max(384, case['tokens']))
        return {'run': functools.partial(_run_prefill, dec, d.ints(case['tokens'], lo=0, hi=cfg.vocab))}
    d = _Draws(seed)
    if kind == 'sample':
        return {'run': functools.partial(_run_sample, _sample_model(case, d), case['pos'])}
    if kind == 'map':
        x = d.uniform(case['n'], lo=-8, hi=8) if case['program'] == 'sigmoid' else d.normal(2, case['n'])
        return {'run': functools.partial(_map_op(case['program']), x)}
    if kind == 'rows':
        return {'run': functools.partial(_rows_op(case['program'], case['dtype']), d.normal(case['rows'], case['cols'], dtype=torch.float32))}
    if kind == 'partition':
        return {'run': functools.partial(autort.ops.partition_even_first_i32, d.ints(case['n'], lo=0, hi=2 ** 31))}
    if kind == 'w4':
        op = _export('w4', patterns.W4A16_IR, tuple(patterns.W4A16_INPUTS))
        lin = d.int4_linear(case['k'], case['n'], 0.02)
        return {'run': functools.partial(op, d.normal(case['m'], case['k']), lin['qweight'], lin['scales'], lin['qzeros'])}
    if kind == 'gemm':
        dtype, m, n, k = case['dtype'], case['m'], case['n'], case['k']
        if dtype == 'int8':
            a, b = d.ints(m, k, lo=-128, hi=128, dtype=torch.int8), d.ints(n, k, lo=-128, hi=128, dtype=torch.int8)
        else:
            a, b = d.normal(m, k, std=0.02, dtype=getattr(torch, dtype)), d.normal(k, n, std=0.02, dtype=getattr(torch, dtype))
            if dtype == 'float16':
                a, b = a * 16, b * 16           # keeps the float16 results out of the subnormal range
        return {'run': functools.partial(_gemm_op(dtype), a, b)}
    dtype = getattr(torch, case['dtype'])
    x = d.normal(case['n'], case['c'], case['hw'], case['hw'], dtype=dtype)
    w = d.normal(case['f'], case['c'], 3, 3, std=1 / math.sqrt(9 * case['c']), dtype=dtype)
    return {'run': functools.partial(_conv_op(case['dtype'], case['n'], case['c'], case['f'], case['hw']), x, w)}


def run(state):
    return state['run']()


def _run_decode(dec, token, pos, steps):
    """The tokens of a prompt, one at a time: every step also picks the next token, which the prompt then overrides."""
    dec.reset(token, pos)
    for _ in range(steps):
        dec.graph.replay()
    return {'logits': dec.logits, 'keys': dec.key_cache[:, pos:pos + steps], 'values': dec.val_cache[:, pos:pos + steps]}


def _run_prefill(dec, tokens):
    logits = dec.prefill(tokens)
    return {'logits': logits, 'keys': dec.key_cache[:, :tokens.numel()], 'values': dec.val_cache[:, :tokens.numel()]}


# -- samples/05_llama2_7b_int4.py as it is written ----------------------------------------------------------------------
def _sample_model(case, d):
    dim, ffn, pos = HEAD * case['heads'], case['ffn'], case['pos']
    inv = 1.0 / (10000.0 ** (torch.arange(0, HEAD, 2).float() / HEAD))
    model = {'linear': _gptq_op(), 'heads': case['heads'], 'x': d.normal(1, dim, dtype=torch.float32), 'rms_end': d.normal(dim, std=0.1, mean=1.0, dtype=torch.float32),
             'inv_freq': torch.cat([inv, inv]).view(HEAD).to(d.dev), 'att_f': torch.tensor([1 / math.sqrt(HEAD)], dtype=torch.float32, device=d.dev),
             'keys': d.normal(case['layers'], pos + 3, dim, dtype=torch.float32), 'values': d.normal(case['layers'], pos + 3, dim, dtype=torch.float32),
             'layers': []}
    for _ in range(case['layers']):
        model['layers'].append({'rms_att': d.normal(dim, std=0.1, mean=1.0, dtype=torch.float32), 'rms_ffn': d.normal(dim, std=0.1, mean=1.0, dtype=torch.float32),
                                'vqk': d.gptq_linear(dim, 3 * dim), 'o': d.gptq_linear(dim, dim), 'f1': d.gptq_linear(dim, ffn), 'f3': d.gptq_linear(dim, ffn),
                                'f2': d.gptq_linear(ffn, dim)})
    return model


def _run_sample(m, pos):
    heads, linear_op, key_cache, val_cache = m['heads'], m['linear'], m['keys'], m['values']
    rows = key_cache.size(1)

    def rmsnorm(x, weight):
        x = x.float()
        vsum = (x * x).sum().view(1)
        return autort.ops.rmsnorm_f32(x.view(-1), vsum, weight.float(), extra=[1.0 / int(x.numel())])

    def matmul_dequat(x, lin, memory_out=None):
        x = x.view(-1)
        memory_out = memory_out if memory_out is not None else torch.empty([lin['qweight'].size(-1)], dtype=x.dtype, device=x.device)
        return linear_op(x, lin['qweight'], lin['scales'], out=memory_out.view(-1))

    with torch.no_grad():
        x = m['x']
        for l, lw in enumerate(m['layers']):
            xb = rmsnorm(x, lw['rms_att'])
            local_cache = val_cache.select(0, l).narrow(0, pos, 3)
            matmul_dequat(xb, lw['vqk'], memory_out=local_cache.view(-1, 3 * xb.size(-1)))
            sq, sk = local_cache[1], local_cache[2]
            sq_out = torch.empty_like(sq).view(heads, HEAD)
            sk_out = key_cache.select(0, l).narrow(0, pos, 1).view(heads, HEAD)
            autort.ops.rotary_f32(sq.view(heads, 2, -1), m['inv_freq'], sq_out, extra=[pos, ])
            autort.ops.rotary_f32(sk.view(heads, 2, -1), m['inv_freq'], sk_out, extra=[pos, ])
            b_sk = key_cache.select(0, l).view(rows, heads, HEAD).narrow(0, 0, pos + 1)
            b_sv = val_cache.select(0, l).view(rows, heads, HEAD).narrow(0, 0, pos + 1)
            xb = autort.ops.attention_f32(sq_out, b_sk, b_sv, m['att_f'])
            x = x + matmul_dequat(xb, lw['o'])
            xb = rmsnorm(x, lw['rms_ffn'])
            xb = torch.nn.functional.silu(matmul_dequat(xb, lw['f1'])) * matmul_dequat(xb, lw['f3'])
            x = x + matmul_dequat(xb, lw['f2'])
        x = rmsnorm(x, m['rms_end'])
    return {'hidden': x, 'keys': key_cache[:, pos], 'values': val_cache[:, pos:pos + 3]}


# -- what a pass cannot do without -------------------------------------------------------------------------------------
def _layer_shapes(case):
    dim, ffn = HEAD * case['heads'], case['ffn']
    return [(dim, 3 * dim), (dim, dim), (dim, 2 * ffn), (ffn, dim)]


def work(case):
    kind = case['kind']
    if kind == 'map':
        return {'bytes': case['n'] * (8 if case['program'] == 'sigmoid' else 6), 'flops': 4 * case['n']}
    if kind == 'rows':
        return {'bytes': 8 * case['rows'] * case['cols'], 'flops': 5 * case['rows'] * case['cols']}
    if kind == 'partition':
        return {'bytes': 8 * case['n'], 'flops': 0}
    if kind == 'w4':
        return {'bytes': workloads.w4_bytes(case['m'], case['k'], case['n']), 'flops': 2 * case['m'] * case['k'] * case['n']}
    if kind in ('decode', 'prefill'):
        dim, layers = HEAD * case['heads'], case['layers']
        weights = layers * sum(workloads.w4_bytes(0, k, n) for k, n in _layer_shapes(case))
        head = workloads.w4_bytes(0, dim, case['vocab'])
        per_token = 2 * layers * sum(k * n for k, n in _layer_shapes(case))
        last = 2 * dim * case['vocab']
        if kind == 'prefill':
            t = case['tokens']
            return {'bytes': weights + head + 2 * t * dim * (1 + 2 * layers), 'flops': t * per_token + last + 2 * layers * t * (t + 1) * dim}
        steps = case['steps']
        attended = sum(case['pos'] + i + 1 for i in range(steps))
        return {'bytes': steps * (weights + head) + 4 * layers * dim * (attended + steps), 'flops': steps * (per_token + last) + 4 * layers * dim * attended}
    if kind == 'gemm':
        m, n, k = case['m'], case['n'], case['k']
        size, out = {'float16': (2, 2), 'float32': (4, 4), 'int8': (1, 4)}[case['dtype']]
        return {'bytes': size * (m * k + k * n) + out * m * n, 'flops': 2 * m * n * k}
    if kind == 'conv':
        size = 2 if case['dtype'] == 'float16' else 4
        n, c, f, hw = case['n'], case['c'], case['f'], case['hw']
        return {'bytes': size * (n * c * hw * hw + 9 * f * c) + 4 * n * f * hw * hw, 'flops': 2 * 9 * n * f * c * hw * hw}
    dim, ffn, layers = HEAD * case['heads'], case['ffn'], case['layers']
    weights = sum(k * n // 2 + (k // 128) * n * 4 for k, n in [(dim, 3 * dim), (dim, dim), (dim, ffn), (dim, ffn), (ffn, dim)])
    flops = 2 * sum(k * n for k, n in _layer_shapes(case))
    return {'bytes': layers * (weights + 8 * dim * (case['pos'] + 4)), 'flops': layers * flops}


def tolerance(case):
    kind = case['kind']
    if kind == 'partition' or (kind == 'gemm' and case['dtype'] == 'int8'):
        return 'exact'
    if kind in ('decode', 'prefill'):
        # float16 roundings of up to 32 layers, one behind the other: the package's own decoders, which differ only in
        # where they round and in which order they sum, are 0.4-0.7 % apart
        return {'rel': 1.5e-2, 'max': 0.1}
    if kind == 'sample':
        return {'rel': 1e-4}                    # float32 sums of thousands of terms, through several layers
    if kind == 'w4' or (kind == 'gemm' and case['dtype'] == 'float16') or (kind == 'map' and case['program'] == 'silu_mul'):
        return {'rel': 1e-3, 'max': 1e-2}       # float16 results of float32 sums
    return {'rel': 1e-5}                        # float32
