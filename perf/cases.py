"""Performance cases of the task-graph executor: what a program that uses it has it do, from the smallest graph to the
largest, through its public entry points.

A pass is one run of a submitted graph, as a training or serving loop makes it: Executor.relaunch(), Executor.finish().
The buffers live on the GPU for as long as the program does; the outputs are those buffers, seen as torch tensors.

Kinds of cases:
  mlp      independent MLPs trained together (kvm_amd.workloads.mlp), some steps per graph, f32
  gpt      GPT training steps (kvm_amd.workloads.gpt): tiny f32, bf16 storage, the f32 shape
  layer    forward and backward of one decoder layer of RMSNorm, RoPE, grouped-query attention and SwiGLU, built from
           registry operators: f32, or bf16 storage with f32 SwiGLU operands ("bf16")
  prefill  forward of decoder layers over whole prompts, bf16 storage and weights, filling the KV cache
  decode   one greedy decode step (kvm_amd.workloads.qwen3) at a given context
  tail     the end of a decode step with sampling: final norm, LM head, top-k temperature sampling
  head     a language model's training head: logits, cross entropy, both gradients, bf16 storage
Sizes: the configurations of the generators, the benchmark and the tests; token counts, batches and contexts are any
number, as data has them, while model widths and vocabularies are padded to whole vectors.
"""
from __future__ import annotations

import functools
import math

import torch

from kvm_amd import bundle as bl
from kvm_amd import compiler
from kvm_amd.executor import PATH_AUTO, Executor
from kvm_amd.workloads import Builder, Workload, gpt, mlp, qwen3, split

DEV = 'cuda'
GPT162M = dict(d=768, heads=12, ffn=3072)
GPT355M = dict(d=1024, heads=16, ffn=4096)
QWEN3_8B = dict(d=4096, heads=32, kv=8, hd=128, ffn=12288)


def listed():
    return [
        # one small model, one step per launch: the launch and the length of the chain are what it costs
        dict(name='mlp_one_small', kind='mlp', widths='64', batch=64, steps=1),
        # eight models of different widths sharing the chip, several steps per launch (benchmark configuration 2's shape)
        dict(name='mlp_eight', kind='mlp', widths='64,96,128,192,256,384,512,768', batch=256, steps=10),
        # benchmark configuration 1: a model small enough that every task is short
        dict(name='gpt_tiny', kind='gpt', dtype='f32', layers=2, d=128, heads=4, ffn=512, T=64, batch=8, vocab=256, steps=10),
        # benchmark configuration 3, the whole call: pretraining step in bf16 storage
        dict(name='gpt_162m', kind='gpt', dtype='bf16', layers=12, T=1024, batch=4, vocab=50304, steps=1, **GPT162M),
        # its layer on sequences that are no multiple of anything (fine-tuning data, last batches)
        dict(name='gpt_layer_ragged', kind='gpt', dtype='bf16', layers=1, T=1000, batch=3, vocab=8192, steps=1, **GPT162M),
        # benchmark configuration 4's layer, in exact fp32
        dict(name='gpt_layer_f32', kind='gpt', dtype='f32', layers=1, T=1024, batch=4, vocab=4096, steps=1, **GPT355M),
        # a decoder layer as the operators' other family spells it, trained in f32, with a ragged length
        dict(name='layer_f32', kind='layer', dtype='f32', d=1024, heads=8, kv=2, hd=128, ffn=2816, T=500, batch=2),
        # the same family in bf16 at a serving model's head size, as it is fine-tuned
        dict(name='layer_bf16', kind='layer', dtype='bf16', d=2048, heads=16, kv=4, hd=128, ffn=6144, T=1024, batch=2),
        # a prompt through one layer of the benchmark's decode model
        dict(name='prefill', kind='prefill', layers=1, T=1531, batch=1, **QWEN3_8B),
        # benchmark configuration 5, the whole call at batch 1
        dict(name='decode_b1', kind='decode', layers=36, ctx=4096, batch=1, vocab=151936, **QWEN3_8B),
        # layers of it at the benchmark's batch
        dict(name='decode_b8', kind='decode', layers=6, ctx=4096, batch=8, vocab=32000, **QWEN3_8B),
        # choosing tokens by sampling, as served text is
        dict(name='tail_sampled', kind='tail', batch=4, d=4096, vocab=32000, topk=50),
    ]


def _log(rng, lo, hi, to=1):
    """An integer of [lo, hi], spread over its logarithm, a multiple of `to`."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / to)) * to))


def draw(rng):
    kind = rng.choice(['mlp', 'gpt', 'gpt', 'layer', 'layer', 'prefill', 'decode', 'decode', 'tail', 'head'])
    if kind == 'mlp':
        n = rng.randint(1, 8)
        widths = ','.join(str(w) for w in sorted(rng.sample(mlp.WIDTHS, n)))
        return dict(kind=kind, widths=widths, batch=_log(rng, 16, 512), steps=rng.randint(1, 10))
    if kind == 'gpt':
        dtype = rng.choice(['f32', 'bf16', 'bf16'])
        T = rng.choice([_log(rng, 32, 1024), _log(rng, 64, 1024, 64)])
        batch = max(1, min(8, rng.randint(1, 4096) // T + 1))
        if T * batch <= 512 and dtype == 'f32':
            return dict(kind=kind, dtype=dtype, layers=rng.randint(1, 2), d=128, heads=4, ffn=512, T=min(T, 128), batch=batch, vocab=256,
                        steps=rng.randint(1, 6))
        return dict(kind=kind, dtype=dtype, layers=1, T=T, batch=batch, vocab=_log(rng, 1024, 16384, 64), steps=1,
                    **(GPT162M if dtype == 'bf16' else rng.choice([GPT162M, GPT355M])))
    if kind == 'layer':
        hd = rng.choice([64, 128])
        kv = rng.choice([1, 2, 4])
        heads = kv * rng.choice([1, 2, 4])
        d = rng.choice([512, 1024, 2048])
        T = rng.choice([_log(rng, 64, 1536), _log(rng, 64, 1536, 128)])
        return dict(kind=kind, dtype=rng.choice(['f32', 'bf16']), d=d, heads=heads, kv=kv, hd=hd, ffn=_log(rng, d, 3 * d, 64), T=T,
                    batch=rng.randint(1, max(1, min(4, 2048 // T))))
    if kind == 'prefill':
        d = rng.choice([1024, 2048, 4096])
        batch = rng.randint(1, 4)
        return dict(kind=kind, layers=1, T=_log(rng, 32, 2048 // batch), batch=batch, d=d, heads=d // 128, kv=rng.choice([4, 8]), hd=128,
                    ffn=_log(rng, 2 * d, 3 * d, 64))
    if kind == 'decode':
        d = rng.choice([1024, 2048, 4096])
        return dict(kind=kind, layers=rng.randint(1, 4), ctx=_log(rng, 16, 8192), batch=rng.choice([1, 1, 2, 3, 4, 6, 8, 12, 16]),
                    vocab=_log(rng, 4096, 65536, 64), d=d, heads=d // 128, kv=d // 512 if rng.random() < 0.7 else d // 256, hd=128, ffn=3 * d)
    if kind == 'tail':
        return dict(kind=kind, batch=rng.randint(1, 8), d=rng.choice([1024, 2048, 4096]), vocab=_log(rng, 4096, 65536, 64),
                    topk=rng.choice([0, 20, 50, 200]))
    return dict(kind=kind, rows=_log(rng, 64, 4096), d=768, vocab=_log(rng, 4096, 50304, 64))


# ------------------------------------------------------------------------------------------------ graphs

class Phases(Builder):
    """A graph of phases: the tasks of one follow all tasks of the one before, through one no-op."""

    def __init__(self):
        super().__init__(0)
        self.after, self.open = [], []

    def add(self, op, **args):
        self.open.append(self.task(op, after=self.after, **args))

    def barrier(self):
        self.after = self.join(self.open, len(self.open))
        self.open = []

    def rows(self, op, n, parts=256, **args):
        for r0, r1 in split(n, parts):
            self.add(op, r0=r0, r1=r1, **args)

    def flat(self, op, n, **args):
        """n elements, in whole vectors of 8 but for the last ones."""
        for lo, hi in split(-(-n // 8), 256):
            self.add(op, e0=8 * lo, e1=min(n, 8 * hi), **args)

    def gemm(self, dtype, a, b, out, M, N, K, flags=0, bias=None, res=None, pre=None):
        """The tiles that the GPT generator gives a GEMM of this shape."""
        t = lambda tm, tn: -(-M // tm) * -(-N // tn)   # noqa: E731
        if dtype == 'bf16':
            op, tm, tn, fl = ('matmul_mma_bf16', 128, 256, flags) if t(128, 256) >= gpt.GPTBuilder.TILES_MMA else \
                             ('matmul_tile_bf16', 128, 128, flags | 32)
        else:
            op, (tm, tn, fl) = 'matmul_tile', self.tile_f32(M, N, flags)
        for m0 in range(0, M, tm):
            for n0 in range(0, N, tn):
                self.add(op, a=a, b=b, out=out, bias=bias, res=res, pre=pre, m0=m0, n0=n0, M=M, N=N, K=K, flags=fl, alpha=1.0)

    @staticmethod
    def tile_f32(M, N, flags):
        t = lambda tm, tn: -(-M // tm) * -(-N // tn)   # noqa: E731
        if M >= 256 and N >= 128 and t(256, 128) >= gpt.GPTBuilder.F32_TILES_256:
            return 256, 128, flags | 64
        if M >= 128 and N >= 128 and t(128, 128) >= gpt.GPTBuilder.F32_TILES_128:
            return 128, 128, flags | 32
        return 64, 64, flags

    def attention(self, op, batch, T, H, Hkv, per_kv=False, **args):
        for b in range(batch):
            for h in range(Hkv if per_kv else H):
                for t0 in range(0, T, 128):
                    if per_kv:
                        self.add(op, b=b, kvh=h, k0=t0, T=T, H=H, **args)
                    else:
                        self.add(op, b=b, h=h, q0=t0, T=T, H=H, Hkv=Hkv, **args)


THETA, EPS = 1e6, 1e-6


def _layer_graph(c):
    """Forward and backward of a decoder layer. x and the gradient dy of its output are given."""
    d, H, Hkv, hd, F, T, N = c['d'], c['heads'], c['kv'], c['hd'], c['ffn'], c['T'], c['T'] * c['batch']
    dt, nq, nkv = c['dtype'], c['heads'] * c['hd'], c['kv'] * c['hd']
    g = Phases()
    g.normal('x', N, d, dt, scale=1.0)
    g.normal('dy', N, d, dt, scale=1.0)
    for n, r, k in (('wq', nq, d), ('wk', nkv, d), ('wv', nkv, d), ('wo', d, nq), ('wg', F, d), ('wu', F, d), ('wd', d, F)):
        g.normal(n, r, k, dt, scale=1.0 / math.sqrt(k))
        g.fill('d.' + n, r, k)
    for n in ('g1', 'g2'):
        g.fill(n, 1, d, value=1.0)
        g.fill('d.' + n, 1, d)
    for n, k in (('h1', d), ('q', nq), ('k', nkv), ('v', nkv), ('qr', nq), ('kr', nkv), ('o', nq), ('xm', d), ('h2', d), ('y', d), ('dh', d),
                 ('dn', d), ('dxm', d), ('do', nq), ('dqr', nq), ('dkr', nkv), ('dq', nq), ('dk', nkv), ('dv', nkv), ('dx', d)):
        g.fill(n, N, k, dt)
    for n in ('gate', 'up', 'h', 'dhh', 'dgate', 'dup'):      # the SwiGLU operators' storage is f32
        g.fill(n, N, F)
    for n in ('rs1', 'rs2'):
        g.fill(n, N)
    g.fill('lse', N * H), g.fill('delta', N * H)
    scale, fused = 1.0 / math.sqrt(hd), dt == 'f32'
    rope = dict(pos=None, T=T, hd=hd, theta=THETA)

    g.rows('rmsnorm_fwd', N, x='x', gamma='g1', out='h1', rstd='rs1', d=d, eps=EPS), g.barrier()
    for n, k in (('q', nq), ('k', nkv), ('v', nkv)):
        g.gemm(dt, 'h1', 'w' + n, n, N, k, d, flags=2)
    g.barrier()
    g.rows('rope_fwd', N, x='q', out='qr', H=H, **rope), g.rows('rope_fwd', N, x='k', out='kr', H=Hkv, **rope), g.barrier()
    g.attention('attn_fwd', c['batch'], T, H, Hkv, q='qr', k='kr', v='v', o='o', lse='lse', hd=hd, scale=scale), g.barrier()
    g.gemm(dt, 'o', 'wo', 'xm', N, d, nq, flags=2, res='x'), g.barrier()
    g.rows('rmsnorm_fwd', N, x='xm', gamma='g2', out='h2', rstd='rs2', d=d, eps=EPS), g.barrier()
    g.gemm(dt, 'h2', 'wg', 'gate', N, F, d, flags=2)
    if fused:
        g.barrier()
        tm, tn, fl = g.tile_f32(N, F, 2)
        for m0 in range(0, N, tm):
            for n0 in range(0, F, tn):
                g.add('matmul_tile_silu_mul', a='h2', b='wu', out='h', gate='gate', up='up', m0=m0, n0=n0, M=N, N=F, K=d, flags=fl, alpha=1.0)
    else:
        g.gemm(dt, 'h2', 'wu', 'up', N, F, d, flags=2), g.barrier()
        g.flat('silu_mul_fwd', N * F, gate='gate', up='up', out='h')
    g.barrier()
    g.gemm(dt, 'h', 'wd', 'y', N, d, F, flags=2, res='xm')
    # backward
    g.gemm(dt, 'dy', 'h', 'd.wd', d, F, N, flags=1)
    if fused:
        tm, tn, fl = g.tile_f32(N, F, 0)
        for m0 in range(0, N, tm):
            for n0 in range(0, F, tn):
                g.add('matmul_tile_silu_mul_bwd', a='dy', b='wd', gate='gate', up='up', dgate='dgate', dup='dup', m0=m0, n0=n0, M=N, N=F, K=d,
                      flags=fl, alpha=1.0)
    else:
        g.gemm(dt, 'dy', 'wd', 'dhh', N, F, d), g.barrier()
        g.flat('silu_mul_bwd', N * F, gate='gate', up='up', dy='dhh', dgate='dgate', dup='dup', acc=0)
    g.barrier()
    g.gemm(dt, 'dgate', 'wg', 'dh', N, d, F), g.gemm(dt, 'dgate', 'h2', 'd.wg', F, d, N, flags=1)
    g.gemm(dt, 'dup', 'h2', 'd.wu', F, d, N, flags=1), g.barrier()
    g.gemm(dt, 'dup', 'wu', 'dh', N, d, F, flags=4), g.barrier()
    _norm_bwd(g, N, d, 'xm', 'dh', 'g2', 'rs2')
    g.flat('residual_add', N * d, a='dn', b='dy', out='dxm'), g.barrier()
    g.gemm(dt, 'dxm', 'wo', 'do', N, nq, d), g.gemm(dt, 'dxm', 'o', 'd.wo', d, nq, N, flags=1), g.barrier()
    g.rows('attn_bwd_delta', N, o='o', do='do', delta='delta', T=T, H=H, hd=hd), g.barrier()
    kw = dict(q='qr', k='kr', v='v', do='do', lse='lse', delta='delta', hd=hd, scale=scale)
    g.attention('attn_bwd_dq', c['batch'], T, H, Hkv, dq='dqr', **kw)
    g.attention('attn_bwd_dkv', c['batch'], T, H, Hkv, per_kv=True, dk='dkr', dv='dv', **kw), g.barrier()
    g.rows('rope_bwd', N, x='dqr', out='dq', H=H, **rope), g.rows('rope_bwd', N, x='dkr', out='dk', H=Hkv, **rope), g.barrier()
    for i, n in enumerate(('q', 'k', 'v')):
        k = nq if n == 'q' else nkv
        g.gemm(dt, 'd' + n, 'w' + n, 'dh', N, d, k, flags=4 if i else 0)
        g.gemm(dt, 'd' + n, 'h1', 'd.w' + n, k, d, N, flags=1), g.barrier()
    _norm_bwd(g, N, d, 'x', 'dh', 'g1', 'rs1')
    g.flat('residual_add', N * d, a='dn', b='dxm', out='dx')
    return Workload(g.spec('layer'), g.init_override)


def _norm_bwd(g, N, d, x, dy, gamma, rstd):
    for c0, c1 in split(d, d // 64):
        g.add('norm_bwd_params', x=x, dy=dy, mean=None, rstd=rstd, dgamma='d.' + gamma, dbeta=None, R=N, d=d, c0=c0, c1=c1, acc=0)
    g.rows('rmsnorm_bwd_dx', N, x=x, dy=dy, gamma=gamma, rstd=rstd, dx='dn', d=d, acc=0), g.barrier()


def _prefill_graph(c):
    d, H, Hkv, hd, F, T, B = c['d'], c['heads'], c['kv'], c['hd'], c['ffn'], c['T'], c['batch']
    N, nq, nkv, Tmax, dt = T * B, H * hd, Hkv * hd, T + 64, 'bf16'
    g = Phases()
    g.normal('x', N, d, dt, scale=1.0)
    g.values('lens', [0] * B, B)
    for n, k in (('h', d), ('q', nq), ('k', nkv), ('v', nkv), ('o', nq), ('gate', F), ('up', F)):
        g.fill(n, N, k, dt)
    g.fill('rs', N), g.fill('lse', N * H)
    for l in range(c['layers']):
        for n, r, k in (('wq', nq, d), ('wk', nkv, d), ('wv', nkv, d), ('wo', d, nq), ('wg', F, d), ('wu', F, d), ('wd', d, F)):
            g.normal(f'{n}.{l}', r, k, dt, scale=1.0 / math.sqrt(k))
        for n, k in (('g1', d), ('g2', d), ('qn', hd), ('kn', hd)):
            g.fill(f'{n}.{l}', 1, k, value=1.0)
        g.fill(f'kc.{l}', B * Hkv * Tmax, hd, dt), g.fill(f'vc.{l}', B * Hkv * Tmax, hd, dt)
        g.fill(f'xm.{l}', N, d, dt), g.fill(f'y.{l}', N, d, dt)
    x = 'x'
    for l in range(c['layers']):
        g.rows('rmsnorm_fwd', N, x=x, gamma=f'g1.{l}', out='h', rstd='rs', d=d, eps=EPS), g.barrier()
        for n, k in (('q', nq), ('k', nkv), ('v', nkv)):
            g.gemm(dt, 'h', f'w{n}.{l}', n, N, k, d, flags=2)
        g.barrier()
        for n, heads in (('q', H), ('k', Hkv)):
            g.rows('head_rmsnorm', N, x=n, gamma=f'{n}n.{l}', out=n, H=heads, hd=hd, eps=EPS)
        g.barrier()
        for n, heads in (('q', H), ('k', Hkv)):
            g.rows('rope_fwd', N, x=n, out=n, pos=None, T=T, H=heads, hd=hd, theta=THETA)
        g.barrier()
        for b in range(B):
            g.add('kv_append', knew='k', vnew='v', kc=f'kc.{l}', vc=f'vc.{l}', lens='lens', b0=b, b1=b + 1, n_new=T, Hkv=Hkv, hd=hd, Tmax=Tmax)
        g.attention('attn_fwd', B, T, H, Hkv, q='q', k='k', v='v', o='o', lse='lse', hd=hd, scale=1.0 / math.sqrt(hd)), g.barrier()
        g.gemm(dt, 'o', f'wo.{l}', f'xm.{l}', N, d, nq, flags=2, res=x), g.barrier()
        g.rows('rmsnorm_fwd', N, x=f'xm.{l}', gamma=f'g2.{l}', out='h', rstd='rs', d=d, eps=EPS), g.barrier()
        g.gemm(dt, 'h', f'wg.{l}', 'gate', N, F, d, flags=2), g.gemm(dt, 'h', f'wu.{l}', 'up', N, F, d, flags=2), g.barrier()
        g.flat('silu_mul_fwd', N * F, gate='gate', up='up', out='gate'), g.barrier()
        g.gemm(dt, 'gate', f'wd.{l}', f'y.{l}', N, d, F, flags=2, res=f'xm.{l}'), g.barrier()
        x = f'y.{l}'
    return Workload(g.spec('prefill'), g.init_override)


def _decode_graph(c):
    """The generator's decode step, made one that can be passed again: the context stays and the chosen token has a
    buffer of its own, so that every pass is the same position of the same text."""
    w = qwen3.build(qwen3.Qwen3Config(layers=c['layers'], hidden=c['d'], heads=c['heads'], kv_heads=c['kv'], head_dim=c['hd'], ffn=c['ffn'],
                                      vocab=c['vocab'], ctx=c['ctx'], batch=c['batch'], max_new=64))
    w.spec['buffers'].append({'name': 'next', 'rows': c['batch'], 'cols': 1, 'dtype': 'i32'})
    tasks = w.spec['graphs'][0]['tasks']
    tasks[:] = [t for t in tasks if t['op'] != 'counter_inc']
    for t in tasks:
        if t['op'] == 'argmax':
            t['args']['out'] = 'next'
    return w


def _tail_graph(c):
    B, d, V = c['batch'], c['d'], c['vocab']
    g = Phases()
    g.normal('x', B, d, scale=1.0)
    g.fill('gf', 1, d, value=1.0)
    g.normal('whead', V, d, 'bf16', scale=4.0 / math.sqrt(d))      # logits of the spread that trained models have
    g.fill('logits', B, V)
    g.values('tok', [0] * B, B)
    for lo, hi in split(V // 16, 512):
        if B == 1:
            g.add('gemv_bf16', x='x', x2=None, gamma='gf', w='whead', out='logits', res=None, n0=16 * lo, n1=16 * hi, K=d, pro=1, eps=EPS)
        else:
            g.add('gemv_bf16_rows', x='x', x2=None, gamma='gf', w='whead', out='logits', res=None, n0=16 * lo, n1=16 * hi, K=d, M=B, pro=1, eps=EPS)
    g.barrier()
    for b in range(B):
        g.add('sample', logits='logits', out='tok', ctr=None, r0=b, r1=b + 1, V=V, temp=0.8, topk=c['topk'], seed=1234)
    return Workload(g.spec('tail'), g.init_override)


def _head_graph(c):
    N, d, V, dt = c['rows'], c['d'], c['vocab'], 'bf16'
    g = Phases()
    g.normal('h', N, d, dt, scale=1.0)
    g.normal('w', V, d, dt, scale=1.0 / math.sqrt(d))
    g.values('tgt', [0] * N, N)
    g.fill('logits', N, V, dt), g.fill('dlogits', N, V, dt)
    g.fill('rowloss', N), g.fill('lse', N), g.fill('loss', 2)
    g.fill('dh', N, d, dt), g.fill('d.w', V, d)
    g.gemm(dt, 'h', 'w', 'logits', N, V, d, flags=2), g.barrier()
    g.rows('softmax_ce_fused', N, parts=512, logits='logits', tgt='tgt', rowloss='rowloss', lse='lse', dlogits='dlogits', V=V, ignore=-1, N=N, scale=1.0)
    g.barrier()
    g.add('softmax_ce_reduce', rowloss='rowloss', tgt='tgt', loss='loss', N=N, ignore=-1)
    g.gemm(dt, 'dlogits', 'w', 'dh', N, d, V), g.gemm(dt, 'dlogits', 'h', 'd.w', V, d, N, flags=1)
    return Workload(g.spec('head'), g.init_override)


def _gpt_config(c):
    tiny = dict(tasks_target=64, opt_chunk=8192) if c['d'] <= 128 else {}      # the generator's choice for tiny models
    return gpt.GPTConfig(layers=c['layers'], d=c['d'], heads=c['heads'], T=c['T'], vocab=c['vocab'], ffn=c['ffn'], batch=c['batch'],
                         dtype=c['dtype'], steps=c['steps'], **tiny)


def _widths(c):
    return tuple(int(w) for w in c['widths'].split(','))


@functools.lru_cache(maxsize=None)
def _graph(items):
    """(loaded bundle, executor-side initialisers) of a case: compiled once, as a program does."""
    c = dict(items)
    if c['kind'] == 'mlp':
        w = mlp.build(mlp.MLPConfig(widths=_widths(c), batch=c['batch'], steps=c['steps']))
    elif c['kind'] == 'gpt':
        w = gpt.build(_gpt_config(c))
    else:
        w = {'layer': _layer_graph, 'prefill': _prefill_graph, 'decode': _decode_graph, 'tail': _tail_graph, 'head': _head_graph}[c['kind']](c)
    scales = {b['name']: b['init']['scale'] for b in w.spec['buffers'] if b.get('init', {}).get('kind') == 'seeded'}
    scales.update({n: i['scale'] for n, i in w.init_override.items()})
    return bl.load(compiler.compile_spec(w.spec)), scales


def _key(case):
    return tuple(sorted((k, v) for k, v in case.items() if k != 'name'))


# ------------------------------------------------------------------------------------------------ state

class _View:
    """A device buffer of an executor in the form that torch takes; keeps the executor while a tensor is alive."""

    def __init__(self, ex, name, shape, kind):
        self.ex = ex
        self.__cuda_array_interface__ = dict(shape=shape, typestr=kind, data=(ex.device_ptr(name), False), version=2)


KINDS = {bl.DT_F32: ('<f4', torch.float32), bl.DT_I32: ('<i4', torch.int32), bl.DT_BF16: ('<i2', torch.bfloat16)}


def _view(ex, m):
    kind, dtype = KINDS[m['dtype']]
    t = torch.as_tensor(_View(ex, m['name'], (m['rows'], m['cols']), kind), device=DEV)
    return t.view(dtype) if dtype is torch.bfloat16 else t


def _modulus(case, name):
    """What the integers of input `name` run over, or None where it is no input."""
    if name in ('ids', 'tgt', 'tok') and case['kind'] in ('gpt', 'head', 'decode'):
        return case['vocab']
    return 10 if case['kind'] == 'mlp' and name.endswith('.y') else None


def _inputs(case, seed, take):
    """Fills every input buffer from the seed: take(m) gives the tensor of metadata entry m. The random numbers come in
    the order of the buffer table. Returns name -> tensor."""
    lb, scales = _graph(_key(case))
    rng = torch.Generator(device=DEV).manual_seed(seed)
    got = {}
    for m in lb.metadata['buffers']:
        name = m['name']
        if name.endswith('.bf') and name[:-3] in got:           # the GEMM copy of a weight starts as the weight, rounded
            got[name] = take(m).copy_(got[name[:-3]])
        elif name in scales:
            got[name] = take(m).normal_(0.0, scales[name], generator=rng)
        elif _modulus(case, name):
            got[name] = take(m).random_(0, _modulus(case, name), generator=rng)
        elif m['init']['kind'] == 'fill' and m['init']['value'] == 1:   # gains: near one
            got[name] = take(m).normal_(1.0, 0.1, generator=rng)
    return got


def _outputs(case):
    """Names of the buffers that a pass computes and a program reads."""
    k = case['kind']
    if k == 'mlp':
        nets = range(len(_widths(case)))                     # after many steps on one batch the last gradients are noise
        return [f'm{i}.{n}' for i in nets for n in ('logits', 'loss', 'W0', 'b0', 'W1', 'W2')] + \
               ([f'd.m{i}.W0' for i in nets] if case['steps'] == 1 else [])
    if k == 'gpt':
        L = case['layers']
        per = ('wq', 'wk', 'wv', 'wo', 'w1', 'w2', 'bq', 'b1', 'ln1g', 'ln2b') if L <= 3 else ('wq', 'wo', 'w1', 'w2')
        return ['loss', 'logits', 'gscale', 'wte', 'd.wte', 'd.wpe', 'd.lnfg'] + [f'd.{n}.{l}' for l in range(L) for n in per]
    if k == 'layer':
        return ['y', 'dx'] + ['d.' + n for n in ('wq', 'wk', 'wv', 'wo', 'wg', 'wu', 'wd', 'g1', 'g2')]
    if k == 'prefill':
        return [f'{n}.{l}' for l in range(case['layers']) for n in ('y', 'kc', 'vc')]
    if k == 'decode':     # a batch's tokens too; a single one says nothing that its logits do not, but for a near-tie all of it
        return ['logits', 'x', f'kc.{case["layers"] - 1}', f'vc.{case["layers"] - 1}'] + (['next'] if case['batch'] > 1 else [])
    if k == 'tail':
        return ['logits', 'tok']
    return ['loss', 'logits', 'dlogits', 'dh', 'd.w']


def prepare(case, seed):
    lb, _ = _graph(_key(case))
    ex = Executor(num_vars=max(1, len(lb.metadata['variables'])), trace=False, timeout_s=60.0, path=PATH_AUTO)
    for m in lb.metadata['buffers']:
        plain = m['init'] if m['init']['kind'] in ('fill', 'values') else None
        ex.add_buffer(m['name'], m['rows'], m['cols'], m['dtype'], init=plain)
    for v in lb.metadata['variables']:
        ex.set_version(v['id'], v['base_version'])
    ex.submit(lb)
    torch.cuda.synchronize()                                     # the executor's own initialisation is on its own stream
    _inputs(case, seed, lambda m: _view(ex, m))
    torch.cuda.synchronize()
    by = {m['name']: m for m in lb.metadata['buffers']}
    return {'ex': ex, 'out': {n: _view(ex, by[n]) for n in _outputs(case)}}


def run(state):
    state['ex'].relaunch()
    state['ex'].finish()
    return state['out']


# ------------------------------------------------------------------------------------------------ what a pass needs

def work(case):
    """Bytes: inputs, state and weights read once, outputs and state written once. flops: products and attention."""
    k, c = case['kind'], case
    if k == 'mlp':
        m = mlp.MLPConfig(widths=_widths(c), batch=c['batch'])
        return {'bytes': 28 * mlp.param_count(m) + 4 * len(m.widths) * m.batch * m.d_in, 'flops': mlp.step_flops(m) * c['steps']}
    if k == 'gpt':
        g = _gpt_config(c)
        return {'bytes': (30 if c['dtype'] == 'bf16' else 28) * gpt.param_count(g) + (2 if c['dtype'] == 'bf16' else 4) * c['T'] * c['batch'] * c['vocab'],
                'flops': gpt.step_flops(g)['total'] * c['steps']}
    if k == 'head':
        return {'bytes': 2 * (2 * c['rows'] * c['d'] + c['vocab'] * c['d'] + 2 * c['rows'] * c['vocab']) + 4 * c['vocab'] * c['d'],
                'flops': 6.0 * c['rows'] * c['d'] * c['vocab']}
    if k == 'tail':
        return {'bytes': 2 * c['d'] * c['vocab'] + 4 * c['batch'] * (c['vocab'] + c['d']), 'flops': 2.0 * c['batch'] * c['d'] * c['vocab']}
    nq, nkv = c['heads'] * c['hd'], c['kv'] * c['hd']
    W = c['d'] * (2 * nq + 2 * nkv + 3 * c['ffn'])
    if k == 'decode':
        kv = 2 * nkv * (c['ctx'] + 1) * c['batch']
        return {'bytes': 2 * (c['layers'] * (W + kv) + c['vocab'] * c['d']) + 4 * c['batch'] * c['vocab'],
                'flops': 2.0 * c['batch'] * (c['layers'] * W + c['vocab'] * c['d']) + 4.0 * c['layers'] * c['batch'] * nq * (c['ctx'] + 1)}
    N, pairs = c['T'] * c['batch'], c['batch'] * c['heads'] * c['T'] * (c['T'] + 1) / 2
    if k == 'prefill':
        return {'bytes': 2 * c['layers'] * (W + 2 * N * nkv) + 4 * N * c['d'], 'flops': c['layers'] * (2.0 * N * W + 4.0 * pairs * c['hd'])}
    es = 2 if c['dtype'] == 'bf16' else 4
    return {'bytes': (es + 4) * W + es * 4 * N * c['d'], 'flops': 6.0 * N * W + 14.0 * pairs * c['hd']}


def tolerance(case):
    """About four times the largest error against 64 bits that was measured over the listed and thirty drawn cases (in
    brackets). AdamW's first steps are close to the gradient's sign: where it is near zero they carry rounding into the
    weights, so several steps, and many layers of bf16, are looser than one."""
    k = case['kind']
    if k == 'mlp':
        return {'rel': 2e-2 if case['steps'] > 1 else 1e-4}                    # 5.5e-3; 1.5e-6, and a second step after it
    if k == 'gpt' and case['dtype'] == 'bf16':
        return {'rel': 9e-2 if case['layers'] > 3 else 3e-2}                   # 2.3e-2, 7.4e-3
    if k == 'gpt':
        return {'rel': 1e-3 if case['steps'] > 1 else 1e-4}                    # 9.5e-5; 7.6e-6, and a second step after it
    if k == 'layer':
        return {'rel': 3e-2 if case['dtype'] == 'bf16' else 1e-5}              # 7.3e-3, 2.4e-6
    if k == 'prefill':
        return {'rel': 1.5e-2}                                                 # 3.6e-3
    if k == 'decode':
        return {'rel': 9e-2 if case['layers'] > 6 else 3.5e-2, 'differ': 0.5}  # 2.3e-2, 9.1e-3; tokens may be near-ties
    if k == 'tail':
        return {'rel': 7e-3, 'differ': 0.5}                                    # 1.7e-3
    return {'rel': 1.1e-2}                                                     # 2.7e-3


# ------------------------------------------------------------------------------------------------ the same in 64 bits

def exact(case, seed):
    new = lambda m: torch.empty(m['rows'], m['cols'], dtype=KINDS[m['dtype']][1], device=DEV)   # noqa: E731
    p = {n: t.double() if t.is_floating_point() else t for n, t in _inputs(case, seed, new).items()}
    with torch.enable_grad():
        r = {'mlp': _mlp64, 'gpt': _gpt64, 'layer': _layer64, 'prefill': _prefill64, 'decode': _decode64, 'tail': _tail64,
             'head': _head64}[case['kind']](case, p)
    lb, _ = _graph(_key(case))
    by = {m['name']: m for m in lb.metadata['buffers']}
    return {n: None if r.get(n) is None else r[n].detach().reshape(by[n]['rows'], by[n]['cols']) for n in _outputs(case)}


def _adamw(p, g, m, v, t, lr, b1, b2, eps, wd):
    m.mul_(b1).add_(g, alpha=1 - b1)
    v.mul_(b2).addcmul_(g, g, value=1 - b2)
    step = lr * (m / (1 - b1 ** t)) / ((v / (1 - b2 ** t)).sqrt() + eps)
    p.sub_(lr * wd * p + step)


def _mlp64(case, p):
    c, r = mlp.MLPConfig(widths=_widths(case), batch=case['batch'], steps=case['steps']), {}
    for i, w in enumerate(c.widths):
        n = f'm{i}.'
        ps = []
        for l, (fi, fo) in enumerate(((c.d_in, w), (w, w), (w, c.classes))):
            ps += [(f'{n}W{l}', p[f'{n}W{l}']), (f'{n}b{l}', torch.zeros(1, fo, dtype=torch.float64, device=DEV))]
        mom = {k: (torch.zeros_like(t), torch.zeros_like(t)) for k, t in ps}
        y = p[n + 'y'].reshape(-1).long()
        for s in range(c.steps):
            ts = [t.requires_grad_() for _, t in ps]
            a = p[n + 'x']
            for l in range(3):
                a = a @ ts[2 * l].T + ts[2 * l + 1]
                a = a.relu() if l < 2 else a
            loss = torch.nn.functional.cross_entropy(a, y)
            gs = torch.autograd.grad(loss, ts)
            with torch.no_grad():
                for (k, t), g in zip(ps, gs):
                    t.detach_()
                    _adamw(t, g, *mom[k], s + 1, c.lr, c.b1, c.b2, c.eps, c.wd if '.W' in k else 0.0)
        r.update(dict(ps))
        r[n + 'logits'], r['d.' + n + 'W0'] = a, gs[0]
        r[n + 'loss'] = torch.tensor([[loss.item()], [1.0 / c.batch]], dtype=torch.float64, device=DEV)
    return r


def _attend(q, k, v, B, T, H, Hkv, hd):
    """Causal grouped-query attention of [B*T, heads*hd] tensors, one sequence and head group at a time."""
    q, k, v = q.view(B, T, Hkv, H // Hkv, hd), k.view(B, T, Hkv, hd), v.view(B, T, Hkv, hd)
    mask = torch.ones(T, T, dtype=torch.bool, device=DEV).triu(1)
    rows = []
    for b in range(B):
        heads = []
        for h in range(H):
            s = (q[b, :, h // (H // Hkv), h % (H // Hkv)] @ k[b, :, h // (H // Hkv)].T / math.sqrt(hd)).masked_fill(mask, -math.inf)
            heads.append(s.softmax(-1) @ v[b, :, h // (H // Hkv)])
        rows.append(torch.cat(heads, 1))
    return torch.cat(rows)


def _gpt64(case, p):
    c = _gpt_config(case)
    N, d, bf, L = c.batch * c.T, c.d, c.dtype == 'bf16', c.layers
    z = lambda n: torch.zeros(1, n, dtype=torch.float64, device=DEV)   # noqa: E731
    names = ['wte', 'wpe']
    for l in range(L):
        names += [f'{n}.{l}' for n in ('wq', 'wk', 'wv', 'wo', 'ln1g', 'ln2g', 'w1', 'w2')]
        p.update({f'{n}.{l}': z(c.ffn if n == 'b1' else d) for n in ('bq', 'bk', 'bv', 'bo', 'ln1b', 'ln2b', 'b1', 'b2')})
        names += [f'{n}.{l}' for n in ('bq', 'bk', 'bv', 'bo', 'ln1b', 'ln2b', 'b1', 'b2')]
    p['lnfb'] = z(d)
    names += ['lnfg', 'lnfb']
    dec = {n for n in names if n.split('.')[0] in ('wte', 'wpe', 'wq', 'wk', 'wv', 'wo', 'w1', 'w2')}
    ids, tgt = p['ids'].reshape(-1).long(), p['tgt'].reshape(-1).long()
    mom = {n: (torch.zeros_like(p[n]), torch.zeros_like(p[n])) for n in names}
    norm = torch.nn.functional.layer_norm
    r = {}
    for s in range(c.steps):
        w = {n: p[n].detach().requires_grad_() for n in names}
        # GEMMs read a weight's bf16 copy: the gradient is taken at the rounded weight
        g = {n: (w[n] + (p[n].float().bfloat16().double() - p[n])) if bf and n in dec else w[n] for n in names}
        x = w['wte'][ids] + w['wpe'][torch.arange(N, device=DEV) % c.T]
        for l in range(L):
            h = norm(x, (d,), w[f'ln1g.{l}'].view(-1), w[f'ln1b.{l}'].view(-1), 1e-5)
            q, k, v = (h @ g[f'w{n}.{l}'].T + w[f'b{n}.{l}'] for n in 'qkv')
            x = x + _attend(q, k, v, c.batch, c.T, c.heads, c.heads, d // c.heads) @ g[f'wo.{l}'].T + w[f'bo.{l}']
            h = norm(x, (d,), w[f'ln2g.{l}'].view(-1), w[f'ln2b.{l}'].view(-1), 1e-5)
            x = x + torch.nn.functional.gelu(h @ g[f'w1.{l}'].T + w[f'b1.{l}'], approximate='tanh') @ g[f'w2.{l}'].T + w[f'b2.{l}']
        logits = norm(x, (d,), w['lnfg'].view(-1), w['lnfb'].view(-1), 1e-5) @ g['wte'].T
        loss = torch.nn.functional.cross_entropy(logits, tgt)
        gs = dict(zip(names, torch.autograd.grad(loss, [w[n] for n in names])))
        with torch.no_grad():
            total = math.sqrt(sum(t.square().sum().item() for t in gs.values()))
            clip = min(1.0, c.clip / (total + 1e-6))
            r = {'d.' + n: gs[n] for n in names}
            for n in names:
                p[n] = p[n].detach()
                _adamw(p[n], gs[n] * clip, *mom[n], s + 1, c.lr, c.b1, c.b2, c.eps, c.wd if n in dec else 0.0)
    f64 = lambda *v: torch.tensor(v, dtype=torch.float64, device=DEV)   # noqa: E731
    r.update(logits=logits, loss=f64(loss.item(), 1.0 / N), gscale=f64(clip, total), wte=p['wte'])
    return r


def _rms(x, g):
    return x * (x.square().mean(-1, keepdim=True) + EPS).rsqrt() * g.reshape(-1)


def _rope(x, pos, heads, hd):
    inv = THETA ** (-torch.arange(0, hd, 2, dtype=torch.float64, device=DEV) / hd)
    ang = (pos.double()[:, None] * inv)[:, None, :]
    x = x.view(-1, heads, hd)
    a, b = x[..., :hd // 2], x[..., hd // 2:]
    return torch.cat([a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos()], -1).reshape(-1, heads * hd)


def _layer64(case, p):
    c = case
    N, silu = c['T'] * c['batch'], torch.nn.functional.silu
    pos = torch.arange(N, device=DEV) % c['T']
    names = ('x', 'wq', 'wk', 'wv', 'wo', 'wg', 'wu', 'wd', 'g1', 'g2')
    w = {n: p[n].requires_grad_() for n in names}
    h = _rms(w['x'], w['g1'])
    q, k = _rope(h @ w['wq'].T, pos, c['heads'], c['hd']), _rope(h @ w['wk'].T, pos, c['kv'], c['hd'])
    xm = w['x'] + _attend(q, k, h @ w['wv'].T, c['batch'], c['T'], c['heads'], c['kv'], c['hd']) @ w['wo'].T
    h = _rms(xm, w['g2'])
    y = xm + (silu(h @ w['wg'].T) * (h @ w['wu'].T)) @ w['wd'].T
    gs = torch.autograd.grad(y, [w[n] for n in names], p['dy'])
    return {'y': y, **{('dx' if n == 'x' else 'd.' + n): g for n, g in zip(names, gs)}}


def _prefill64(case, p):
    c, r, x = case, {}, p['x']
    T, B, Hkv, hd = c['T'], c['batch'], c['kv'], c['hd']
    pos = torch.arange(T * B, device=DEV) % T
    with torch.no_grad():
        for l in range(c['layers']):
            h = _rms(x, p[f'g1.{l}'])
            q, k, v = (h @ p[f'w{n}.{l}'].T for n in 'qkv')
            q = _rope(_rms(q.view(-1, hd), p[f'qn.{l}']).view(q.shape), pos, c['heads'], hd)
            k = _rope(_rms(k.reshape(-1, hd), p[f'kn.{l}']).view(k.shape), pos, Hkv, hd)
            for n, t in (('kc', k), ('vc', v)):
                r[f'{n}.{l}'] = torch.nn.functional.pad(t.reshape(B, T, Hkv, hd).transpose(1, 2), (0, 0, 0, 64))
            x = x + _attend(q, k, v, B, T, c['heads'], Hkv, hd) @ p[f'wo.{l}'].T
            h = _rms(x, p[f'g2.{l}'])
            x = x + (torch.nn.functional.silu(h @ p[f'wg.{l}'].T) * (h @ p[f'wu.{l}'].T)) @ p[f'wd.{l}'].T
            r[f'y.{l}'] = x
    return r


def _decode64(case, p):
    c = case
    B, H, Hkv, hd, n = c['batch'], c['heads'], c['kv'], c['hd'], c['ctx']
    pos = torch.full((B,), n, device=DEV)
    with torch.no_grad():
        x = p['wte'][p['tok'].reshape(-1).long()]
        for l in range(c['layers']):
            h = _rms(x, p[f'ln1.{l}'])
            q, k, v = (h @ p[f'w{m}.{l}'].T for m in 'qkv')
            q = _rope(_rms(q.view(-1, hd), p[f'qn.{l}']).view(q.shape), pos, H, hd).view(B, Hkv, H // Hkv, hd)
            k = _rope(_rms(k.view(-1, hd), p[f'kn.{l}']).view(k.shape), pos, Hkv, hd)
            kc, vc = (p[f'{m}.{l}'].view(B, Hkv, n + 64, hd) for m in ('kc', 'vc'))
            kc[:, :, n], vc[:, :, n] = k.view(B, Hkv, hd), v.view(B, Hkv, hd)
            s = (q @ kc[:, :, :n + 1].transpose(2, 3) / math.sqrt(hd)).softmax(-1)
            x = x + (s @ vc[:, :, :n + 1]).reshape(B, H * hd) @ p[f'wo.{l}'].T
            h = _rms(x, p[f'ln2.{l}'])
            x = x + (torch.nn.functional.silu(h @ p[f'wg.{l}'].T) * (h @ p[f'wu.{l}'].T)) @ p[f'wd.{l}'].T
        last = c['layers'] - 1
        return {'x': x, 'logits': _rms(x, p['lnf']) @ p['whead'].T, f'kc.{last}': p[f'kc.{last}'], f'vc.{last}': p[f'vc.{last}']}


def _tail64(case, p):
    return {'logits': _rms(p['x'], p['gf']) @ p['whead'].T}      # the tokens are drawn, by a generator of the operator's own


def _head64(case, p):
    h, w = p['h'].requires_grad_(), p['w'].requires_grad_()
    logits = h @ w.T
    loss = torch.nn.functional.cross_entropy(logits, p['tgt'].reshape(-1).long())
    dl, dh, dw = torch.autograd.grad(loss, [logits, h, w])
    return {'loss': torch.tensor([loss.item(), 1.0 / case['rows']], dtype=torch.float64, device=DEV), 'logits': logits, 'dlogits': dl, 'dh': dh, 'd.w': dw}
