"""GPU parity of the vectorised elementwise and per-head operators (ops 40-44, 49, 98, 99, 300) with the CPU oracle: ranges
that start and end off the vector grid, f32, bf16 and mixed storage, accumulation, in place, head sizes with and without
whole vectors, rows with padding columns, appends at a length.

Tolerances: f32 outputs 1e-6 relative L2 for arithmetic alone, 2e-6 where an exponential, a sine or a root is in it (the
oracle works in double; a few f32 roundings of 6e-8 each), bf16 outputs 4e-3 (half an ulp is 2e-3). RoPE angles are f32
products p * theta^(-2i/hd): at position p one f32 ulp of the angle is p * 6e-8, so T stays below 64 here (4e-6).
"""
import numpy as np
import pytest

import oracle
from gpu_check import compare_run
from kvm_amd import bundle as bl
from kvm_amd import compiler
from kvm_amd.executor import Executor
from kvm_amd.workloads import Builder, Workload

pytestmark = pytest.mark.gpu


def _check(b, tol_f32, edit=None):
    lb = bl.load(compiler.compile_spec(Workload(b.spec()).spec))
    init = [oracle.materialize(m, b.init_override.get(m['name'])) for m in lb.metadata['buffers']]
    if edit:
        edit({m['name']: x for m, x in zip(lb.metadata['buffers'], init)})
    ref = oracle.run(lb, [x.copy() for x in init])
    ex = Executor.from_bundle(lb, buffers=[x.copy() for x in init])
    ex.run()
    bad = compare_run(ex, lb.metadata, ref, tol_f32=tol_f32, tol_bf16=4e-3)
    ex.close()
    assert not bad, bad


RANGES = [(0, 8), (3, 5), (1, 4099), (8, 9000), (7, 8192), (0, 40000)]


@pytest.mark.parametrize('dts', [('f32', 'f32', 'f32'), ('bf16', 'bf16', 'bf16'), ('f32', 'bf16', 'f32'), ('bf16', 'f32', 'bf16')])
@pytest.mark.parametrize('e0,e1', RANGES)
def test_flat(dts, e0, e1):
    print(f'flat {dts} {e0} {e1}', flush=True)
    for op, names in (('residual_add', ('a', 'b', 'out')), ('silu_mul_fwd', ('gate', 'up', 'out')), ('gelu_bwd', ('x', 'dy', 'dx'))):
        for acc in ((0, 1) if op == 'gelu_bwd' else (None,)):
            b = Builder(1)
            for n, dt in zip(names, dts):
                b.normal(n, 1, e1 + 5, dt, scale=3.0)
            kw = {} if acc is None else {'acc': acc}
            b.task(op, e0=e0, e1=e1, **{n: n for n in names}, **kw)
            _check(b, 2e-6)


@pytest.mark.parametrize('e0,e1', RANGES)
def test_flat_f32(e0, e1):
    print(f'flat f32 {e0} {e1}', flush=True)
    for acc in (0, 1):
        b = Builder(2)
        for n in ('gate', 'up', 'dy', 'dgate', 'dup', 'x'):
            b.normal(n, 1, e1 + 5, scale=3.0)
        b.fill('y', 1, e1 + 5)
        t = b.task('silu_mul_bwd', gate='gate', up='up', dy='dy', dgate='dgate', dup='dup', e0=e0, e1=e1, acc=acc)
        b.task('gelu_fwd', x='x', out='y', e0=e0, e1=e1)
        b.task('silu_mul_fwd', after=[t], gate='gate', up='up', out='gate', e0=e0, e1=e1)     # in place
        _check(b, 2e-6)


def test_silu_extremes():
    """Saturated, tiny and non-finite gates: sigmoid's ends, and NaN only where the product makes one."""
    print('silu extremes', flush=True)
    b = Builder(3)
    for n in ('gate', 'up'):
        b.normal(n, 1, 64, scale=1.0)
    b.fill('out', 1, 64)
    b.task('silu_mul_fwd', gate='gate', up='up', out='out', e0=0, e1=64)

    def edit(x):
        x['gate'][:12] = [0.0, -0.0, 1e-38, -1e-38, 80.0, -80.0, 200.0, -86.0, np.inf, np.nan, 17.0, -17.0]
        x['up'][:12] = 1.0

    lb = bl.load(compiler.compile_spec(Workload(b.spec()).spec))
    init = [oracle.materialize(m) for m in lb.metadata['buffers']]
    edit({m['name']: v for m, v in zip(lb.metadata['buffers'], init)})
    ref = oracle.run(lb, [v.copy() for v in init])['buffers'][2]
    ex = Executor.from_bundle(lb, buffers=[v.copy() for v in init])
    ex.run()
    got = ex.read('out')
    ex.close()
    assert np.allclose(got, ref, rtol=1e-6, atol=1e-36, equal_nan=True), (got[:12], ref[:12])


@pytest.mark.parametrize('dti,dto', [('f32', 'f32'), ('bf16', 'bf16'), ('f32', 'bf16')])
@pytest.mark.parametrize('H,hd,R,pad', [(1, 16, 3, 0), (3, 64, 37, 8), (4, 128, 50, 0), (2, 40, 9, 0), (2, 12, 5, 0), (5, 8, 300, 0)])
def test_rope_head_norm(dti, dto, H, hd, R, pad):
    print(f'rope {dti} {dto} H {H} hd {hd} R {R}', flush=True)
    b = Builder(4)
    b.normal('x', R, H * hd + pad, dti, scale=1.0)
    b.normal('z', R, H * hd + pad, dti, scale=1.0)
    b.normal('g', 1, hd, scale=1.0)
    for n in ('f', 'b', 'n'):
        b.fill(n, R, H * hd, dto)
    b.values('pos', [5], 1)
    for r0 in range(0, R, 7):
        r1 = min(R, r0 + 7)
        b.task('rope_fwd', x='x', out='f', pos='pos', r0=r0, r1=r1, T=23, H=H, hd=hd, theta=1e4)
        b.task('rope_bwd', x='x', out='b', pos=None, r0=r0, r1=r1, T=23, H=H, hd=hd, theta=1e4)
        b.task('head_rmsnorm', x='x', gamma='g', out='n', r0=r0, r1=r1, H=H, hd=hd, eps=1e-6)
    b.task('rope_fwd', x='z', out='z', pos=None, r0=0, r1=R, T=50, H=H, hd=hd, theta=1e4)        # in place, all rows
    _check(b, 4e-6)


@pytest.mark.parametrize('dtn,dtc', [('f32', 'f32'), ('bf16', 'bf16'), ('f32', 'bf16')])
@pytest.mark.parametrize('B,nn,Hkv,hd', [(1, 1, 1, 8), (2, 37, 3, 64), (1, 130, 2, 128), (2, 5, 2, 20), (70, 1, 1, 64), (9, 3, 5, 56)])
def test_kv_append(dtn, dtc, B, nn, Hkv, hd):
    print(f'kv_append {dtn} {dtc} B {B} n {nn} H {Hkv} hd {hd}', flush=True)
    Tmax = nn + 9
    b = Builder(6)
    for n in ('k', 'v'):
        b.normal(n, B * nn, Hkv * hd, dtn, scale=1.0)
        b.normal(n + 'c', B * Hkv * Tmax, hd, dtc, scale=1.0)
    b.values('lens', [4 + i % 6 for i in range(B)], B)
    b.task('kv_append', knew='k', vnew='v', kc='kc', vc='vc', lens='lens', b0=0, b1=B, n_new=nn, Hkv=Hkv, hd=hd, Tmax=Tmax)
    _check(b, 0.0 if dtn == dtc else 1e-9)
