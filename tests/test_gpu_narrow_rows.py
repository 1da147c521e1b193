"""GPU parity of the narrow-row forms: norms forward and backward (ops 35-38, 309) at d <= 512, attention delta (op 46) at
other row widths, fused cross entropy (op 127) at V <= 512, embedding backward (op 33) with repeated ids, f32 GEMM
tiles (op 34) whose rows are not whole 16-byte vectors. Row counts below, at and above a round of rows; widths at and
around 64 lanes. f32 storage, 2e-5 relative L2 (test_gpu_exec's bound for f32); bf16 delta sums f32 products of bf16 values.
"""
import pytest

import oracle
from gpu_check import compare_run
from kvm_amd import bundle as bl
from kvm_amd import compiler
from kvm_amd.executor import PATH_DYNAMIC, PATH_STATIC, Executor
from kvm_amd.workloads import Builder, Workload

pytestmark = pytest.mark.gpu


def _check(b):
    lb = bl.load(compiler.compile_spec(Workload(b.spec()).spec))
    init = [oracle.materialize(m, b.init_override.get(m['name'])) for m in lb.metadata['buffers']]
    ref = oracle.run(lb, [x.copy() for x in init])
    for path in (PATH_DYNAMIC, PATH_STATIC):
        ex = Executor.from_bundle(lb, buffers=[x.copy() for x in init], path=path)
        ex.run()
        bad = compare_run(ex, lb.metadata, ref, tol_f32=2e-5)
        ex.close()
        assert not bad, (path, bad)


@pytest.mark.parametrize('d', [3, 64, 100, 128, 129, 320, 511])
@pytest.mark.parametrize('R', [1, 5, 16, 33])
def test_norms(R, d):
    print(f'norms R {R} d {d}', flush=True)
    b = Builder(1)
    for n in ('x', 'dy', 'res', 'dxa', 'dxr'):
        b.normal(n, R, d + 1, scale=1.0)
    for n in ('g', 'be'):
        b.normal(n, 1, d, scale=1.0)
    for n in ('ln', 'rms', 'dxo'):
        b.fill(n, R, d)
    for n in ('mu', 'rs', 'rs2'):
        b.fill(n, R)
    half = (R + 1) // 2
    for r0, r1 in ((0, half), (half, R)):
        if r0 == r1:
            continue
        t = b.task('layernorm_fwd', x='x', gamma='g', beta='be', out='ln', mean='mu', rstd='rs', r0=r0, r1=r1, d=d, eps=1e-5)
        u = b.task('rmsnorm_fwd', x='x', gamma='g', out='rms', rstd='rs2', r0=r0, r1=r1, d=d, eps=1e-6)
        b.task('layernorm_bwd_dx', after=[t], x='x', dy='dy', gamma='g', mean='mu', rstd='rs', dx='dxa', r0=r0, r1=r1, d=d, acc=1)
        b.task('rmsnorm_bwd_dx', after=[u], x='x', dy='dy', gamma='g', rstd='rs2', dx='dxo', r0=r0, r1=r1, d=d, acc=0)
        b.task('layernorm_bwd_dx_res', after=[t], x='x', dy='dy', gamma='g', mean='mu', rstd='rs', dx='dxr', res='res', r0=r0, r1=r1, d=d)
    _check(b)


@pytest.mark.parametrize('dt', ['f32', 'bf16'])
@pytest.mark.parametrize('H,hd,rows', [(1, 32, (1, 15, 16, 17)), (3, 16, (5, 6)), (3, 64, (10, 11)), (1, 64, (31, 32, 33))])
def test_delta_few_pairs(dt, H, hd, rows):
    """Around the numbers of (row, head) pairs from which a task takes a lane per element."""
    print(f'delta few pairs {dt} H {H} hd {hd}', flush=True)
    for R in rows:
        b = Builder(9)
        for n in ('o', 'do'):
            b.normal(n, R, H * hd, dt, scale=1.0)
        b.fill('delta', R * H)
        b.task('attn_bwd_delta', o='o', do='do', delta='delta', r0=0, r1=R, T=R, H=H, hd=hd)
        _check(b)


@pytest.mark.parametrize('dt', ['f32', 'bf16'])
@pytest.mark.parametrize('H,hd,T,B', [(1, 8, 5, 1), (4, 32, 7, 3), (3, 64, 20, 2), (5, 16, 33, 1)])
def test_delta(dt, H, hd, T, B):
    print(f'delta {dt} H {H} hd {hd} T {T}', flush=True)
    b = Builder(2)
    for n in ('o', 'do'):
        b.normal(n, B * T, H * hd, dt, scale=1.0)
    b.fill('delta', B * H * T)
    for r0 in range(0, B * T, 9):
        b.task('attn_bwd_delta', o='o', do='do', delta='delta', r0=r0, r1=min(B * T, r0 + 9), T=T, H=H, hd=hd)
    _check(b)


@pytest.mark.parametrize('V', [8, 40, 256, 504, 512])
@pytest.mark.parametrize('R', [1, 4, 19])
def test_cross_entropy(R, V):
    print(f'ce R {R} V {V}', flush=True)
    b = Builder(3)
    b.normal('l', R, V, scale=4.0)
    b.values('t', [(7 * i + 3) % V if i % 5 != 2 else -1 for i in range(R)], R)
    for n in ('rl', 'ls'):
        b.fill(n, R)
    b.fill('dl', R, V, value=9.0)
    b.task('softmax_ce_fused', logits='l', tgt='t', rowloss='rl', lse='ls', dlogits='dl', r0=0, r1=R, V=V, ignore=-1, N=R, scale=1.0)
    _check(b)


@pytest.mark.parametrize('N,V,d', [(1, 4, 64), (7, 3, 100), (300, 11, 260), (64, 64, 300)])
def test_embedding_bwd_repeats(N, V, d):
    print(f'embedding_bwd N {N} V {V} d {d}', flush=True)
    for acc in (0, 1):
        b = Builder(4)
        b.values('ids', [(i * i + i // 3) % V for i in range(N)], N)
        b.normal('g', N, d, scale=1.0)
        b.normal('t', V, d, scale=1.0)
        for v0 in range(0, V, 5):
            b.task('embedding_bwd', ids='ids', dout='g', dtab='t', N=N, mod=0, v0=v0, v1=min(V, v0 + 5), d=d, acc=acc)
        _check(b)


@pytest.mark.parametrize('flags', [0, 1, 2, 3, 2 | 8, 4])
@pytest.mark.parametrize('M,N,K', [(1, 1, 1), (64, 10, 33), (70, 65, 10), (10, 130, 50), (130, 7, 257)])
def test_f32_tile_unaligned_rows(M, N, K, flags):
    print(f'f32 tile rows {M}x{N}x{K} flags {flags}', flush=True)
    b = Builder(5)
    ta, tb = flags & 1, flags & 2
    b.normal('a', K if ta else M, M if ta else K, scale=1.0)
    b.normal('b', N if tb else K, K if tb else N, scale=1.0)
    b.normal('c', M, N, scale=1.0)
    b.normal('bias', 1, N, scale=1.0)
    for m0 in range(0, M, 64):
        for n0 in range(0, N, 64):
            b.task('matmul_tile', a='a', b='b', out='c', bias='bias', res=None, pre=None, m0=m0, n0=n0, M=M, N=N, K=K, flags=flags, alpha=0.5)
    _check(b)
