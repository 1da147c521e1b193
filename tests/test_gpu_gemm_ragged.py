"""GPU parity of the GEMM tile operators on ragged shapes whose rows are whole 16-byte vectors, which take the staged
vector loads with clamped edges: bf16 operands (direct to LDS), f32 and mixed operands of the bf16 tiles (through
registers), f32 tiles (op 34). Edges in M and N at and around a tile's and a vector's, K below, at and above a slab's
multiple, odd K; every orientation; what lies past M, N and K in wider buffers is NaN and must not be read into results.

Tolerances as in test_gpu_gemm: f32 outputs 2e-5, bf16 outputs 4e-3 (relative L2).
"""
import numpy as np
import pytest

import oracle
from gpu_check import compare_run
from kvm_amd import bundle as bl
from kvm_amd import compiler, executor
from kvm_amd.executor import PATH_DYNAMIC, PATH_STATIC, Executor
from kvm_amd.workloads import Builder, Workload

pytestmark = pytest.mark.gpu


def _up(n, m):
    return -(-n // m) * m


def _check(op, tiles, fl, M, N, K, flags, adt, bdt, odt, pad=0):
    """pad: extra columns (a multiple of 8) of the operands, NaN, like the columns that round rows up to vectors."""
    b = Builder(5)
    ta, tb = flags & 1, flags & 2
    shape = {'A': (K, M) if ta else (M, K), 'B': (N, K) if tb else (K, N)}
    for n, dt in (('A', adt), ('B', bdt)):
        r, c = shape[n]
        b.normal(n, r + (3 if pad else 0), _up(c, 8 if dt == 'bf16' else 4) + pad, dt, scale=1.0)
    b.normal('C', M, _up(N, 4), odt, scale=1.0)
    b.normal('bias', 1, N, 'f32', scale=1.0)
    for m0 in range(0, M, tiles[0]):
        for n0 in range(0, N, tiles[1]):
            b.task(op, a='A', b='B', out='C', bias='bias', res=None, pre=None, m0=m0, n0=n0, M=M, N=N, K=K, flags=flags | fl, alpha=0.5)
    w = Workload(b.spec(), b.init_override)
    lb = bl.load(compiler.compile_spec(w.spec))
    init = [oracle.materialize(m, w.init_override.get(m['name'])) for m in lb.metadata['buffers']]
    for m, x in zip(lb.metadata['buffers'], init):
        if m['name'] in shape:
            r, c = shape[m['name']]
            v = x.reshape(m['rows'], m['cols'])
            v[:, c:] = np.nan
            v[r:] = np.nan
    ref = oracle.run(lb, [x.copy() for x in init])
    for path in (PATH_DYNAMIC, PATH_STATIC):
        ex = Executor.from_bundle(lb, buffers=[x.copy() for x in init], path=path)
        ex.run()
        names = [m['name'] for m in lb.metadata['buffers']]
        i = names.index('C')
        bad = compare_run(ex, {'buffers': [lb.metadata['buffers'][i]]}, {'buffers': [ref['buffers'][i]]}, tol_f32=2e-5, tol_bf16=4e-3)
        assert np.isfinite(ex.read('C')).all()
        ex.close()
        assert not bad, (path, bad)


@pytest.mark.parametrize('flags', [0, 1, 2, 3])
@pytest.mark.parametrize('op,tiles,fl', [('matmul_mma_bf16', (128, 256), 0), ('matmul_tile_bf16', (128, 128), 32), ('matmul_tile_bf16', (64, 64), 0)])
@pytest.mark.parametrize('M,N,K', [(1, 8, 1), (127, 250, 31), (129, 257, 33), (200, 304, 104), (136, 264, 67), (64, 64, 500)])
def test_bf16_ragged(op, tiles, fl, M, N, K, flags):
    print(f'{op} {tiles} {M}x{N}x{K} flags {flags}', flush=True)
    _check(op, tiles, fl, M, N, K, flags, 'bf16', 'bf16', 'bf16', pad=8 if K % 2 else 0)


@pytest.mark.parametrize('flags', [0, 1, 2, 3])
@pytest.mark.parametrize('adt,bdt', [('f32', 'f32'), ('f32', 'bf16'), ('bf16', 'f32')])
@pytest.mark.parametrize('M,N,K', [(128, 256, 128), (132, 260, 68), (130, 300, 97), (60, 68, 64), (4, 12, 4)])
def test_bf16_tiles_f32_operands(adt, bdt, M, N, K, flags):
    print(f'f32 operands {adt} {bdt} {M}x{N}x{K} flags {flags}', flush=True)
    _check('matmul_mma_bf16', (128, 256), 0, M, N, K, flags, adt, bdt, 'f32', pad=8 if K % 2 else 0)
    _check('matmul_tile_bf16', (128, 128), 32, M, N, K, flags, adt, bdt, 'bf16')


@pytest.mark.parametrize('flags', [0, 1, 2, 3])
@pytest.mark.parametrize('tiles,fl', [((64, 64), 0), ((128, 128), 32), ((256, 128), 64)])
@pytest.mark.parametrize('M,N,K', [(1, 4, 3), (63, 60, 15), (130, 68, 17), (260, 132, 40), (257, 129, 101)])
def test_f32_ragged(tiles, fl, M, N, K, flags):
    print(f'f32 tile {tiles} {M}x{N}x{K} flags {flags}', flush=True)
    _check('matmul_tile', tiles, fl, M, N, K, flags, 'f32', 'f32', 'f32', pad=8 if K % 2 else 0)


@pytest.mark.parametrize('tiles,fl', [((64, 64), 0), ((128, 128), 32), ((256, 128), 64)])
@pytest.mark.parametrize('M,N,K', [(1, 4, 3), (64, 64, 32), (130, 68, 17), (257, 129, 101), (256, 256, 64)])
def test_swiglu_tiles(tiles, fl, M, N, K):
    """Ops 120 (both orientations of B) and 121: the tile, then silu of the gate times it, or the gate's and up's gradients."""
    print(f'swiglu tile {tiles} {M}x{N}x{K}', flush=True)
    for bwd, flags in ((0, 2), (0, 0), (1, 0), (1, 3)):
        b = Builder(8)
        ta, tb = flags & 1, flags & 2
        b.normal('a', K if ta else M, M if ta else K, scale=1.0)
        b.normal('b', N if tb else K, K if tb else N, scale=1.0)
        for n in ('gate', 'up', 'o1', 'o2'):
            b.normal(n, M, N, scale=1.0)
        for m0 in range(0, M, tiles[0]):
            for n0 in range(0, N, tiles[1]):
                kw = dict(a='a', b='b', gate='gate', up='up', m0=m0, n0=n0, M=M, N=N, K=K, flags=flags | fl, alpha=0.5)
                if bwd:
                    b.task('matmul_tile_silu_mul_bwd', dgate='o1', dup='o2', **kw)
                else:
                    b.task('matmul_tile_silu_mul', out='o1', **kw)
        lb = bl.load(compiler.compile_spec(Workload(b.spec()).spec))
        init = [oracle.materialize(m) for m in lb.metadata['buffers']]
        ref = oracle.run(lb, [x.copy() for x in init])
        for path in (PATH_DYNAMIC, PATH_STATIC):
            ex = Executor.from_bundle(lb, buffers=[x.copy() for x in init], path=path)
            ex.run()
            bad = compare_run(ex, lb.metadata, ref, tol_f32=2e-5)
            ex.close()
            assert not bad, (bwd, flags, path, bad)


def _splitk(M, N, bounds, flags, adt, bdt, TM=128):
    """Op 302 over the K ranges between `bounds` (the last one ends with the operands), and the sum of the parts."""
    b = Builder(6)
    ta, tb, K, S = flags & 1, flags & 2, bounds[-1], len(bounds) - 1
    b.normal('A', K if ta else M, M if ta else K, adt, scale=1.0)
    b.normal('B', N if tb else K, K if tb else N, bdt, scale=1.0)
    b.fill('P', S * M, N, 'f32')
    b.fill('C', M, N, 'f32')
    ts = [b.task('matmul_mma_bf16_kr', a='A', b='B', out='P', bias=None, res=None, pre=None, m0=m0, n0=n0, M=M, N=N, K=bounds[s + 1] - bounds[s],
                 flags=flags | (64 if TM == 256 else 0), alpha=1.0, k0=bounds[s], om0=s * M)
          for s in range(S) for m0 in range(0, M, TM) for n0 in range(0, N, 256)]
    for r0 in range(0, M, 64):
        b.task('splitk_reduce', after=ts, part='P', out='C', M=M, N=N, S=S, r0=r0, r1=min(M, r0 + 64))
    lb = bl.load(compiler.compile_spec(Workload(b.spec(), b.init_override).spec))
    init = [oracle.materialize(m) for m in lb.metadata['buffers']]
    ref = oracle.run(lb, [x.copy() for x in init])
    for path in (PATH_DYNAMIC, PATH_STATIC):
        ex = Executor.from_bundle(lb, buffers=[x.copy() for x in init], path=path)
        ex.run()
        bad = compare_run(ex, lb.metadata, ref, tol_f32=2e-5)
        ex.close()
        assert not bad, (path, bad)


@pytest.mark.parametrize('flags', [0, 1, 2, 3])
@pytest.mark.parametrize('adt,bdt', [('bf16', 'bf16'), ('f32', 'bf16'), ('bf16', 'f32')])
@pytest.mark.parametrize('bounds', [(0, 32, 72), (0, 256, 416), (0, 200, 1000, 2000)])
def test_splitk_ragged_ranges(bounds, adt, bdt, flags):
    """The last range ends at the operands' last column, no whole number of slabs on."""
    print(f'split-K ranges {bounds} {adt} {bdt} flags {flags}', flush=True)
    _splitk(128, 264, bounds, flags, adt, bdt)
    _splitk(256, 256, bounds, flags, adt, bdt, TM=256)


@pytest.mark.parametrize('flags', [0, 1, 2, 3])
@pytest.mark.parametrize('adt,bdt', [('bf16', 'bf16'), ('f32', 'bf16')])
@pytest.mark.parametrize('bounds', [(0, 4, 72), (0, 33, 104)])
def test_splitk_unaligned_ranges(bounds, adt, bdt, flags):
    """A k-contiguous operand's range that starts between vectors: no 16-byte loads."""
    print(f'split-K unaligned ranges {bounds} {adt} {bdt} flags {flags}', flush=True)
    _splitk(128, 264, bounds, flags, adt, bdt)


@pytest.mark.parametrize('op,tiles,fl,dt', [('matmul_mma_bf16', (128, 256), 2, 'bf16'), ('matmul_tile_bf16', (64, 64), 1, 'bf16'), ('matmul_mma_bf16', (128, 256), 2, 'f32'),
                                            ('matmul_tile', (64, 64), 2, 'f32'), ('matmul_tile', (128, 128), 32, 'f32'), ('matmul_tile_silu_mul', (64, 64), 2, 'f32'),
                                            ('matmul_tile_silu_mul_bwd', (128, 128), 32, 'f32')])
def test_operands_at_any_element(op, tiles, fl, dt):
    """A caller's own buffers (kvm_run_noalloc) that start one element past a vector; the SwiGLU tiles' all of them."""
    print(f'{op} {tiles} {dt} at one element past a vector', flush=True)
    M, N, K = 136, 264, 72
    b = Builder(9)
    ta, tb = fl & 1, fl & 2
    b.normal('a', K if ta else M, M if ta else K, dt, scale=1.0)
    b.normal('b', N if tb else K, K if tb else N, dt, scale=1.0)
    for n in ('gate', 'up', 'o1', 'o2'):
        b.normal(n, M, N, scale=1.0)
    for m0 in range(0, M, tiles[0]):
        for n0 in range(0, N, tiles[1]):
            kw = dict(a='a', b='b', m0=m0, n0=n0, M=M, N=N, K=K, flags=fl, alpha=0.5)
            if op.endswith('_bwd'):
                b.task(op, gate='gate', up='up', dgate='o1', dup='o2', **kw)
            elif op.endswith('_mul'):
                b.task(op, gate='gate', up='up', out='o1', **kw)
            else:
                b.task(op, out='o1', bias=None, res=None, pre=None, **kw)
    lb = bl.load(compiler.compile_spec(Workload(b.spec(), b.init_override).spec))
    init = [oracle.materialize(m) for m in lb.metadata['buffers']]
    ref = oracle.run(lb, [x.copy() for x in init])
    mem, ptrs, off = Executor(num_vars=1, trace=False), [], []
    for m, x in zip(lb.metadata['buffers'], init):
        off.append(1 if 'silu' in op or m['name'] in ('a', 'b') else 0)
        mem.add_buffer(m['name'], 1, x.size + 1, m['dtype'], data=np.concatenate([np.zeros(off[-1], np.float32), x.ravel(), np.zeros(1 - off[-1], np.float32)]))
        ptrs.append(mem.device_ptr(m['name']) + off[-1] * (2 if m['dtype'] == bl.DT_BF16 else 4))
    res, _ = executor.run_noalloc(lb, ptrs, [0])
    assert res['rc'] == 0 and res['done'] == lb.ntasks, res
    for m, want, o in zip(lb.metadata['buffers'], ref['buffers'], off):
        got = np.asarray(mem.read(m['name']), np.float64)[o:o + want.size]
        err = np.linalg.norm(got - want.ravel()) / max(np.linalg.norm(want), 1e-30)
        assert err <= 2e-5, (m['name'], err)
    mem.close()
