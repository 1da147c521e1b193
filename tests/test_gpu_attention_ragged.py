"""GPU parity of causal attention (ops 45-48) where the MFMA bodies mask ragged rows and keep fp32 probabilities: T not
a multiple of 64 (below, at and above a block's and a task's edge), and the backward at hd 128; bf16 and f32 storage.

Tolerances: on bf16 storage the probabilities stay f32 values through the second product, so only the stored values are
rounded to bf16: 4e-3 relative L2 (half an ulp is 2^-9 relative, the L2 mean of it below 2e-3). delta is
computed from the bf16 o (one rounding per element, averaged over a row's products): 1e-2. f32 storage: 2e-5.
"""
import numpy as np
import pytest

import oracle
from gpu_check import compare_run
from kvm_amd import bundle as bl
from kvm_amd import compiler
from kvm_amd.executor import Executor
from test_gpu_attention import _attn_graph

pytestmark = pytest.mark.gpu


def _run(w, poke=None):
    lb = bl.load(compiler.compile_spec(w.spec))
    init = [oracle.materialize(m, w.init_override.get(m['name'])) for m in lb.metadata['buffers']]
    names = [m['name'] for m in lb.metadata['buffers']]
    if poke:
        poke(init, names)
    ref = oracle.run(lb, [x.copy() for x in init])
    ex = Executor.from_bundle(lb, buffers=init)
    ex.run()
    return lb, names, ref, ex


@pytest.mark.parametrize('dt', ['bf16', 'f32'])
@pytest.mark.parametrize('hd,H,Hkv,T', [(64, 2, 1, 1), (64, 2, 1, 17), (64, 2, 2, 63), (32, 4, 2, 65), (64, 2, 2, 129), (128, 4, 1, 127), (128, 2, 2, 193),
                                        (128, 4, 2, 256), (64, 4, 1, 330)])
def test_attention_ragged(dt, hd, H, Hkv, T):
    print(f'attn ragged {dt} hd {hd} H {H} Hkv {Hkv} T {T}', flush=True)
    # one token attends to itself alone: dP - delta, and with it dQ and dK, is nothing but the rounding of o
    lb, names, ref, ex = _run(_attn_graph(2, H, Hkv, T, hd, ('fwd', 'bwd') if T > 1 else ('fwd',), dt=dt))
    skip = ('delta',) if dt == 'bf16' and T > 1 else ()
    bad = compare_run(ex, lb.metadata, ref, tol_f32=2e-5, tol_bf16=4e-3, skip=skip)
    for n in skip:
        i = names.index(n)
        bad += compare_run(ex, {'buffers': [lb.metadata['buffers'][i]]}, {'buffers': [ref['buffers'][i]]}, tol_f32=1e-2)
    ex.close()
    assert not bad, bad


@pytest.mark.parametrize('dt', ['bf16', 'f32'])
@pytest.mark.parametrize('hd,T,value', [(64, 100, np.inf), (128, 150, np.nan)])
def test_attention_masked_nonfinite(dt, hd, T, value):
    """A non-finite value in the last key's row reaches the outputs that see that key, and no others: a masked key's
    weight of 0 must not meet it in a product."""
    print(f'attn nonfinite {dt} hd {hd} T {T} {value}', flush=True)

    def poke(init, names):
        v = init[names.index('v')].reshape(T, -1)
        v[T - 1, 3] = value

    lb, names, ref, ex = _run(_attn_graph(1, 2, 2, T, hd, ('fwd', 'bwd'), dt=dt), poke)
    for m, want in zip(lb.metadata['buffers'], ref['buffers']):
        got, want = np.asarray(ex.read(m['name']), np.float64), np.asarray(want, np.float64)
        fin = np.isfinite(want)
        assert np.array_equal(np.isfinite(got), fin), m['name']
        err = np.linalg.norm(got[fin] - want[fin]) / max(np.linalg.norm(want[fin]), 1e-30)
        assert err <= (1e-2 if dt == 'bf16' else 2e-5), (m['name'], err)
    assert np.isfinite(ex.read('o').reshape(T, -1)[:T - 1]).all() and np.isfinite(ex.read('dq').reshape(T, -1)[:T - 1]).all()
    ex.close()


def _bf16(x):
    u = np.asarray(x, np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7fff + ((u >> 16) & 1)) & 0xffff0000).astype(np.uint32).view(np.float32)


def _cancelling(rng, w, n):
    """n columns c of bf16 values with sum(w c) below 2^-17 of sum(w |c|)."""
    w, cols = np.asarray(w, np.float64), []
    while len(cols) < n:
        c = _bf16(rng.normal(size=(20000, len(w))) * 8).astype(np.float64)
        c[:, -1] = _bf16(-(c[:, :-1] @ w[:-1]) / w[-1])
        cols += list(c[np.abs(c @ w) < 2.0 ** -17 * (np.abs(c) @ w)])
    return np.array(cols[:n]).T


def _two_pieces(w):
    """What bf16(w) + bf16(w - bf16(w)) leaves of f32 weights."""
    w = np.asarray(w, np.float32)
    hi = _bf16(w)
    return (w - hi - _bf16(w - hi)).astype(np.float64)


@pytest.mark.parametrize('hd', [64, 128])
def test_attention_f32_weights(hd):
    """Values whose weighted sum all but vanishes (o of the last query, dv of the first key) show the weights' own error:
    a few of 2^-24 (the score's sum, the exponential), where weights of 16 significant bits would leave 2^-18 of the sum of
    magnitudes. The bound, 6e-7 of it, lies between: scores of a few units carry ~1.5e-7, two bf16 pieces of the weights
    chosen here at least 1.8e-6."""
    T, H = 3, 6
    rng = np.random.default_rng(hd)
    q, k, v, do = (np.zeros((T, H * hd), np.float32) for _ in range(4))
    want, size, left = {}, {}, {'o': [], 'dv': []}
    for h in range(H):
        s = slice(h * hd, (h + 1) * hd)
        best = None
        for _ in range(400):
            qq, kk = _bf16(rng.normal(size=(T, hd))), _bf16(rng.normal(size=(T, hd)))
            sc = np.where(np.tri(T) > 0, qq.astype(np.float64) @ kk.astype(np.float64).T / np.sqrt(hd), -np.inf)
            e = np.exp(sc - sc.max(1, keepdims=True))
            P = e / e.sum(1, keepdims=True)
            r = min(np.abs(_two_pieces(e[-1])).sum() / e[-1].sum(), np.abs(_two_pieces(P[:, 0])).sum() / P[:, 0].sum())
            if best is None or r > best[0]:
                best = (r, qq, kk, e[-1], P)
        _, q[:, s], k[:, s], e, P = best
        v[:, s], do[:, s] = _cancelling(rng, e, hd), _cancelling(rng, P[:, 0], hd)
        for n, w, c, by in (('o', e, v[:, s], e.sum()), ('dv', P[:, 0], do[:, s], 1.0)):
            c = c.astype(np.float64)
            want[n, h], size[n, h] = w @ c / by, w @ np.abs(c) / by
            left[n].append(_two_pieces(w) @ c / by / size[n, h])
    print(f'attn f32 weights hd {hd}', flush=True)

    def poke(init, names):
        for n, x in (('q', q), ('k', k), ('v', v), ('do', do)):
            init[names.index(n)].reshape(T, -1)[:] = x

    _, _, _, ex = _run(_attn_graph(1, H, H, T, hd, ('fwd', 'bwd'), dt='bf16'), poke)
    got = {'o': ex.read('o').reshape(T, -1)[-1], 'dv': ex.read('dv').reshape(T, -1)[0]}
    ex.close()
    for n in got:
        err = np.concatenate([(got[n][h * hd:(h + 1) * hd] - want[n, h]) / size[n, h] for h in range(H)])
        rms = lambda x: float(np.sqrt(np.mean(np.square(x))))   # noqa: E731
        print(n, rms(err), rms(np.concatenate(left[n])), flush=True)
        assert rms(np.concatenate(left[n])) > 1.8e-6
        assert rms(err) < 6e-7, (n, rms(err))
