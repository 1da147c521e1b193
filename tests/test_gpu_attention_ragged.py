"""GPU parity of causal attention (ops 45-48) where the MFMA bodies mask ragged rows and keep fp32 probabilities: T not
a multiple of 64 (below, at and above a block's and a task's edge), and the backward at hd 128; bf16 and f32 storage.

Tolerances: on bf16 storage the probabilities keep ~2^-17 through the second product (bf16 + remainder), so only the
stored values are rounded to bf16: 4e-3 relative L2 (half an ulp is 2^-9 relative, the L2 mean of it below 2e-3). delta is
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
