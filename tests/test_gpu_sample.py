"""GPU parity of token sampling (op 57) with the CPU oracle, whose choice is made value by value in double: the token is
the same integer. Row lengths around a tile (256 values) and around the vector length, selections of one value, some, all
but one and all of them, ties at the k-th value, rows that hold NaN and infinities, temperatures below and above 1.
"""
import numpy as np
import pytest

import oracle
from kvm_amd import bundle as bl
from kvm_amd import compiler
from kvm_amd.executor import Executor
from kvm_amd.workloads import Builder, Workload

pytestmark = pytest.mark.gpu
ROWS = 24


def _check(V, topk, temp, edit=None):
    b = Builder(3)
    b.normal('x', ROWS, V, scale=3.0)
    b.values('ctr', [7], 1)
    b.values('tok', [-1] * ROWS, ROWS)
    for r in range(0, ROWS, 6):
        b.task('sample', logits='x', out='tok', ctr='ctr' if r % 12 else None, r0=r, r1=r + 6, V=V, temp=temp, topk=topk, seed=77)
    lb = bl.load(compiler.compile_spec(Workload(b.spec()).spec))
    init = [oracle.materialize(m) for m in lb.metadata['buffers']]
    if edit:
        edit(init[0].reshape(ROWS, V))
    ref = oracle.run(lb, [x.copy() for x in init])
    ex = Executor.from_bundle(lb, buffers=init)
    ex.run()
    got = ex.read('tok')
    ex.close()
    assert np.array_equal(got, ref['buffers'][2]), (got, ref['buffers'][2])


@pytest.mark.parametrize('V,topk', [(1, 0), (3, 1), (255, 0), (256, 255), (257, 256), (1000, 1), (1000, 50), (4099, 4099), (4099, 200), (32000, 50),
                                    (32000, 0)])
def test_sample(V, topk):
    print(f'sample V {V} topk {topk}', flush=True)
    _check(V, topk, 0.8)


def test_sample_ties_and_temperature():
    print('sample ties', flush=True)
    _check(1500, 40, 1.7, lambda x: np.round(x, 0, out=x))          # a handful of distinct values: many ties at the k-th


def test_sample_nonfinite():
    """NaN is never chosen but counts among the largest keys; -inf has weight 0; a row of NaN, of -inf, one with +inf."""
    print('sample nonfinite', flush=True)

    def edit(x):
        x[:, 5::7] = np.nan
        x[:, 4::9] = -np.inf
        x[1] = np.nan
        x[2] = -np.inf
        x[3, 100] = np.inf

    _check(700, 30, 0.9, edit)
    _check(700, 0, 0.9, edit)
    _check(700, 150, 0.9, edit)
