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


def _check(V, topk, temp, edit=None, rows=ROWS):
    b = Builder(3)
    b.normal('x', rows, V, scale=3.0)
    b.values('ctr', [7], 1)
    b.values('tok', [-1] * rows, rows)
    for r in range(0, rows, 6):
        b.task('sample', logits='x', out='tok', ctr='ctr' if r % 12 else None, r0=r, r1=min(rows, r + 6), V=V, temp=temp, topk=topk, seed=77)
    lb = bl.load(compiler.compile_spec(Workload(b.spec()).spec))
    init = [oracle.materialize(m) for m in lb.metadata['buffers']]
    if edit:
        edit(init[0].reshape(rows, V))
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


@pytest.mark.parametrize('V,topk', [(2097152, 0), (2097152 + 300, 0), (4194304 + 700, 0), (4194304 + 700, 50)])
def test_sample_long_rows(V, topk):
    """More tiles than the kept sums: one, two and three tiles to a sum, the last sum of one or two tiles, one of them ragged."""
    print(f'sample long rows V {V} topk {topk}', flush=True)
    _check(V, topk, 0.8, rows=3)
