"""The byte range that a GEMM tile's buffer descriptor covers (common.h: skip_k, bytes_from_row), on the host: for every
form of a K range (op 302) the descriptor of any tile row starts in the operand and ends where the operand ends, so that a
slab load that runs past a ragged K returns 0 instead of leaving the buffer, and every element of the range is inside. And the rules that choose
the vector loads (ops_gemm.h).
"""
import shutil
import subprocess

import pytest

from kvm_amd import build as kb

PROGRAM = r'''
#include "common.h"
#include <cstdio>
int main() {
  long long bad = 0, forms = 0;
  char* const base = (char*)(uintptr_t)0x10000000;
  for (int es : {2, 4})
    for (int kc : {0, 1})
      for (int k : {1, 31, 40, 72, 160, 416, 2000})               // the operand's whole K
        for (int n : {1, 127, 128, 300})                          // its tile rows (M or N)
          for (int pad : {0, 8, 24})                              // columns past them
            for (int k0 : {0, 1, 4, 8, 31, 32, 256, 1000}) {
              if (k0 >= k) continue;
              const int rows = kc ? n : k, cols = (kc ? k : n) + pad, K = k - k0;
              View v{base, rows, cols, es == 2 ? 2 : 0};
              const char* end = base + (long long)rows * cols * es;
              skip_k(v, kc, k0);
              ++forms;
              if (kc) {
                for (int r0 = 0; r0 < n; r0 += 64) {
                  const char* p = (const char*)v.p + (long long)r0 * cols * es;
                  const long long bytes = bytes_from_row(v, r0);
                  bad += p < base || p + bytes != end || ((long long)(n - 1 - r0) * cols + K) * es > bytes;
                }
              } else {                                            // the whole rest of the operand
                bad += (const char*)v.p + (long long)v.rows * v.cols * es != end || v.rows < K;
              }
            }
  printf("%lld forms, %lld outside\n", forms, bad);
  return bad != 0;
}
'''


def _host_run(tmp_path, program):
    if not shutil.which(kb.HIPCC) and not kb.Path(kb.HIPCC).exists():
        pytest.skip('hipcc not available')
    src, exe = tmp_path / 'ranges.hip', tmp_path / 'ranges'
    src.write_text(program)
    r = subprocess.run([kb.HIPCC, *kb.FLAGS, '-O1', f'-I{kb.CSRC}', str(src), '-o', str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


def test_descriptor_ends_with_the_operand(tmp_path):
    _host_run(tmp_path, PROGRAM)


ALIGNED = r'''
#include "ops_gemm.h"
#include <cstdio>
int main() {
  using namespace kvm;
  long long bad = 0, forms = 0;
  char* const base = (char*)(uintptr_t)0x10000000;
  for (int dtype : {2, 0})
    for (int kc : {0, 1})
      for (int cols : {8, 72, 300, 304, 512})
        for (int off : {0, 1, 3, 4, 8, 12})                       // elements into a caller's allocation
          for (int k0 : {0, 1, 4, 8, 33, 40}) {                   // a K range (op 302)
            View v{base + off * (dtype == 2 ? 2 : 4), 300, cols, dtype};
            skip_k(v, kc, k0);
            const bool aligned = ((uintptr_t)v.p & 15) == 0;      // with whole vectors in a row: every row of the tile
            bad += gemm_fast_operand(v, kc, 0, 128, 64) != (aligned && dtype == 2 && cols % 8 == 0);
            bad += gemm_vec_operand(v, kc, 0, 128, 64) != (aligned && cols % (dtype == 2 ? 8 : 4) == 0);
            bad += gemm_f32_fast_operand(v, kc, 0, 128, 64) != (aligned && dtype == 0 && cols % 4 == 0);
            bad += gemm_f32_fast_operand(v, kc, 0, 64, 64, 1) != (dtype == 0);
            ++forms;
          }
  printf("%lld forms, %lld wrong\n", forms, bad);
  return bad != 0;
}
'''


def test_vector_loads_need_aligned_rows(tmp_path):
    """The forms that load operands by 16-byte vectors are chosen only where every vector is aligned."""
    _host_run(tmp_path, ALIGNED)
