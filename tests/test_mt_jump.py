"""The jump-ahead polynomials of csrc/mt_jump.h against the MT19937 stream itself (CPU)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r'''
#include <stdio.h>
#include <vector>
#include "mt_jump.h"
int main() {
  using namespace mt_jump;
  std::vector<uint32_t> x((size_t)624 * 3 * 32 + 2 * 19937);
  seed_state(5489u, x.data());
  for (size_t n = 624; n < x.size(); ++n) {
    const uint32_t y = (x[n - 624] & 0x80000000u) | (x[n - 623] & 0x7fffffffu);
    x[n] = x[n - 227] ^ (y >> 1) ^ ((y & 1u) ? 0x9908b0dfu : 0u);
  }
  int bad = 0;
  const int es[] = {5, 0, 3};           // out of order, twice
  for (int k = 0; k < 6; ++k) {
    const int e = es[k % 3];
    for (int r = 1; r <= 3; ++r) {
      const Poly& p = powers(e)[r - 1];
      const size_t J = ((size_t)624 * r) << e;
      for (int t = 0; t < 624; t += 13) {
        uint32_t s = 0;
        for (int i = 0; i < kDeg; ++i)
          if ((p.w[i >> 6] >> (i & 63)) & 1u) s ^= x[i + t];
        bad += t == 0 ? (s ^ x[J]) >> 31 : s != x[J + t];   // the first word's top bit counts
      }
      bad += (int)(p.w[kW64 - 1] >> (kDeg & 63) != 0);      // nothing at or above the degree
    }
  }
  bad += powers(-1) != nullptr || powers(kMaxE + 1) != nullptr || powers(kMaxE) == nullptr;
  printf("%u %u %d\n", x[1], x[623], bad);
  return bad != 0;
}
'''


def test_jump_polynomials_reproduce_the_stream(tmp_path):
    cxx = shutil.which('g++')
    if cxx is None:
        pytest.skip('no host C++ compiler')
    import numpy as np
    src = tmp_path / 'jump.cpp'
    src.write_text(SRC)
    exe = tmp_path / 'jump'
    subprocess.run([cxx, '-O2', '-std=c++17',
                    '-I', os.path.join(ROOT, 'brainstate_amd', 'csrc'), str(src), '-o', str(exe)],
                   check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out
    state = np.random.RandomState(5489).get_state()[1]
    assert out.stdout.split() == [str(state[1]), str(state[623]), '0']


# draws, bound and the segments their stream is cut into: the plans measured as the fastest
@pytest.mark.parametrize('n_pre,k,n_post,segs', [(800_000, 100, 1_000_000, 263),
                                                 (200_000, 80, 200_000, 263),
                                                 (3200, 80, 4000, 14), (100, 100, 4000, 1)])
def test_segments_of_a_stream(n_pre, k, n_post, segs):
    import math

    from brainstate_amd import _native as N
    p = n_post / 2.0 ** (n_post - 1).bit_length()
    words = int(n_pre * k / p + 12 * math.sqrt(n_pre * k * (1 - p)) / p) + 2 * 624
    blocks = -(-words // 624)
    pad = lambda n: -(-n // 256) * 256  # noqa: E731
    size = lambda s: pad(blocks * 2496) + pad(blocks * 4) + pad(s * 4) + pad(s * 2496) + 256  # noqa: E731
    assert N.lib().bs_conn_fixed_num_workspace_size(n_pre, k, n_post, 0) == size(segs)
