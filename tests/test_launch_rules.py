"""The host code's launch rules (wendy_amd/csrc/wdy_rules.h) over everything the
entry points accept, compiled by themselves: no GPU."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

PAIRS = r'''
#include "wdy_rules.h"
#include <cstdio>
using namespace wdy;
int main() {
  const uint32_t ns[] = {0, 1, 2, 255, 256, 1023, 1024, 1025, 2047, 4096, 30000,
                         131072, 1000003, (1u << 30) - 1};
  const uint32_t nys[] = {1, 3, 4, 5, 4095, 4096, 4097, 30000, 1u << 20, (1u << 31) - 1};
  for (uint32_t n : ns)
    for (uint32_t ny : nys) {
      const PairPlan p = pair_plan(n, ny, 256);
      const uint64_t all = (uint64_t)p.splits * p.per;
      // every sheet in one stretch, none of them empty (unless there are none)
      if (p.per < 1 || p.splits < 1 || p.splits > 128 || all < n ||
          (n > 0 && all - p.per >= n) || (n == 0 && p.splits != 1)) {
        std::printf("n=%u ny=%u: %u stretches of %u\n", n, ny, p.splits, p.per);
        return 1;
      }
    }
  return 0;
}
'''

# Launch q meets words that earlier launches left (0, or 1 + one of them) and,
# once a window of it has failed, 1 + q: never both answers.
LEAVES = r'''
#include "wdy_rules.h"
#include <cstdio>
using namespace wdy;
int main() {
  for (uint32_t q = 0; q < 70; ++q)
    for (uint32_t before = 0; before <= q; ++before) {
      const bool leaves = span_leaves(before, q);
      if (leaves != (before != 0) || (!leaves && span_leaves(q + 1, q))) {
        std::printf("launch %u, word %u\n", q, before);
        return 1;
      }
    }
  return 0;
}
'''

RING = r'''
#include "wdy_rules.h"
#include <cstdio>
using namespace wdy;
int main() {
  for (uint32_t first : {0u, 1u, 1000u, LAUNCH_RING - 3, LAUNCH_RING - 1}) {
    uint32_t q = first;
    for (int k = 0; k < 10; ++k, q = next_launch(q))
      if (q >= LAUNCH_RING || q + 1 == 0 || launch_of(q, first, 7) != (k < 7 ? k : -1)) {
        std::printf("launch %u from %u: place %lld\n", q, first,
                    (long long)launch_of(q, first, 7));
        return 1;
      }
  }
  return 0;
}
'''

SPLITS = r'''
#include "wdy_rules.h"
#include <cstdio>
using namespace wdy;
int main() {
  const int ns[] = {1, 2, 7, 8, 9, 100, 1001, 1 << 30, 1879048193, 2147483647};
  for (int nleap : ns) {
    int tried = 0, most = 0;
    bool ok = true;
    each_split(nleap, [&](int K, int launches) {
      ok = ok && K >= 1 && launches >= 1 && (int64_t)K * launches >= nleap &&
           (int64_t)K * (launches - 1) < nleap;
      tried += 1;
      most = launches > most ? launches : most;
    });
    if (!ok || tried > 200 || most < (nleap < 9 ? nleap : nleap / 2)) {
      std::printf("nleap=%d: %d tried, at most %d launches\n", nleap, tried, most);
      return 1;
    }
  }
  return 0;
}
'''


def run(tmp_path, source):
    cxx = os.environ.get('CXX') or shutil.which('g++')
    assert cxx, 'no C++ compiler'
    src = tmp_path / 't.cpp'
    src.write_text(source)
    exe = str(tmp_path / 't')
    subprocess.run([cxx, '-std=c++17', '-O1', '-Wall', '-Werror', '-I',
                    os.path.join(ROOT, 'wendy_amd', 'csrc'), str(src), '-o', exe], check=True)
    got = subprocess.run([exe], capture_output=True, text=True)
    assert got.returncode == 0, (got.returncode, got.stdout)


@pytest.mark.parametrize('source', [PAIRS, LEAVES, RING, SPLITS],
                         ids=['pairs', 'leaves', 'ring', 'splits'])
def test_rules(tmp_path, source):
    run(tmp_path, source)
