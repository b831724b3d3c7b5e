"""The closed-form item numbering of the operator's grids (csrc/ca_kernels.h)
against a walk over the groups, over passes, chunk lengths and sizes (CPU)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "continuum-attention_amd", "csrc", "ca_kernels.h")

PROGRAM = r"""
#include "%s"
#include <cstdio>
using namespace ca;
int main() {
  long bad = 0, n = 0;
  for (int T : {1, 31, 32, 33, 127, 128, 129, 500, 512, 1001, 2048, 2049, 5000, 8192, 20000})
    for (int C : {1, 2, 3, 5, 7, 8, 12, 16, 21, 24, 28, 48, 100, 700}) {
      const int G = (T + 127) / 128, all = (T + 31) / 32;
      int item = 0;
      for (int g = G - 1; g >= 0; --g) {
        const int nt = 4 * g + 4 < all ? 4 * g + 4 : all, ns = (nt + C - 1) / C;
        for (int s = 0; s < ns; ++s, ++item, ++n) {
          const ItemPos p = fwd_find_item(item, G, T, C);
          bad += p.group != G - 1 - g || p.chunk != s || p.chunks != ns;
        }
      }
      bad += fwd_find_item(item, G, T, C).chunks != 0 || item != fwd_num_items(T, C);
      const int Q = dq_num_groups(T);
      for (int g0 : {0, Q / 3, Q / 2})
        for (int g1 : {g0 + 1, (g0 + Q + 1) / 2, Q}) {
          if (g1 <= g0 || g1 > Q) continue;
          const BwdPass p = bwd_pass(T, g0, g1);
          int it = 0;
          for (int q = g1 - 1; q >= g0; --q) {
            const int nc = dq_group_chunks(q, T, C);
            bad += dq_items_before(g1 - 1 - q, T, g0, g1, C) != it;
            for (int s = 0; s < nc; ++s, ++it, ++n) {
              const ItemPos x = dq_find_item(it, T, g0, g1, C);
              bad += x.group != g1 - 1 - q || x.chunk != s || x.chunks != nc;
            }
          }
          it = 0;
          for (int w = 0; w < p.kv_groups; ++w) {
            const int nc = dkdv_group_chunks(w, p, C);
            bad += dkdv_items_before(w, p, C) != it;
            for (int s = 0; s < nc; ++s, ++it, ++n) {
              const ItemPos x = dkdv_find_item(it, p, C);
              bad += x.group != w || x.chunk != s || x.chunks != nc;
            }
          }
        }
    }
  std::printf("%%ld items, %%ld wrong\n", n, bad);
  return bad != 0;
}
"""


def test_item_numbering(tmp_path):
    hipcc = os.environ.get("HIPCC") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc) and shutil.which("hipcc") is None:
        pytest.skip("hipcc not installed")
    src, exe = tmp_path / "items.hip", tmp_path / "items"
    src.write_text(PROGRAM % HEADER)
    subprocess.run([hipcc if os.path.exists(hipcc) else "hipcc", "--offload-arch=gfx950", "-O2",
                    "-std=c++17", "-w", str(src), "-o", str(exe)], check=True, capture_output=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.endswith(" 0 wrong\n"), out.stdout
