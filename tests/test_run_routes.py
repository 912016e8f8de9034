"""CPU check of the rule that sends a 2D run through the multi-operation kernels
(``multi2d_takes`` of csrc/step_impl.hpp, compiled for the host): which launch
reads and writes which buffer, over run lengths and buffers that overlap."""

import subprocess

from vivsim_amd import _build

PROGRAM = r"""
#include <climits>
#include <cstdio>
#include "step_impl.hpp"
using namespace vsx;

// whether some launch of a multi-operation run reads a buffer that it writes
static bool clash(const char *in, const char *out, const char *wa, const char *wb, int64_t f, int64_t w, int n) {
  const int64_t launches = ((int64_t)n + 1 + kRunOps - 1) / kRunOps;
  const char *bufs[2] = {wa, wb}, *cur = in;
  int64_t cur_bytes = f;
  for (int64_t j = 0; j < launches; ++j) {
    const bool last = j == launches - 1;
    const char *dst = last ? out : bufs[j & 1];
    const int64_t bytes = last ? f : w;
    if (cur < dst + bytes && dst < cur + cur_bytes) return true;
    cur = dst;
    cur_bytes = bytes;
  }
  return false;
}

int main() {
  VsxLbm p{};
  p.nx = 64;
  p.ny = 50;
  p.nz = 1;
  int bad = 0;
  for (int n = INT_MAX - 8; n > 0 && n <= INT_MAX - 1; ++n) bad += run_launches(n) != n / kRunOps + 1;
  bad += run_launches(INT_MAX) != INT_MAX / kRunOps + 1 || run_launches(5) != 1 || run_launches(6) != 2;
  if (bad) printf("launches of the longest runs\n");
  for (int storage = 0; storage < 2; ++storage) {
    p.storage = storage;
    const StepCtx c = make_ctx<D2Q9>(p, Window{nullptr, nullptr, {0, 0, 0}});
    const int64_t f = 36 * c.n, w = 9 * c.n * (int64_t)store_bytes(storage);
    // four buffers one after the other, and every pair of them moved onto one another, wholly and by a part
    char *base = reinterpret_cast<char *>(uintptr_t(1) << 32);
    for (int n = 1; n <= 40; ++n)
      for (int a = 0; a < 4; ++a)
        for (int b = 0; b < 4; ++b)
          for (int64_t shift : {int64_t(0), f / 2, -f / 2, w - 4, 4 - w}) {
            if ((a == 2 && b == 3) || (a == 3 && b == 2)) continue;   // the two work buffers are distinct
            char *q[4] = {base, base + 2 * f, base + 4 * f, base + 6 * f};   // f_in, f_out, work_a, work_b
            if (a != b) q[a] = q[b] + shift;
            const bool takes = multi2d_takes(c, (const float *)q[0], (const float *)q[1], q[2], q[3], n);
            if (takes == clash(q[0], q[1], q[2], q[3], f, w, n)) {
              printf("storage %d n %d buffers %d, %d shift %lld: takes %d\n", storage, n, a, b, (long long)shift, takes);
              ++bad;
            }
          }
  }
  return bad ? 1 : 0;
}
"""


def test_buffers_of_a_run(tmp_path):
    """A run takes the multi-operation kernels where no launch reads what it
    writes, and the single passes otherwise: a run in place, an input that is a work
    buffer (collided in place), an output that is the idle work buffer."""
    src, exe = tmp_path / "routes.hip", tmp_path / "routes"
    src.write_text(PROGRAM)
    subprocess.run([_build.HIPCC, *_build.FLAGS, "--offload-host-only", "-O1", "-I", _build.CSRC, "-c", str(src),
                    "-o", str(tmp_path / "routes.o")], check=True, capture_output=True)
    subprocess.run([_build.HIPCC, str(tmp_path / "routes.o"), _build.LIB, "-o", str(exe),
                    f"-Wl,-rpath,{_build.HERE}"], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr
