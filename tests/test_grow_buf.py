"""The contexts' buffers (scriptonait_amd/csrc/grow_buf.h) on the CPU: a
request that grows a little from call to call, as a generation's history
makes it, reallocates once per doubling and not on every call."""
import subprocess
import textwrap
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "scriptonait_amd" / "csrc"

MAIN = textwrap.dedent(r"""
    #include <stdint.h>
    #include <stdio.h>
    #include <stdlib.h>
    #include "grow_buf.h"
    static int allocs = 0, frees = 0, fail = 0;
    static size_t last = 0;
    struct Mem {
      static int alloc(void** p, size_t n) { if (fail) return 7; ++allocs; last = n; *p = malloc(1); return 0; }
      static int free(void* p) { ++frees; ::free(p); return 0; }
    };
    int main(int argc, char** argv) {
      const size_t base = strtoull(argv[1], 0, 10), step = strtoull(argv[2], 0, 10), n = strtoull(argv[3], 0, 10);
      llmhip::GrowBuf<Mem> b;
      int bad = 0;
      for (size_t i = 0; i < n; ++i) {
        const size_t want = base + i * step;
        bad += b.ensure(want) != 0 || b.cap < want || b.cap != last;
        bad += want > ((size_t)8 << 20) && b.cap > base + n * step;  /* no rounding of large buffers */
      }
      bad += allocs != frees + 1;
      fail = 1;
      bad += b.ensure(b.cap + 1) != 7 || b.ptr || b.cap;  /* a failed call leaves it empty */
      bad += frees != allocs || b.release() != 0 || frees != allocs;
      printf("%d %d\n", allocs, bad);
    }
""")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("grow")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run(["g++", "-O1", "-std=c++17", f"-I{CSRC}", str(d / "main.cpp"), "-o", str(d / "main")], check=True)
    return d / "main"


# One row of 32000 logits and its history (4 bytes an id); an empty start; the
# sizes around 8 MiB, up to which requests are rounded; larger ones.
@pytest.mark.parametrize("base,step,n,most", [(130_432, 4, 4096, 2), (1, 1, 1 << 20, 13), ((8 << 20) - 8, 4, 3, 1),
                                              ((8 << 20) + 4, 1 << 20, 4, 4)])
def test_growing_requests_reallocate_once_per_doubling(exe, base, step, n, most):
    out = subprocess.run([str(exe), str(base), str(step), str(n)], check=True, capture_output=True, text=True).stdout
    allocs, bad = map(int, out.split())
    assert bad == 0
    assert allocs <= most
