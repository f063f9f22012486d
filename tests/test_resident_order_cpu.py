"""Ordering of the resident mailbox (ResArgs): between the stores that empty a
slot's words and the sends of the next hand-off the wave waits until its vector
stores are in memory.  Checked in the code that the compiler makes for gfx950:
the wait itself, between two mailbox stores, and in every step loop that a tile
body of the resident kernel ends a block with."""
import os
import re
import subprocess

import pytest

from fdtd_pic_amd import build

SRC = """
#include "stencil_kernels.hpp"
namespace fdtd {
__global__ void between(unsigned long long* p, unsigned long long v) {
    st_dev(p, kResEmpty);
    stores_done();
    st_dev(p + 64, v);
}
template __global__ void stencil_resident<float, true, SLAB_DIEL, 2>(const SimDev<float>*, const int4*, int, long long,
                                                                     long long, ResArgs);
}
"""


@pytest.fixture(scope="module")
def functions(tmp_path_factory):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("order")
    src, out = d / "order.hip", d / "order.s"
    src.write_text(SRC)
    subprocess.run([build.HIPCC] + build.FLAGS + ["-I", build.CSRC, "--offload-device-only", "-S", str(src), "-o",
                                                  str(out)], check=True, capture_output=True)
    got, name = {}, None
    for line in out.read_text().split("\n"):
        m = re.match(r"^(_Z\w+):", line)
        if m:
            name = m.group(1)
            got[name] = []
        elif line.startswith(".Lfunc_end"):
            name = None
        elif name:
            got[name].append(line.strip())
    return got


def test_stores_wait_between(functions):
    code = next(v for k, v in functions.items() if "between" in k)
    at = [i for i, x in enumerate(code) if x.startswith("global_store_dwordx2") and " sc1" in x]
    assert len(at) == 2
    waits = [x for x in code[at[0]:at[1]] if x.startswith("s_waitcnt")]
    assert any("vmcnt(0)" in x for x in waits), waits


def test_every_step_loop_of_the_resident_kernel_waits(functions):
    """K = 4: one loop; K = 1 and 2 of plain tiles: plain, strip, and strip with
    source, probe or both.  Each ends with the wait as inline code."""
    code = "\n".join(next(v for k, v in functions.items() if "stencil_resident" in k))
    waits = re.findall(r";+#?ASMSTART\ns_waitcnt vmcnt\(0\)\n;+#?ASMEND", code)
    assert len(waits) >= 1 + 2 * 5, len(waits)
