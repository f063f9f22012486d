"""The steps at which a resident launch cuts its blocks to store a snapshot row
(snap_step, run on the CPU): the positive multiples of the interval, for any
interval that the library takes, the largest int among them."""
import os
import subprocess

import pytest

from fdtd_pic_amd import build

SRC = r"""
#include <cstdio>
#include "device_common.hpp"
int main() {
    int t0s, k0, kend, interval;
    while (std::scanf("%d %d %d %d", &t0s, &k0, &kend, &interval) == 4)
        std::printf("%d\n", fdtd::snap_step(t0s, k0, kend, interval));
}
"""
TOP = 2 ** 31 - 1


@pytest.fixture(scope="module")
def snap_step(tmp_path_factory):
    if not os.path.exists(build.HIPCC):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("snap")
    (d / "snap.hip").write_text(SRC)
    subprocess.run([build.HIPCC] + build.FLAGS + ["-I", build.CSRC, str(d / "snap.hip"), "-o", str(d / "snap")],
                   check=True, capture_output=True)

    def ask(rows):
        text = "\n".join(" ".join(map(str, r)) for r in rows)
        r = subprocess.run([str(d / "snap")], input=text, text=True, check=True, capture_output=True)
        return [int(x) for x in r.stdout.split()]
    return ask


def test_snapshot_steps(snap_step):
    rows = []
    for interval in (1, 2, 3, 7, 48, 50, 1000, TOP // 2, TOP // 2 + 1, TOP - 1, TOP):
        for t0s in (0, 1, 5, 49, 997, interval - 60, interval - 1, interval, TOP - 70):
            if 0 <= t0s <= TOP - 64:
                rows += [(t0s, k0, k0 + n, interval) for k0 in (0, 1, 2, 13) for n in (1, 2, 17, 48)]
    for row, got in zip(rows, snap_step(rows)):
        t0s, k0, kend, interval = row
        want = next((k for k in range(k0, kend) if t0s + k > 0 and (t0s + k) % interval == 0), kend)
        assert got == want, row
