"""Settings that belong to a device (the dynamic LDS that a kernel may take) are
made on each device that a process uses, not on its first one alone: the host
helper csrc/per_device.h, built here and driven with a recording stand-in for
the HIP call."""
import re
import subprocess

from conftest import ROOT

CSRC = ROOT / "10_20_amd" / "csrc"

PROGRAM = r"""
#include <stdio.h>
#include <initializer_list>
#include "per_device.h"
int main() {
    v1::OncePerDevice once, other;
    int calls[66] = {0}, fail = 0;
    auto on = [&](v1::OncePerDevice& o, int dev) {
        return o.run(dev, [&] { ++calls[dev < 0 ? 65 : dev]; return fail; });
    };
    int bad = 0;
    // every device once, whichever came first
    for (int k = 0; k < 3; ++k) for (int dev : {0, 1, 7, 63}) bad |= on(once, dev);
    bad |= calls[0] != 1 || calls[1] != 1 || calls[7] != 1 || calls[63] != 1;
    bad |= (on(other, 0) | on(other, 0)) || calls[0] != 2;  // another kernel's
    // a failure is returned and tried again, and leaves the other devices alone
    fail = -3;
    bad |= on(once, 2) != -3 || on(once, 2) != -3 || calls[2] != 2 || on(once, 0) != 0;
    fail = 0;
    bad |= (on(once, 2) | on(once, 2)) || calls[2] != 3;
    // devices that have no bit, and an unknown one: each time
    bad |= (on(once, 64) | on(once, 64)) || calls[64] != 2 || (on(once, -1) | on(once, -1)) || calls[65] != 2;
    printf("%s\n", bad ? "bad" : "ok");
    return bad;
}
"""


def test_once_per_device(tmp_path):
    src = tmp_path / "t.cpp"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-I", str(CSRC), str(src), "-o", str(tmp_path / "t")], check=True)
    assert subprocess.run([str(tmp_path / "t")], capture_output=True, text=True).stdout == "ok\n"


def test_lds_limits_are_set_through_it():
    for path in CSRC.glob("*.hip"):
        text = path.read_text()
        assert "call_once" not in text and "hipFuncSetAttribute" not in text, path.name
    assert len(re.findall(r"hipFuncSetAttribute", (CSRC / "common.h").read_text())) == 1
