"""Which calls with waiting workgroups may run at once on a device (csrc/
residency.hpp), on the host: one whose places are refused runs panels that do
not wait."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "multifloatlinearalgebra.jl_amd", "csrc")

MAIN = r"""
#include <cstdio>
#include <cstdlib>
#include <memory>
#include "residency.hpp"
int main(int argc, char **argv) {   // device:groups:per_cu:cus takes and keeps, "-" gives the oldest back
    std::list<std::unique_ptr<mfk::WaitingPlaces>> held;
    for (int i = 1; i < argc; ++i) {
        if (argv[i][0] == '-') { held.pop_front(); continue; }
        int dev; long long g, p, c;
        std::sscanf(argv[i], "%d:%lld:%lld:%lld", &dev, &g, &p, &c);
        auto w = std::make_unique<mfk::WaitingPlaces>();
        const bool ok = w->take(dev, {g, p, c});
        std::printf("%d", ok);
        if (ok) held.push_back(std::move(w));
    }
}
"""


@pytest.fixture(scope="module")
def takes(tmp_path_factory):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("residency")
    (d / "main.cpp").write_text(MAIN)
    subprocess.run([cxx, "-std=c++17", "-I", CSRC, str(d / "main.cpp"), "-o", str(d / "main"), "-lpthread"], check=True)
    return lambda *a: subprocess.run([str(d / "main"), *a], check=True, capture_output=True, text=True).stdout


@pytest.mark.parametrize("calls,want", [
    # lu!: two workgroups a CU. Four largest panels fill the device, a fifth waits for none of them
    (["0:128:2:256"] * 5, "11110"),
    (["0:64:2:256"] * 9, "111111110"),
    # on one 32-CU mask a single panel of 64, and again once it has ended
    (["0:64:2:32", "0:64:2:32", "-", "0:64:2:32"], "101"),
    (["0:65:2:32", "0:64:2:32"], "01"),
    # nine workgroups are two on the first XCD, whose share of the mask is four CUs
    (["0:9:1:32"] * 3, "110"),
    (["0:8:1:32"] * 5, "11110"),
    (["0:16:2:8", "0:17:2:8", "0:2:2:7"], "100"),
    # ldlt!'s panels, one a CU, all on the same 32 CUs; on the device's CUs instead
    (["0:32:1:32", "0:32:1:32", "0:32:1:256"], "101"),
    (["0:64:1:256"] * 5, "11110"),
    # lu! over the device ends whatever ldlt! holds, and then ldlt! does
    (["0:128:2:256", "0:32:1:32"], "11"),
    (["0:32:1:32", "0:128:2:256", "0:128:2:256"], "111"),
    # on the same mask each could keep the other out; ldlt! over the device ends first
    (["0:32:1:32", "0:64:2:32"], "10"),
    (["0:32:1:256", "0:64:2:32"], "11"),
    # devices do not share CUs
    (["0:64:2:32", "1:64:2:32"], "11"),
    (["64:1:2:256", "99:1:2:256"], "00"),
])
def test_places(takes, calls, want):
    assert takes(*calls) == want
