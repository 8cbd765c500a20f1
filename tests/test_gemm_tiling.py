"""The rule that picks the many-rows GEMM's tiling, on the CPU: the shapes with
which the GPU tests reach each tiling do so."""
import os
import shutil
import subprocess

import pytest
from test_gpu_gemm import TILINGS, TILINGS_SWIGLU

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("gemm") / "gemm_tiling")
    subprocess.run([gxx, "-O2", "-std=c++17", "-I", os.path.join(ROOT, "vllm-lite_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "gemm_tiling.cpp"), "-o", exe],
                   check=True)

    def run(m, wrows, k, silu):
        r = subprocess.run([exe], input=f"{m} {wrows} {k} {int(silu)}", check=True,
                           capture_output=True, text=True)
        return r.stdout.strip()
    return run


def test_tilings_of_the_gpu_tests(choose):
    for (m, n, k), tiling in TILINGS.items():
        assert choose(m, n, k, False) == tiling, (m, n, k)
    for (m, n, k), tiling in TILINGS_SWIGLU.items():
        assert choose(m, 2 * n, k, True) == tiling, (m, n, k)
    for t in (TILINGS, TILINGS_SWIGLU):
        # every tiling; the lowest two with K steps of 128 and of 64
        assert set(t.values()) == {"64x64", "64x128", "128x128", "128x128 pair", "256x128",
                                   "256x256"}
        for low in ("64x64", "64x128"):
            assert {k % 128 == 0 for (_, _, k), v in t.items() if v == low} == {True, False}
