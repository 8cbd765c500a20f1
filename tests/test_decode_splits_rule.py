"""The rule for the workgroups that share a decode context, on the CPU: split
where that was measured faster, one workgroup where it was not or where no
workspace holds the partial results."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def splits(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("decode") / "decode_splits")
    subprocess.run([gxx, "-O2", "-std=c++17", "-I", os.path.join(ROOT, "vllm-lite_amd", "csrc"),
                    os.path.join(ROOT, "tests", "native", "decode_splits.cpp"), "-o", exe],
                   check=True)

    def run(*args):
        r = subprocess.run([exe], input=" ".join(map(str, args)), check=True,
                           capture_output=True, text=True)
        return int(r.stdout)
    return run


WS = 64 << 20


@pytest.mark.parametrize("b,hq,hkv,d,ctx", [
    (32, 14, 2, 64, 768), (32, 14, 2, 64, 640), (64, 14, 2, 64, 1024),
    (1, 14, 2, 64, 512), (1, 32, 8, 128, 256), (32, 32, 8, 128, 2000), (64, 32, 8, 128, 4096)])
def test_one_workgroup(splits, b, hq, hkv, d, ctx):
    assert splits(b, hq, hkv, d, ctx, 2, WS) == 1


@pytest.mark.parametrize("b,hq,hkv,d,ctx,es", [
    (1, 14, 2, 64, 2000, 2), (32, 14, 2, 64, 2000, 2), (1, 32, 8, 128, 1024, 2),
    (4, 32, 8, 128, 2000, 2), (16, 32, 8, 128, 4000, 2), (48, 32, 8, 128, 4096, 2),
    (8, 32, 8, 128, 512, 2),
    (16, 32, 8, 128, 8000, 1), (1, 32, 8, 128, 2000, 1), (4, 32, 8, 128, 512, 1)])
def test_several_workgroups(splits, b, hq, hkv, d, ctx, es):
    s = splits(b, hq, hkv, d, ctx, es, WS)
    assert s > 1 and ctx >= 64 * s
    row = b * hq * (d + 2) * 4  # one partial result of every row
    assert splits(b, hq, hkv, d, ctx, es, s * row - 1) < s
    assert splits(b, hq, hkv, d, ctx, es, 0) == 1
