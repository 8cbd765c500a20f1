"""Wait states that the compiler cannot add, checked in the built device code:
it sees into no inline assembly, so what a hand-written sequence needs has to
be written there."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
LDS_LOAD = re.compile(r"^(global_load_lds_|buffer_load_\w+ .*\blds\b)")


@pytest.fixture(scope="module")
def listings(tmp_path_factory):
    """The instructions of every gfx950 code object in libpa.so, in order."""
    lib = os.path.join(ROOT, "vllm-lite_amd", "libpa.so")
    if not os.path.exists(lib) or not os.path.exists(OBJDUMP):
        pytest.skip("no built library or no disassembler")
    d = tmp_path_factory.mktemp("device_code")
    shutil.copy(lib, d / "libpa.so")
    subprocess.run([OBJDUMP, "--offloading", "libpa.so"], cwd=d, check=True, capture_output=True)
    out = []
    for name in sorted(os.listdir(d)):
        if "gfx950" not in name:
            continue
        r = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", name], cwd=d, check=True,
                           capture_output=True, text=True)
        out.append([line.split("//")[0].strip() for line in r.stdout.splitlines()
                    if line.startswith("\t")])
    assert out, "no gfx950 code in libpa.so"
    return out


def test_m0_before_lds_loads(listings):
    """A scalar write of m0 and a load to LDS, which takes its LDS address from
    m0, are one wait state apart at least."""
    loads = 0
    for insns in listings:
        for prev, cur in zip(insns, insns[1:]):
            if LDS_LOAD.match(cur):
                loads += 1
                assert not re.match(r"s_\w+ m0\b", prev), f"{prev} / {cur}"
    assert loads > 0
