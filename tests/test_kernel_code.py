"""What the compiler made of the kernels, read from the assembly of a build of
its own (CPU only): properties that a result cannot show and a timing shows
only at some sizes."""

import re
import shutil
import subprocess
from pathlib import Path

import pytest

REPO = Path(__file__).resolve().parent.parent

pytestmark = pytest.mark.skipif(shutil.which("hipcc") is None
                                and not Path("/opt/rocm/bin/hipcc").exists(),
                                reason="hipcc is missing")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Kernel name -> its instructions and labels, in order."""
    from aegaeon_amd import build as lib_build

    out = tmp_path_factory.mktemp("asm") / "aegkv.s"
    flags = [f for f in lib_build.HIPCC_FLAGS if f not in ("-shared", "-fPIC")]
    res = subprocess.run([lib_build.hipcc(), *flags, "--cuda-device-only", "-S",
                          f"-I{REPO / 'include'}",
                          str(REPO / "aegaeon_amd" / "csrc" / "aegkv.hip"), "-o", str(out)],
                         capture_output=True, text=True, timeout=600)
    assert res.returncode == 0, res.stderr
    found = {}
    for m in re.finditer(r"^(_Z\w+_kernel\w+):.*?$(.*?)^\s+s_endpgm", out.read_text(),
                         re.M | re.S):
        found[m[1]] = [line.strip() for line in m[2].splitlines()]
    return found


def test_persistent_swaps_wait_for_an_item_s_stores(kernels):
    """A swap's workgroups take one item after another and wait for an item's
    stores before they load the next. The compiler places that wait, and the
    rate of work beside the swaps depends on it (move_tail16)."""
    checked = 0
    for name, lines in kernels.items():
        # <WG, U, TO_HOST, VEC = true, NT> with the loads per lane of persistent grids
        if not re.search(r"swap_tiles_kernelILi256ELi[24]ELb\dELb1E|swap_inline_kernelILb\dELb1E",
                         name):
            continue
        loop = next(i for i, x in enumerate(lines) if re.search(r"Loop Header: Depth=1", x))
        load = next(i for i, x in enumerate(lines) if i > loop and x.startswith("global_load"))
        assert any(x.startswith("s_waitcnt") and "vmcnt(0)" in x for x in lines[loop:load]), name
        checked += 1
    assert checked >= 8
