"""The projections' kernels wait for an image in LDS with a count of what was issued behind its loads.  The source pins that order; here
it is read off the code that the compiler made, on the CPU."""
import os
import re
import shutil
import subprocess

import pytest

from qml_lightning_amd import build

# (kernel, what the wait lets stay on its way, how many of them)
KERNELS = [("typed_gemm_f16_kernelILi64E", "r", 4), ("typed_gemm_bt_rows_f16_kernelILi64E", "w", 16),
           ("typed_gemm_bt_rows_f16_kernelILi128E", "w", 16), ("typed_gemm_bt_rows_f16_kernelILi256E", "w", 16)]


def operations(text):
    """One letter per instruction: L load into LDS, r load, w store, B barrier, W wait for all but the last operations (a count), 0 wait
    for all of them."""
    out = ""
    for line in text.split("\n"):
        op = line.split("//")[0].split(";")[0].strip()
        if op.startswith(("global_load_lds", "buffer_load_lds")):
            out += "L"
        elif op.startswith(("global_load", "scratch_load")):
            out += "r"
        elif op.startswith(("global_store", "scratch_store")):
            out += "w"
        elif op.startswith("s_barrier"):
            out += "B"
        elif op.startswith("s_waitcnt") and "vmcnt" in op:
            out += "0" if "vmcnt(0)" in op else "W"
    return out


def images_are_waited_for(ops, kind, count):
    """Every wait that counts stands behind an image's loads and `count` operations of `kind` after them, and every barrier is followed by
    the next image's loads before anything else."""
    waits = [m.start() for m in re.finditer("W", ops)]
    for at in waits:
        behind = ops[ops.rindex("L", 0, at) + 1:at] if "L" in ops[:at] else ""
        if behind.count(kind) < count:
            return False
    return bool(waits) and all(ops[m.end():m.end() + 1] == "L" for m in re.finditer("B", ops))


def test_what_is_looked_for():
    good = "LLLrrrrrrrr" + "WBLLrrrr" * 3 + "WBLLwww"
    assert images_are_waited_for(good, "r", 4)
    assert not images_are_waited_for(good.replace("BLLrrrr", "BrLLrrr", 1), "r", 4)       # a load ahead of the image's
    assert not images_are_waited_for("LLLrrrrWBLLrrrWBLL", "r", 4)                        # one too few behind them
    assert not images_are_waited_for("LL0BLL" + "w" * 15 + "LWBLL", "w", 16)               # an image's load behind the stores
    assert images_are_waited_for("LL0BLL" + "w" * 16 + "WBLL", "w", 16)


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    if shutil.which(build.HIPCC) is None:
        pytest.skip("no compiler")
    out = str(tmp_path_factory.mktemp("asm") / "project.s")
    cmd = [build.HIPCC] + build.FLAGS + ["-x", "hip", "-S", "--cuda-device-only", os.path.join(build.CSRC, "project.hip"), "-o", out]
    subprocess.run(cmd, check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    return open(out).read()


@pytest.mark.parametrize("kernel,kind,count", KERNELS)
def test_images_are_issued_ahead(assembly, kernel, kind, count):
    text = re.search(r"^_ZN\S*%s\S*:(.*?)^\s*\.section" % kernel, assembly, re.S | re.M).group(1)
    assert images_are_waited_for(operations(text), kind, count)
