"""The projections' kernels as the compiler makes them, on the CPU.  They wait for an image in LDS with a count of what was issued behind
its loads: the source pins that order, which is read off the assembly here."""
import os
import re
import shutil
import subprocess

import pytest

from qml_lightning_amd import build

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


def images_are_waited_for(ops, count):
    """Every wait that counts stands behind an image's loads and `count` loads after them, and every barrier is followed by the next
    image's loads before anything else."""
    waits = [m.start() for m in re.finditer("W", ops)]
    for at in waits:
        behind = ops[ops.rindex("L", 0, at) + 1:at] if "L" in ops[:at] else ""
        if behind.count("r") < count:
            return False
    return bool(waits) and all(ops[m.end():m.end() + 1] == "L" for m in re.finditer("B", ops))


def test_what_is_looked_for():
    good = "LLLrrrrrrrr" + "WBLLrrrr" * 3 + "WBLLwww"
    assert images_are_waited_for(good, 4)
    assert not images_are_waited_for(good.replace("BLLrrrr", "BrLLrrr", 1), 4)       # a load ahead of the image's
    assert not images_are_waited_for("LLLrrrrWBLLrrrWBLL", 4)                        # one too few behind them
    assert not images_are_waited_for("LLLrrrrWBLLrrrLrWBLL", 4)                      # an image's load among them


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    if shutil.which(build.HIPCC) is None:
        pytest.skip("no compiler")
    out = str(tmp_path_factory.mktemp("asm") / "project.s")
    cmd = [build.HIPCC] + build.FLAGS + ["-x", "hip", "-S", "--cuda-device-only", os.path.join(build.CSRC, "project.hip"), "-o", out]
    subprocess.run(cmd, check=True, stdout=subprocess.DEVNULL, stderr=subprocess.DEVNULL)
    return open(out).read()


def code(assembly, kernel):
    return operations(re.search(r"^_ZN\S*%s\S*:(.*?)^\s*\.section" % kernel, assembly, re.S | re.M).group(1))


def test_images_are_issued_ahead(assembly):
    assert images_are_waited_for(code(assembly, "typed_gemm_f16_kernelILi64E"), 4)


@pytest.mark.parametrize("columns", [64, 128, 256])
def test_an_image_on_its_way_is_not_waited_for(assembly, columns):
    """In the transposed kernel the next image's loads overlap the products: no wait for all of them between the image's loads and the
    stores of the block."""
    ops = code(assembly, "typed_gemm_bt_rows_f16_kernelILi%dE" % columns)
    assert "W" not in ops
    for m in re.finditer("BL+", ops):
        assert ops[m.end()] == "w"
