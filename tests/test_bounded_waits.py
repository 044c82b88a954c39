"""The waits of the Cholesky panels, read off the source: a wait that runs out cannot be had from a healthy device.  A workgroup that leaves
early does not set the flags that others wait for, so every wait also looks at info (else each of the others polls for seconds, with a CU to itself)."""
import re
from pathlib import Path

SOURCE = (Path(__file__).parents[1] / "qml_lightning_amd" / "csrc" / "solve.hip").read_text()


def body(start):
    """from `start` to the closing brace in the first column"""
    at = SOURCE.index(start)
    return SOURCE[at:SOURCE.index("\n}\n", at)]


def test_every_wait_looks_at_info():
    waits = [body("__device__ __forceinline__ unsigned await("), body("__device__ __forceinline__ bool follow_block(")]
    for text in waits:
        loop = text[text.index("n < spin_limit"):text.index("atomicCAS(info, 0, -1)")]
        assert re.search(r"\(n & \d+\) == \d+(, 0\))? && __hip_atomic_load\(info, [^;]*\) != 0\)?\s+(break|n = spin_limit - 1);", loop)
    # the other bounded loops are those of the two triangular solves, which hand on a NaN
    solves = [body("void fwd_solve_kernel("), body("void bwd_solve_kernel(")]
    assert [text.count("n < spin_limit") for text in waits + solves] == [1, 1, 1, 1]
    assert SOURCE.count("n < spin_limit") == 4 and SOURCE.count("atomicCAS(info, 0, -1)") == 2
