"""The waits of the Cholesky panels, read off the source: a wait that runs out cannot be had from a healthy device.  Every one of them
polls in the same loop, which also looks for a failure elsewhere, and an owner of the chain of factorisations that leaves early hands its
failure on to those who wait for it (else each of them polls for seconds, with a CU to itself)."""
import re
from pathlib import Path

SOURCE = (Path(__file__).parents[1] / "qml_lightning_amd" / "csrc" / "solve.hip").read_text()


def body(start):
    """from `start` to the closing brace in the first column"""
    at = SOURCE.index(start)
    return SOURCE[at:SOURCE.index("\n}\n", at)]


def test_every_wait_looks_at_info():
    poll = body("__device__ __forceinline__ unsigned poll(")
    loop = poll[poll.index("for ("):]
    assert "__hip_atomic_load(info" in loop and "break" in loop
    assert SOURCE.count("atomicCAS(info, 0, -1)") == poll.count("atomicCAS(info, 0, -1)") == 1
    # the other bounded loops are those of the two triangular solves, which hand on a NaN
    bounded = [body(k).count("n < spin_limit") for k in ("void fwd_solve_kernel(", "void bwd_solve_kernel(")]
    assert bounded == [1, 1] and SOURCE.count("n < spin_limit") == 3
    assert "poll<" in body("__device__ __forceinline__ unsigned await(") and "poll<" in body("__device__ __forceinline__ bool follow_block(")


def test_owners_of_the_chain_hand_their_failure_on():
    kernel = body("__global__ __launch_bounds__(PT, 2) void panel_kernel(")
    give_up = kernel[kernel.index("auto give_up"):kernel.index("};", kernel.index("auto give_up"))]
    for flag in ("flags + PBLK + l * PBLK + bid", "flags + STEPS + bid", "flags + bid"):
        assert "store_past_caches(%s, FLAG_FAILED)" % flag in give_up
    assert "await(heads_done + w, (unsigned)(mine + 1), spin_limit, info, seen) == FLAG_FAILED) return give_up(0);" in kernel
    chain = kernel[kernel.index("for (int l = 0; l < bid; ++l)"):kernel.index("potrf_block<true>")]
    assert len(re.findall(r"\breturn\b", chain)) == len(re.findall(r"return give_up\(l\);", chain)) == 2
