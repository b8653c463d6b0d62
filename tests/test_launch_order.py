"""What the built kernel library launches, and in which order, on the CPU: tests/sanitizer/launch_order.cc lists the launches
of a call instead of performing them."""
import os
import subprocess

import pytest

from ugache_amd import build

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "sanitizer")


@pytest.fixture(scope="module")
def launches():
    proc = subprocess.run(["make", "-C", HERE, "_build/launch_order"], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert proc.returncode == 0, proc.stdout[-4000:]
    if not os.path.exists(build.HIP_LIB):
        build.build_hip()

    def run(call, number):
        out = subprocess.run([os.path.join(HERE, "_build", "launch_order"), build.HIP_LIB, call, str(number)], check=True,
                             stdout=subprocess.PIPE, text=True).stdout
        lines = [ln.split() for ln in out.splitlines()]
        return [(ln[0], ln[1], [int(w, 16) for w in ln[2:]]) for ln in lines]

    return run


# on both sides of the length from which on a placement ends with a scan, and at the largest table the library is used with
@pytest.mark.parametrize("num_rows", [1000, 1 << 26, (1 << 26) + 1, 500_000_000, (1 << 32) - 2])
def test_a_placement_leaves_its_ticket_behind_everything_the_host_goes_on_with(launches, num_rows):
    """once the ticket is there, launches on any stream may read the bitmap and the two workspaces: no launch of the placement
    behind the one that leaves the ticket may still write them"""
    new_bits, evict_ws, insert_ws, ticket = 0x1003_0000_0000, 0x1007_0000_0000, 0x1008_0000_0000, 0xABCD
    done = launches("place_with_ticket", num_rows)
    assert len({stream for _, stream, _ in done}) == 1
    leaves = [i for i, (_, _, args) in enumerate(done) if ticket in args]
    assert len(leaves) == 1, done
    writes = [i for i, (_, _, args) in enumerate(done) if {new_bits, evict_ws, insert_ws} & set(args)]
    assert writes and max(writes) <= leaves[0], done
