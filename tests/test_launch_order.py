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

    def run(call, *numbers):
        """-> the launches, (kernel, template arguments, stream, arguments) each, and the number of words they leave"""
        out = subprocess.run([os.path.join(HERE, "_build", "launch_order"), build.HIP_LIB, call, *map(str, numbers)], check=True,
                             stdout=subprocess.PIPE, text=True).stdout
        *lines, (word, n) = [ln.split() for ln in out.splitlines()]
        assert word == "words"
        return [(ln[0], ln[1], ln[2], [int(w, 16) for w in ln[3:]]) for ln in lines], int(n)

    return run


# on both sides of the length from which on a placement ends with a scan, and at the largest table the library is used with
@pytest.mark.parametrize("num_rows", [1000, 1 << 26, (1 << 26) + 1, 500_000_000, (1 << 32) - 2])
def test_a_placement_leaves_its_ticket_behind_everything_the_host_goes_on_with(launches, num_rows):
    """once the ticket is there, launches on any stream may read the bitmap and the two workspaces: no launch of the placement
    behind the one that leaves the ticket may still write them"""
    new_bits, evict_ws, insert_ws, ticket = 0x1003_0000_0000, 0x1007_0000_0000, 0x1008_0000_0000, 0xABCD
    done, _ = launches("place", num_rows)
    assert len({stream for _, _, stream, _ in done}) == 1
    leaves = [i for i, (_, _, _, args) in enumerate(done) if ticket in args]
    assert len(leaves) == 1, done
    writes = [i for i, (_, _, _, args) in enumerate(done) if {new_bits, evict_ws, insert_ws} & set(args)]
    assert writes and max(writes) <= leaves[0], done


# rows and samples of every shape of the kernel and of the two that load by two hints, clipped ones among them
@pytest.mark.parametrize("id_bytes", [4, 8])
@pytest.mark.parametrize("row_bytes,bag,max_norm", [(64, 1, 0), (64, 8, 0), (128, 4, 0), (256, 4, 0), (256, 40, 0), (512, 1, 0),
                                                    (512, 4, 0), (384, 40, 0), (512, 16, 0), (1024, 4, 0), (1024, 40, 0),
                                                    (2048, 4, 0), (4096, 4, 0), (512, 4, 1), (2048, 4, 1), (4096, 4, 1)])
def test_a_pooled_lookup_nobody_polls_for_is_a_kernel_without_words(launches, id_bytes, row_bytes, bag, max_norm):
    """stream-ordered pooled lookups do not pay for what a polled launch stores and leaves: the two are different kernels"""
    plain, none = launches("pool", id_bytes, row_bytes, 1000 * bag, 1000, max_norm, 0)
    polled, words = launches("pool", id_bytes, row_bytes, 1000 * bag, 1000, max_norm, 1)
    assert none == 0 and words > 0 and len(plain) == len(polled) == 1
    assert plain[0][0] == polled[0][0] == "extract_pool_kernel"
    assert plain[0][1] != polled[0][1]
