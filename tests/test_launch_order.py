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
        run.grids = [tuple(map(int, ln[3].split("x"))) for ln in lines]
        return [(ln[0], ln[1], ln[2], [int(w, 16) for w in ln[4:]]) for ln in lines], int(n)

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


# (table, row bytes, keys): eight rows of a lane on their way in small launches of long rows, four in the others
@pytest.mark.parametrize("kind,row_bytes,n,rows", [(3, 512, 8_192, 4), (3, 1024, 8_192, 8), (3, 512, 8_193, 8), (3, 512, 65_536, 8),
                                                   (3, 512, 65_537, 4), (3, 512, 262_145, 4), (3, 1024, 400_000, 4), (2, 4096, 65_536, 8),
                                                   (2, 4096, 270_000, 4), (1, 1024, 4_096, 8), (1, 1024, 4_097, 4)])
@pytest.mark.parametrize("words", [0, 1])
def test_rows_on_their_way_in_a_mixed_lookup(launches, kind, row_bytes, n, rows, words):
    templ = launches("mix", row_bytes, n, words, kind)[0][0][1].strip("<>").split(",")
    assert templ[1] == str(kind) and int(templ[4]) == rows, templ


@pytest.mark.parametrize("row_bytes", [16, 20, 32])
def test_a_polled_gather_of_short_rows_is_one_kernel_at_every_size(launches, row_bytes):
    """its stores need no room in the L2s, so that as many lines as those hold are no reason to read past them"""
    seen = {launches("gather", row_bytes, rows, 1)[0][0][:2] for rows in (170_000, 180_224, 180_225, 262_144, 458_752, 458_753, 900_000)}
    assert len(seen) == 1


# (row bytes, megabytes of output, when words come, against a ticket kernel): on both sides of every line of the rules
@pytest.mark.parametrize("call,row_bytes,mb,told", [
    ("gather", 512, 8, "sooner"), ("gather", 64, 8, "sooner"), ("gather", 12, 8, "sooner"), ("gather", 2048, 8, "sooner"),
    ("gather", 1040, 8, "sooner"), ("gather", 4096, 0.1, "sooner"), ("gather", 4096, 33, "sooner"), ("gather", 4096, 34, "sooner"),
    ("gather", 8192, 8, "sooner"), ("gather", 200, 8, "sooner"), ("gather", 3200, 8, "sooner"), ("gather", 1204, 8, "sooner"),
    ("gather", 193, 1, "too late"), ("gather", 193, 34, "too late"), ("gather", 98, 1, "too late"), ("gather", 15, 1, "too late"),
    ("mix", 1024, 8, "sooner"), ("mix", 1040, 8, "sooner"), ("mix", 1204, 30, "sooner"), ("mix", 4096, 33, "sooner"),
    ("mix", 4096, 34, "sooner"), ("mix", 4112, 100, "sooner"), ("mix", 36, 8, "sooner"),
])
def test_a_lookup_is_told_its_end_by_words_where_they_are_sooner(launches, call, row_bytes, mb, told):
    rows = int(mb * 1e6 / row_bytes)
    plain, none = launches(call, row_bytes, rows, 0)
    done, words = launches(call, row_bytes, rows, 2)
    assert none == 0 and (words > 0) == (told == "sooner")
    assert (done[0][:2] == plain[0][:2]) == (words == 0)  # without words it is the launch nobody polls for
    assert launches(call, row_bytes, rows, 1)[1] > 0  # who insists gets them
    assert (launches(call, row_bytes, rows, 3)[1] > 0) == (told != "too late")  # keys would be copied by a kernel


# (table, row bytes, rows): few long rows and many
@pytest.mark.parametrize("kind,row_bytes,rows", [(1, 1040, 4_032), (1, 1040, 4_034), (1, 4112, 1_020), (1, 4112, 1_021), (3, 1040, 4_034),
                                                 (2, 4112, 8_160), (3, 4112, 5), (3, 4112, 4), (1, 4112, 4), (3, 4096, 4)])
def test_a_mixed_lookup_of_long_rows_is_told_its_end_by_words(launches, kind, row_bytes, rows):
    assert launches("mix", row_bytes, rows, 2, kind)[1] > 0
    assert launches("mix", row_bytes, rows, 1, kind)[1] > 0  # who insists gets them


@pytest.mark.parametrize("row_bytes,bag,mb,told", [(512, 1, 67, True), (512, 1, 67.2, False), (512, 2, 68, False), (512, 3, 68, True),
                                                   (1024, 2, 67, True), (1024, 2, 68, False), (4096, 4, 134, True)])
def test_a_pooled_lookup_is_told_its_end_by_words_where_they_are_sooner(launches, row_bytes, bag, mb, told):
    samples = int(mb * 1e6 / row_bytes)
    words = [launches("pool", 8, row_bytes, samples * bag, samples, 0, how)[1] for how in range(4)]
    assert words[0] == 0 and words[1] > 0 and (words[2] > 0) == (words[3] > 0) == told


@pytest.mark.parametrize("row_bytes", [512, 404, 12, 3])
@pytest.mark.parametrize("words", [1, 3])
def test_a_scattering_gather_takes_the_request_and_leaves_no_words(launches, row_bytes, words):
    """its keys are not those of its output rows, so it could not leave them; nor does the next call see the request"""
    done, left = launches("scatter", row_bytes, 1000, words)
    assert left == 0 and len(done) == 2
    assert not any("Store)2" in templ for _, templ, _, _ in done)


@pytest.mark.parametrize("nbits", [1, 4096, 100_000, 1 << 21, (1 << 21) + 1, 4_000_000, (1 << 25) + 1, 50_500_000, 1 << 26])
def test_lists_out_of_a_bitmap_are_dealt_out_over_the_chip(launches, nbits):
    """a wavefront per chunk that holds any bit; set bits in one run are in a few neighbouring chunks, so there are as many
    workgroups as chunks, or hundreds of them, and no wavefront at or beyond the 8,192 counts of a workspace"""
    words = (nbits + 63) // 64
    per_chunk = ((words + 8191) // 8192 + 63) // 64 * 64
    chunks = (words + per_chunk - 1) // per_chunk
    done, _ = launches("lists", nbits)
    assert [kernel for kernel, _, _, _ in done] == ["bitmap_emit_small_kernel"] * 2
    for groups, threads in launches.grids:
        assert threads % 64 == 0 and threads <= 1024
        assert groups >= min(chunks, 250) and chunks <= groups * (threads // 64) <= 8192
