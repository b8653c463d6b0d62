"""What the compiler makes of the kernels' own assembler, on the CPU (hipcc compiles for gfx950 without a GPU)."""
import os
import re
import subprocess

import pytest

from ugache_amd import build

# a store whose data the next vector instruction overwrites: in C, where the compiler puts the wait states in between that the
# target wants, and by store_through
SOURCE = """
#include "ugk_mix.cuh"
template <typename V, bool THROUGH>
__device__ __forceinline__ void body(V *p, const V *q, unsigned a, int n) {
  V v = q[threadIdx.x];
#pragma unroll 1
  for (int i = 0; i < n; ++i) {
    if constexpr (THROUGH) ugk::store_through(reinterpret_cast<uint64_t>(p + threadIdx.x), v);
    else p[threadIdx.x] = v;
    __builtin_amdgcn_sched_barrier(0);
    v ^= a;
    __builtin_amdgcn_sched_barrier(0);
  }
}
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
#define KERNELS(NAME, V) \\
  __global__ void NAME##_by_compiler(V *p, const V *q, unsigned a, int n) { body<V, false>(p, q, a, n); } \\
  __global__ void NAME##_by_hand(V *p, const V *q, unsigned a, int n) { body<V, true>(p, q, a, n); }
extern "C" {
KERNELS(store16, ugk::u32x4)
KERNELS(store8, u32x2)
KERNELS(store4, unsigned int)
}
"""


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    src = tmp_path_factory.mktemp("device_code") / "store.hip"
    src.write_text(SOURCE)
    cmd = [build.hipcc_path()] + build.HIPCC_FLAGS + ["--cuda-device-only", "-S", "-I", build.INCLUDE, "-I", build.CSRC, str(src),
                                                      "-o", "-"]
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True)
    assert proc.returncode == 0, proc.stderr[-3000:]
    return proc.stdout


def _wait_states_behind_the_store(text, kernel):
    body = text[text.index("\n%s:" % kernel) :]
    code = [ln.split(";")[0].split("//")[0].strip() for ln in body[: body.index("s_endpgm")].splitlines()]
    code = [ln for ln in code if ln and not ln.endswith(":") and not ln.startswith(".")]
    store = [i for i, ln in enumerate(code) if ln.startswith("global_store_dword")]
    assert len(store) == 1, code
    states = 0
    for ln in code[store[0] + 1 :]:
        nop = re.match(r"s_nop (\d+)", ln)
        states += int(nop.group(1)) + 1 if nop else 1
        if ln.startswith("v_"):
            return states - 1
    raise AssertionError(code)


@pytest.mark.parametrize("kernel", ["store16", "store8", "store4"])
def test_a_written_through_store_leaves_its_data_as_long_as_the_compiler_does(assembly, kernel):
    want = _wait_states_behind_the_store(assembly, kernel + "_by_compiler")
    assert _wait_states_behind_the_store(assembly, kernel + "_by_hand") >= want
    assert kernel != "store16" or want == 2  # the case there is a wait for


@pytest.fixture(scope="module")
def gather_kernels():
    """name -> where the number of workgroups stands among the arguments of each kernel of ugk_gather.hip"""
    cmd = [build.hipcc_path()] + build.HIPCC_FLAGS + ["--cuda-device-only", "-S", "-I", build.INCLUDE, "-I", build.CSRC,
                                                      os.path.join(build.CSRC, "ugk_gather.hip"), "-o", "-"]
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True)
    assert proc.returncode == 0, proc.stderr[-3000:]
    found = {}
    for meta in re.findall(r"- \.agpr_count.*?\.wavefront_size: +\d+", proc.stdout, re.S):
        at = re.search(r"\.offset: +(\d+)\n +\.size: +4\n +\.value_kind: +hidden_block_count_x", meta)
        found[re.search(r"\.name: +(\S+)", meta).group(1)] = int(at.group(1)) if at else None
    return found


def test_a_gather_nobody_polls_for_has_its_arguments_in_two_lines(gather_kernels):
    """a launch's arguments are in host memory: the 48 bytes that only a polled launch needs pushed the number of workgroups,
    which stands behind the kernel's own arguments, into a third line of 64 bytes"""
    plain = {k: at for k, at in gather_kernels.items() if "Direct" in k and "StoreE2E" not in k and at is not None}
    assert len(plain) > 20
    assert max(plain.values()) < 128, max(plain, key=plain.get)


@pytest.mark.parametrize("source,kernel,words", [("ugk_partition.hip", "dedup_resolve_kernel", 1),
                                                 ("ugk_partition.hip", "dedup_small_kernel", 1),
                                                 ("ugk_refresh.hip", "rank_combine_observed_kernel", 2)])
def test_a_word_for_the_host_is_there_before_its_launch_has_ended(source, kernel, words):
    """the host reads them once a launch behind this one tells it that all is done; what is acknowledged is in host memory only if
    it was stored at system scope, as tell_host does (before optimisation: two seconds where the kernels take a minute)"""
    cmd = [build.hipcc_path()] + build.HIPCC_FLAGS + ["--cuda-device-only", "-S", "-emit-llvm", "-Xclang", "-disable-llvm-passes",
                                                      "-I", build.INCLUDE, "-I", build.CSRC, os.path.join(build.CSRC, source), "-o", "-"]
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True)
    assert proc.returncode == 0, proc.stderr[-3000:]

    def body(name):
        return re.search(r"\ndefine [^\n]*%s.*?\n}" % name, proc.stdout, re.S).group(0)

    assert len(re.findall(r"call void @\w*tell_host", body(kernel))) >= words
    assert re.search(r"store atomic i32 [^\n]* monotonic", body(r"\w*tell_hostIj"))
    assert "syncscope" not in body(r"\w*tell_hostIj")
