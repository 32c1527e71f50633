"""Loads that write LDS, as they are compiled: the distances that the hardware does not keep itself, and what m0 holds behind them."""
import re
import shutil
import subprocess

import pytest

from sharpinference_amd.csrc import build as kernel_build

SOURCE = r"""
#include "lds_loads.h"
__device__ void out_of_lds(const char* smem, int* out) {
  lds_loads_wait();
  __syncthreads();
  out[threadIdx.x] = *(const int*)(smem + threadIdx.x * 16);
}
template <bool STREAM> __device__ void fresh(const char* p, const int* o, int* out, int n) {
  __shared__ __attribute__((aligned(1024))) char smem[4096];
  u32x4 r = buffer_of(p, n);
  load_to_lds<STREAM>(r, threadIdx.x * 16, o[threadIdx.x], lds_address(smem));
  r[2] = __builtin_amdgcn_readfirstlane(o[threadIdx.x + 64]);
  load_to_lds<STREAM>(r, threadIdx.x * 16, 0, o[threadIdx.x + 128]);
  out_of_lds(smem, out);
}
__global__ void plain(const char* p, const int* o, int* out, int n) { fresh<false>(p, o, out, n); }
__global__ void streamed(const char* p, const int* o, int* out, int n) { fresh<true>(p, o, out, n); }
__global__ void kept(const char* p, int* out, int n) {
  __shared__ __attribute__((aligned(1024))) char smem[4096];
  __builtin_amdgcn_s_sendmsg(2, n);
  load_to_lds(buffer_of(p, n), threadIdx.x * 16, 0, lds_address(smem) + n * 1024);
  __builtin_amdgcn_s_sendmsg(2, n);
  out_of_lds(smem, out);
}
template <bool STREAM> __device__ void fresh_two(const char* p, const int* o, int* out, int n) {
  __shared__ __attribute__((aligned(1024))) char smem[4096];
  u32x4 r = buffer_of(p, n);
  r[2] = __builtin_amdgcn_readfirstlane(o[threadIdx.x + 64]);
  load_two_to_lds<STREAM>(r, threadIdx.x * 16, threadIdx.x * 32, o[threadIdx.x], o[threadIdx.x + 128], o[threadIdx.x + 192]);
  out_of_lds(smem, out);
}
__global__ void two_plain(const char* p, const int* o, int* out, int n) { fresh_two<false>(p, o, out, n); }
__global__ void two_streamed(const char* p, const int* o, int* out, int n) { fresh_two<true>(p, o, out, n); }
__global__ void two_alike(const char* p, int* out, int n) {
  __shared__ __attribute__((aligned(1024))) char smem[4096];
  load_two_to_lds(buffer_of(p, n), threadIdx.x * 16, threadIdx.x * 32, n, n, n + 1024);
  out_of_lds(smem, out);
}
__global__ void two_kept(const char* p, int* out, int n) {
  __shared__ __attribute__((aligned(1024))) char smem[4096];
  __builtin_amdgcn_s_sendmsg(2, n);
  load_two_to_lds(buffer_of(p, n), threadIdx.x * 16, threadIdx.x * 32, 0, lds_address(smem) + n * 1024, lds_address(smem) + n * 2048);
  __builtin_amdgcn_s_sendmsg(2, n);
  out_of_lds(smem, out);
}
"""


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """The instructions of each kernel (compiled only, never run)."""
    if not (shutil.which("hipcc") or shutil.which("/opt/rocm/bin/hipcc")):
        pytest.skip("hipcc is not installed")
    d = tmp_path_factory.mktemp("lds_loads")
    (d / "k.hip").write_text(SOURCE)
    subprocess.run([kernel_build._hipcc(), *kernel_build.HIPCC_FLAGS, "-I", kernel_build.CSRC_DIR, "--cuda-device-only", "-S", str(d / "k.hip"),
                    "-o", str(d / "k.s")], check=True, stderr=subprocess.DEVNULL)
    found, name = {}, None
    for line in (d / "k.s").read_text().splitlines():
        start = re.match(r"_Z\d+(plain|streamed|kept|two_plain|two_streamed|two_alike|two_kept)P", line)
        if start:
            name = start.group(1)
            found[name] = []
        elif name and re.match(r"\s+[svdgb][a-z]*_", line):
            found[name].append(line.split(";")[0].strip())
    return found


def scalars(text):
    """The numbers of the scalar registers named."""
    out = set()
    for a, b, c in re.findall(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b", text):
        out |= set(range(int(a), int(b) + 1)) if a else {int(c)}
    return out | ({"m0"} if re.search(r"\bm0\b", text) else set())


@pytest.mark.parametrize("name", ["plain", "streamed", "two_plain", "two_streamed"])
def test_a_load_lies_five_wait_states_behind_a_vector_write_of_what_it_reads(kernels, name):
    ins = kernels[name]
    loads = [i for i, x in enumerate(ins) if x.startswith("buffer_load") and x.endswith("lds")]
    assert len(loads) == 2 and all(("nt" in ins[i]) == ("streamed" in name) for i in loads)
    near = 0
    for i in loads:
        reads, waited = scalars(ins[i]) | {"m0"}, 0
        for x in reversed(ins[:i]):
            if x.startswith("v_read") and scalars(x.split(",")[0]) & reads:
                assert waited >= 5, (x, ins[i], waited)
                near += 1
            if re.match(r"s_mov_b32 m0\b", x):
                assert waited >= 1
            waited += int(x.split()[1]) + 1 if x.startswith("s_nop") else 1
    assert near >= 2                                       # (both loads read what a lane gave)


@pytest.mark.parametrize("name", ["two_plain", "two_streamed", "two_alike", "two_kept"])
def test_two_loads_have_a_place_each(kernels, name):
    """m0 is written between them and one wait state passes; nothing else that the second one reads lies in it."""
    ins = kernels[name]
    first, second = [i for i, x in enumerate(ins) if x.endswith("lds")]
    between = [x for x in ins[first + 1:second]]
    assert re.match(r"s_mov_b32 m0, s\d+$", between[0]) and between[1:] == ["s_nop 0"]
    assert "m0" not in scalars(ins[first]) | scalars(ins[second])


@pytest.mark.parametrize("name", ["kept", "two_kept"])
def test_m0_is_set_again_behind_a_load_for_who_kept_a_value_there(kernels, name):
    ins = kernels[name]
    load = [i for i, x in enumerate(ins) if x.endswith("lds")][-1]
    first, second = [i for i, x in enumerate(ins) if x.startswith("s_sendmsg")]
    writes = [i for i, x in enumerate(ins) if re.match(r"s_\w+ m0\b", x)]
    assert first < load < second and any(load < i < second for i in writes)
    held = lambda at: ins[max(i for i in writes if i < at)].split(", ", 1)[1]
    assert held(first) == held(second) != held(load)
