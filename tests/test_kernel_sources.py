"""What the kernels' sources promise and no run shows reliably."""
import ctypes
import glob
import os
import re
import shutil
import subprocess

import pytest

from litellmengine_amd.csrc import build

SOURCES = sorted(glob.glob(os.path.join(os.path.dirname(build.__file__), "*.hip")))


@pytest.mark.parametrize("path", SOURCES, ids=os.path.basename)
def test_bare_barriers_wait_for_lds(path):
    """A bare s_barrier waits for nothing: without lgkmcnt(0) ahead of it a wavefront's reads from LDS may still be on their way
    when another one, behind the barrier, fills the buffer anew.  Every path to it has that wait (or a release fence on LDS)."""
    lines = [re.sub(r"//.*", "", line).strip() for line in open(path)]
    lines = [line for line in lines if line]
    for i, line in enumerate(lines):
        if "__builtin_amdgcn_s_barrier()" not in line or line.startswith("#"):
            continue
        before, at = [], i - 1
        while at >= 0 and re.match(r"(if|else|asm volatile\(\"s_waitcnt|__builtin_amdgcn_fence\(__ATOMIC_RELEASE)", lines[at]):
            before.append(lines[at])
            at -= 1
        waits = [w for w in before if "s_waitcnt" in w or "fence" in w]
        assert waits, f"{os.path.basename(path)}: {lines[at]} / {line}"
        assert all("lgkmcnt(0)" in w or "fence" in w for w in waits), (os.path.basename(path), waits)


def test_lds_is_asked_for_on_every_device(tmp_path):
    """A kernel that takes more than 64 KB of LDS asks for it once on each device of the process, and again after a refusal."""
    source = tmp_path / "grant.cpp"
    source.write_text(r'''
#include "lds.h"
static int device = 0, asked = 0;
static hipError_t answer = hipSuccess;
extern "C" hipError_t hipGetDevice(int* d) { return *d = device, hipSuccess; }
extern "C" hipError_t hipGetLastError() { return answer; }
extern "C" hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return ++asked, answer; }
int main() {
    std::atomic<uint64_t> one{0}, other{0};
    auto launch = [&](int on, std::atomic<uint64_t>& kernel, hipError_t says = hipSuccess) {
        device = on, asked = 0, answer = says;
        return lle_grant_lds(nullptr, 1 << 17, kernel) != says ? -1 : asked;
    };
    const int got[] = {launch(0, one), launch(0, one), launch(1, one), launch(63, one), launch(64, one), launch(64, one), launch(1, one),
                       launch(0, other, hipErrorInvalidValue), launch(0, other), launch(0, other)};
    const int want[] = {1, 0, 1, 1, 1, 1, 0, 1, 1, 0};
    for (int i = 0; i < 10; ++i)
        if (got[i] != want[i]) return i + 1;
    return 0;
}
''')
    rocm = os.path.dirname(os.path.dirname(build._hipcc()))
    program = tmp_path / "grant"
    subprocess.run([build._host_compiler(), "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{rocm}/include",
                    f"-I{os.path.dirname(build.__file__)}", str(source), "-o", str(program)], check=True)
    assert subprocess.run([str(program)]).returncode == 0
    assert not [p for p in SOURCES if re.search(r"static bool \w+ =", open(p).read())]  # (asked for once a process)


@pytest.mark.parametrize("name", [n for n, files in build.LIBRARIES.items()
                                  if any("load_into_lds(" in open(os.path.join(os.path.dirname(build.__file__), f)).read() for f in files)])
def test_loads_into_lds_wait_for_their_address(name, tmp_path):
    """Between a scalar write of M0 and a load whose target is LDS stands another instruction: the load may take the M0 before
    otherwise, and nothing in the processor sees to it (the compiler does, for what it writes itself)."""
    objdump = os.path.join(os.path.dirname(os.path.dirname(build._hipcc())), "llvm", "bin", "llvm-objdump")
    if not os.path.isfile(objdump):
        pytest.skip("no llvm-objdump")
    library = shutil.copy(build._find_built(name) or build.compile_library(name), tmp_path)
    subprocess.run([objdump, "--offloading", library], check=True, cwd=tmp_path, capture_output=True)
    code, = glob.glob(f"{library}*{build.ARCH}")
    text = subprocess.run([objdump, "-d", f"--mcpu={build.ARCH}", code], check=True, capture_output=True, text=True).stdout
    code = [line.split("//")[0].split() for line in text.splitlines() if line.startswith("\t")]
    loads = [i for i, words in enumerate(code) if "_load_lds_" in words[0]]
    assert loads
    early = [code[i - 1 : i + 1] for i in loads if code[i - 1][1:2] == ["m0,"]]
    assert not early, (len(early), early[:3])


def test_tiles_of_gate_and_up_follow_the_units_of_the_chip():
    """Which tiles take a product is a matter of rounds, so of how many CUs there are; sizes that the kernel refuses are never taken."""
    form = build.load_library("gemm_wide").lle_gemm_wide_form
    form.argtypes = [ctypes.c_int] * 4
    assert form(2048, 24576, 4096, 256) == 1 and form(262, 16384, 2048, 256) == 10 and form(262, 16384, 2048, 128) == 6
    assert [form(m, 6144, 1024, 256) for m in (129, 144, 160)] == [0, 0, 0]  # (8 % slower there)
    assert form(128, 24576, 4096, 256) == form(2048, 24576, 4090, 256) == form(2048, 24572, 4096, 256) == form(2048, 24576, 4096, 0) == 0
