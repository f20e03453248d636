"""The hand-written copies from memory to LDS, in the assembly that the compiler makes around them.  It does not look into them: m0 has
to be an operand that it writes for each, and their base must not need wait states, which it would not put in front of them."""
import os
import re
import shutil
import subprocess

import pytest

from clusterfusionplus_amd import build

PROBE = r"""
#include <hip/hip_runtime.h>
#include "seq_device.hpp"
using namespace cfpp;
// a base that a vector instruction has just written
__global__ void probe_base(const char* p, const int* at) {
    extern __shared__ __align__(1024) char lds[];
    copy_to_lds16_at(threadIdx.x * 16, uniform(p + at[threadIdx.x]), lds_address(lds));
    copy_to_lds16_once(threadIdx.x * 16, uniform(p + at[threadIdx.x + 64]), lds_address(lds));
}
// copies between two that the compiler makes to one place in LDS
template <int KIND> __device__ void between(const char* p, char* lds) {
    copy_to_lds16(p + threadIdx.x * 16, lds);
    if (KIND == 0) copy_to_lds16_at(threadIdx.x * 16, p + 4096, lds_address(lds) + 1024);
    if (KIND == 1) copy_to_lds16_once(threadIdx.x * 16, p + 4096, lds_address(lds) + 1024);
    if (KIND == 2) copy_to_lds16_from(p + 4096 + threadIdx.x * 16, lds_address(lds) + 1024);
    copy_to_lds16(p + 8192 + threadIdx.x * 16, lds);
}
#define BETWEEN(K) __global__ void probe_m0_##K(const char* p) { extern __shared__ __align__(1024) char lds[]; between<K>(p, lds); }
BETWEEN(0)
BETWEEN(1)
BETWEEN(2)
"""


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Name -> instructions, one per line, of every kernel of the probe."""
    hipcc = os.path.join(build.ROCM, "bin", "hipcc")
    if shutil.which(hipcc) is None:
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("copies")
    (d / "probe.hip").write_text(PROBE)
    flags = [f for f in build.SEQ_FLAGS if f != "-shared" and not f.startswith("-Wl,")]
    res = subprocess.run([hipcc, *flags, f"-I{build.INCLUDE}", f"-I{build.CSRC}", "--cuda-device-only", "-S", str(d / "probe.hip"), "-o", str(d / "probe.s")],
                         stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert res.returncode == 0, res.stdout
    out, name = {}, None
    for line in (d / "probe.s").read_text().splitlines():
        label = re.match(r"_Z\d+(probe_\w+?)(?:PK\w*)?:", line)
        if label:
            name = label[1]
            out[name] = []
        text = line.split(";")[0].strip()
        if name and text and not text.endswith(":") and not text.startswith("."):
            out[name].append(text)
            if text.startswith("s_endpgm"):
                name = None
    return out


def scalars(text):
    """Numbers of the scalar registers in a list of operands."""
    found = {int(m) for m in re.findall(r"(?<![\w\[:])s(\d+)\b", text)}
    for lo, hi in re.findall(r"\bs\[(\d+):(\d+)\]", text):
        found |= set(range(int(lo), int(hi) + 1))
    return found


def too_early(code):
    """(wait states, writing, reading) of the copies that read a scalar register less than five wait states after a vector instruction
    has written it.  Instructions in the order of their addresses: a branch in between would add states."""
    found = []
    for i, text in enumerate(code):
        if not text.startswith("global_load_lds"):
            continue
        wanted, states = scalars(text), 0
        for t in reversed(code[max(0, i - 5):i]):
            if states >= 5 or not wanted:
                break
            op, _, operands = t.partition(" ")
            written = scalars(operands.split(",")[0])
            if op.startswith("v_") and written & wanted:
                found.append((states, t, text))
            if op.startswith("s_") and op not in ("s_nop", "s_waitcnt"):
                wanted -= written            # (a scalar instruction waits for vector results, and its own can be read at once)
            states += int(operands, 0) + 1 if op == "s_nop" else 1
    return found


def test_scalar_base_from_a_vector_instruction(kernels):
    code = kernels["probe_base"]
    assert sum(t.startswith("global_load_lds_dwordx4") for t in code) == 2 and any(t.startswith("v_readfirstlane") for t in code)
    assert too_early(code) == []


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    """Name -> instructions of every kernel of the built library, in the order of their addresses."""
    objdump = os.path.join(build.ROCM, "lib", "llvm", "bin", "llvm-objdump")
    if shutil.which(objdump) is None:
        pytest.skip("no llvm-objdump")
    build.ensure_seq()
    d = tmp_path_factory.mktemp("library")
    lib = shutil.copy(build.SEQ_LIB, d)
    subprocess.run([objdump, "--offloading", lib], cwd=d, check=True, stdout=subprocess.DEVNULL)
    device, = d.glob("*gfx950")
    text = subprocess.run([objdump, "-d", "--no-show-raw-insn", str(device)], check=True, stdout=subprocess.PIPE, text=True).stdout
    out = {}
    for part in re.split(r"\n(?=[0-9a-f]+ <)", text):
        name = re.match(r"[0-9a-f]+ <(.*)>:", part)
        if name:
            out[name[1]] = [line.split("//")[0].strip() for line in part.splitlines()[1:] if line.startswith("\t")]
    return out


def test_no_copy_of_the_library_reads_its_base_too_early(library):
    code = [t for kernel in library.values() for t in kernel]
    assert sum(t.startswith("global_load_lds_dwordx4") for t in code) > 1000
    assert too_early(code) == []


def test_rings_step_on_without_a_jump(library):
    """Between the last copy of a step's request and the step's first read of LDS there is no branch, in any of the products with a ring."""
    rings = {name: code for name, code in library.items() if "k_seq_gemmI" in name}
    assert len(rings) > 50
    for name, code in rings.items():
        read = next(i for i, t in enumerate(code) if t.startswith("ds_read_b128"))
        copy = max(i for i in range(read) if code[i].startswith("global_load_lds_dwordx4"))
        assert [t for t in code[copy:read] if t.startswith(("s_branch", "s_cbranch"))] == [], name


def test_products_of_attention_have_their_reads_in_flight(library):
    """No product of a portion's attention waits for every read of LDS, but where a phase begins or ends."""
    kernels = {name: code for name, code in library.items() if re.search(r"k_seq_attnI", name)}
    assert len(kernels) == 24
    for name, code in kernels.items():
        products = [i for i, t in enumerate(code) if t.startswith("v_mfma")]
        waits = [i for i in products if any(re.match(r"s_waitcnt.*lgkmcnt\(0\)", t) for t in code[i - 2:i])]
        assert len(products) >= 24 and len(waits) <= 8, (name, len(products), len(waits))


@pytest.mark.parametrize("kind", [0, 1, 2], ids=["at", "once", "from"])
def test_compiler_knows_that_m0_is_written(kernels, kind):
    """Every copy is preceded by a write of m0 of its own, and at least one instruction lies between them."""
    last, copies = None, 0
    for i, t in enumerate(kernels[f"probe_m0_{kind}"]):
        if re.match(r"s_\w+ m0,", t):
            last = i
        if t.startswith("global_load_lds_dwordx4"):
            copies += 1
            assert last is not None and i - last >= 2, (copies, t)
            last = None
    assert copies == 3
