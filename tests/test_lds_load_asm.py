"""The LDS load written as assembly (csrc/common.h), checked on the assembly
that the compiler makes of it: m0 is declared as overwritten, and operands that
a vector instruction has just put into scalar registers are waited for (five
wait states before a buffer load reads them; the compiler adds none inside
inline assembly)."""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
PROBE = r"""
#include "common.h"
__global__ void probe(const float* p, const int* at, float* out)
{
    __shared__ float cells[128];
    // every operand comes out of a vector register
    const int lane = threadIdx.x;
    const int off = at[lane], lds = at[lane + 64];
    const rsrc_words r = make_rsrc_words(p + at[lane + 128], (unsigned)at[lane + 192]);
    buf_load_lds(r, 4 * lane, (unsigned)off, (unsigned)(lds + (int)(size_t)(__attribute__((address_space(3))) void*)cells));
    lds_loads_done();
    __syncthreads();
    out[lane] = cells[lane];
}
"""


@pytest.fixture(scope="module")
def emitted(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("ldsasm")
    src = d / "probe.hip"
    src.write_text(PROBE)
    out = {}
    for kind, flags in (("ir", ["-emit-llvm"]), ("asm", [])):
        res = subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature",
                              "-Xclang", "-packed-fp32-ops", "-I", os.path.join(ROOT, "ct-nef_amd", "csrc"),
                              "-I", os.path.join(ROOT, "include"), "--cuda-device-only", "-S", *flags, str(src),
                              "-o", str(d / kind)], capture_output=True, text=True)
        assert res.returncode == 0, res.stderr
        out[kind] = (d / kind).read_text()
    return out


def test_m0_is_a_clobber(emitted):
    calls = [l for l in emitted["ir"].splitlines() if "offen lds" in l and "asm" in l]
    assert calls and all("~{m0}" in l for l in calls), calls


def _scalars(operand):
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", operand) or re.fullmatch(r"s(\d+)()", operand)
    return range(int(m[1]), int(m[2] or m[1]) + 1) if m else ()


def test_operands_from_vector_instructions_are_waited_for(emitted):
    at, written, seen = 0, {}, 0    # wait states so far; when a vector instruction wrote a scalar register
    for line in emitted["asm"].splitlines():
        op = line.split(";")[0].replace(",", " ").split()
        if not op or op[0].startswith(".") or op[0].endswith(":"):
            continue
        if op[0].startswith("buffer_load") and op[-1] == "lds":
            seen += 1
            for operand in op[2:4]:
                for r in _scalars(operand):
                    assert at - written.get(r, -9) > 5, f"s{r} {at - written[r] - 1} wait states before {line.strip()}"
        for r in _scalars(op[1]) if len(op) > 1 else ():
            if op[0].startswith("v_"):
                written[r] = at
            elif op[0].startswith("s_"):
                written.pop(r, None)
        at += int(op[1], 0) + 1 if op[0] == "s_nop" else 1
    assert seen and any(l.strip().startswith("v_readfirstlane") for l in emitted["asm"].splitlines())
