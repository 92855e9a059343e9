"""The loads from memory straight to LDS (csrc/qh_lds.hpp) are inline assembly,
which the compiler's hazard pass does not look into: an SGPR written by a
vector instruction needs 5 wait states before a vector-memory instruction reads
it.  The distances are counted in the assembly that the compiler makes for
gfx950 (no GPU needed), over every path that leads to a load: for a kernel that
uses a descriptor right where it is made, and for the library's kernels.
"""
import re
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "project-ia_amd" / "csrc"
HIPCC = Path("/opt/rocm/bin/hipcc")
WAIT = 5

KERNEL = """
#include "qh_lds.hpp"
extern "C" __global__ void k(const uint8_t* p, const uint32_t* at, float* o) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[1024];
    const qh::rsrc_v r = qh::make_rsrc(p + at[threadIdx.x], 4096u);
    qh::LOAD(r, threadIdx.x * 16u, 0u, qh::lds_address(lds));
    qh::wait_vm<0>();
    o[threadIdx.x] = reinterpret_cast<const float*>(lds)[threadIdx.x];
}
"""


def assembly(src, out):
    if not HIPCC.exists():
        pytest.skip("no hipcc in this image")
    r = subprocess.run([str(HIPCC), "-O3", "-std=c++17", "-ffp-contract=off", "--offload-arch=gfx950", "--cuda-device-only", "-S",
                        "-I", str(CSRC), "-I", str(CSRC.parent.parent / "include"), "-Xclang", "-target-feature", "-Xclang",
                        "-packed-fp32-ops", str(src), "-o", str(out)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    assert "reserved register" not in r.stderr
    return out.read_text()


def sgprs(text):
    out = {int(m) for m in re.findall(r"\bs(\d+)\b", text)}
    for a, b in re.findall(r"\bs\[(\d+):(\d+)\]", text):
        out |= set(range(int(a), int(b) + 1))
    return out


def vector_writes(ins):
    """SGPRs that a vector instruction writes (its scalar destinations)."""
    if not ins.startswith("v_"):
        return set()
    op, _, args = ins.partition(" ")
    args = args.split(",")
    return sgprs(args[0]) | (sgprs(args[1]) if re.match(r"v_(add|sub|subrev|addc|subb|subbrev)_co|v_div_scale|v_mad_[iu]64", op) else set())


def check_loads(text):
    """(loads to LDS, nearest vector write of one of their SGPRs in wait states)."""
    ins, label = [], {}
    for line in text.splitlines():
        line = line.split(";")[0].rstrip()
        m = re.match(r"([.\w$]+):$", line)
        if m:
            label[m[1]] = len(ins)
        elif line.strip() and not line.strip().startswith("."):
            ins.append(re.sub(r"\s+", " ", line.strip()))
    before = [[] for _ in range(len(ins) + 1)]
    for i, s in enumerate(ins):
        if s.startswith(("s_branch", "s_cbranch")):
            before[label[s.split()[1]]].append(i)
        if not s.startswith(("s_branch", "s_endpgm")):
            before[i + 1].append(i)
    loads = [i for i, s in enumerate(ins) if s.startswith("buffer_load") and s.endswith("lds")]
    nearest = WAIT
    for i in loads:
        want, todo, seen = sgprs(ins[i]), [(j, 0) for j in before[i]], set()
        while todo:
            j, waited = todo.pop()
            if waited >= WAIT or (j, waited) in seen:
                continue
            seen.add((j, waited))
            if vector_writes(ins[j]) & want:
                nearest = min(nearest, waited)
            step = int(ins[j].split()[1], 0) + 1 if ins[j].startswith("s_nop") else 1
            todo += [(k, waited + step) for k in before[j]]
    return len(loads), nearest


@pytest.mark.parametrize("load", ["lds_load16", "lds_load4"])
def test_descriptor_wait_states(tmp_path, load):
    src = tmp_path / "k.hip"
    src.write_text(KERNEL.replace("LOAD", load))
    loads, nearest = check_loads(assembly(src, tmp_path / "k.s"))
    assert loads == 1 and nearest >= WAIT


@pytest.mark.parametrize("source", ["k_gemm.hip", "k_prefill.hip"])
def test_kernels_wait_states(tmp_path, source):
    loads, nearest = check_loads(assembly(CSRC / source, tmp_path / "k.s"))
    assert loads > 0 and nearest >= WAIT
