"""A 16-byte store reads its data registers while the next instructions issue, and
the compiler keeps those from writing them only for stores without a scalar
offset (see buf_store_so_nt).  Compiles FP64 kernels of each user of the buffer
stores to assembly and looks for a VALU write of a store's data registers within
two wait states."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
KERNELS = ("k_mhd_x<double,64,4,P5_RHS,false>(MhdXArgs<double>)", "k_p5vv<double,64,4,P5_RHS,false>(P5Args<double>)",
           "k_p5b<double,24,24,P5_RK3,true>(P5Args<double>)", "k_p5b<double,32,8,P5_RK12,false,false,4>(P5Args<double>)")


def _registers(operand):
    m = re.fullmatch(r"([va])\[(\d+):(\d+)\]", operand.strip())
    if m:
        return {(m[1], i) for i in range(int(m[2]), int(m[3]) + 1)}
    m = re.fullmatch(r"([va])(\d+)", operand.strip())
    return {(m[1], int(m[2]))} if m else set()


def overwritten_stores(lines, wait=2):
    """(16- and 12-byte stores, those whose data a VALU instruction writes within `wait` wait states)."""
    code = [s for s in (line.split(";")[0].strip() for line in lines) if s and s[0] != "." and s[-1] != ":"]
    stores, bad = 0, []
    for k, s in enumerate(code):
        m = re.match(r"(buffer|global|flat)_store_dwordx[34] (.*)", s)
        if not m:
            continue
        stores += 1
        data = _registers(m[2].split(",")[0 if m[1] == "buffer" else 1])
        waited = 0
        for t in code[k + 1:k + 1 + wait]:
            if waited >= wait:
                break
            v = re.match(r"v_(?!cmp)\S+ ([^,]+)", t)
            if v and _registers(v[1]) & data:
                bad.append(s + " | " + t)
                break
            n = re.match(r"s_nop (\d+)", t)
            waited += int(n[1]) + 1 if n else 1
    return stores, bad


def test_scan():
    store, write = "buffer_store_dwordx4 v[8:11], v38, s[8:11], s33 offen nt", "v_fma_f64 v[8:9], v[0:1], v[2:3], v[4:5]"
    assert overwritten_stores([store, write]) == (1, [store + " | " + write])
    assert overwritten_stores([store, "s_nop 0", write])[1]
    assert overwritten_stores([store, "s_nop 1", write]) == (1, [])
    assert overwritten_stores([store, "v_add_u32_e32 v7, 1, v7", "s_mov_b32 s0, 0", write]) == (1, [])


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
def test_no_store_data_is_overwritten(tmp_path):
    src, asm = tmp_path / "k.hip", tmp_path / "k.s"
    src.write_text('#include "sdns_kernels.hpp"\nnamespace sdns {\n' +
                   "".join("template __global__ void %s;\n" % k for k in KERNELS) + "}\n")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", "--cuda-device-only", "-S", "-w",
                    "-I", os.path.join(ROOT, "spectraldns_amd", "csrc"), str(src), "-o", str(asm)],
                   check=True, capture_output=True)
    stores, bad = overwritten_stores(asm.read_text().splitlines())
    assert stores >= 60
    assert not bad, bad[:4]
