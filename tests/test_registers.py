"""Registers and spilled bytes of kernels where a step that made them more was measured to cost time, read from the metadata of the
built library."""
import os
import re
import struct
import subprocess

import pytest

from lightop_amd import build

READELF = "/opt/rocm/llvm/bin/llvm-readelf"


def _kernels(tmp_path):
    if not os.path.exists(build.LIB_PATH) or not os.path.exists(READELF):
        pytest.skip("no built library, or no llvm-readelf")
    data = open(build.LIB_PATH, "rb").read()
    magic, at, out = b"__CLANG_OFFLOAD_BUNDLE__", -1, {}
    while (at := data.find(magic, at + 1)) >= 0:
        p = at + len(magic)
        (count,) = struct.unpack_from("<Q", data, p)
        p += 8
        if count > 8:  # (no bundle)
            continue
        for _ in range(count):
            offset, size, name = struct.unpack_from("<QQQ", data, p)
            triple = data[p + 24 : p + 24 + name].decode()
            p += 24 + name
            if "gfx950" not in triple or not size:
                continue
            obj = tmp_path / "code.o"
            obj.write_bytes(data[at + offset : at + offset + size])
            notes = subprocess.run([READELF, "--notes", str(obj)], capture_output=True, text=True, check=True).stdout
            for k in re.split(r"\n\s*- \.a(?:gpr_count|rgs):", notes)[1:]:
                m = {f: re.search(rf"\.{f}:\s+(\S+)", k) for f in ("name", "vgpr_count", "private_segment_fixed_size")}
                if m["vgpr_count"]:
                    names = re.findall(r"\.name:\s+(_Z\S+)", k)
                    out[names[-1]] = (int(m["vgpr_count"].group(1)), int(m["private_segment_fixed_size"].group(1)))
    return out


def test_registers_and_spills(tmp_path):
    kernels = _kernels(tmp_path)
    assert len(kernels) > 200
    # first kernel of few tokens, int4 weights with K-group scales: one token 27.5 us with 20 bytes, 28.5 with 36
    dec = {n: k for n, k in kernels.items() if re.match(r"_ZN2lo16dec_gemm1_kernelILi4ELb1ELb0E", n)}
    assert dec and all(spilled <= 20 for _, spilled in dec.values()), dec
    # weight-streaming first stage of 16-token blocks, int8 in its load-time layout: past 128 registers one workgroup to a CU instead
    # of two (24 tokens of the DeepSeek-V3 share in the separate order 120.0 -> 123.0 us)
    ws = {n: k for n, k in kernels.items() if re.match(r"_ZN2lo18moe_gemm_ws_kernelILi1ELi1ELi[012]ELb1ELi8ELi4ELi2ELb0ELb0E", n)}
    assert len(ws) >= 3 and all(v <= 128 and not spilled for v, spilled in ws.values()), ws
