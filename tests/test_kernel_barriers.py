"""Barriers between a K loop's copies into LDS and an epilogue that uses the same bytes, read from the machine code of the built
library: a wave that runs ahead would spoil what a slower one still copies or reads, in a window so short that results seldom show it."""
import os
import re
import subprocess

import pytest

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
# <activation, scale order, streaming hint, int4, per-channel, token fragments, row-major>: 160 tokens of int4 weights with K-group
# scales, fused first stage; the row scales of its K loop lie where the epilogue exchanges maxima
KERNEL = "_ZN2lo20moe_gemm_t128_kernelILi1ELi{order}ELb1ELb1ELb0ELi10ELb0EEEvNS_8GemmArgsEii"


@pytest.fixture(scope="module")
def code_object(tmp_path_factory):
    from lightop_amd import _lib

    if not (os.path.exists(_lib.LIB_PATH) and os.path.exists(OBJDUMP) and os.path.exists(READELF)):
        pytest.skip("needs the built library and ROCm's llvm-objdump")
    d = tmp_path_factory.mktemp("code")
    os.symlink(os.path.abspath(_lib.LIB_PATH), d / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=d, check=True, capture_output=True)
    for name in sorted(os.listdir(d)):
        if "gfx950" in name and KERNEL.format(order=2) in subprocess.run([READELF, "-sW", name], cwd=d, check=True,
                                                                         capture_output=True, text=True).stdout:
            return d / name
    raise AssertionError("no code object holds the kernel")


def control_flow(path, symbol):
    """[(mnemonic, operands, successors)] of a kernel."""
    text = subprocess.run([OBJDUMP, "-d", f"--disassemble-symbols={symbol}", path], check=True, capture_output=True, text=True).stdout
    code, at = [], {}
    for line in text.splitlines():
        m = re.match(r"\s+(\S+)\s*(.*?)\s*// ([0-9A-F]{12}):", line)
        if m:
            target = re.search(r"<\S+\+0x([0-9a-f]+)>\s*$", line)
            at[int(m[3], 16)] = len(code)
            code.append((m[1], m[2], int(target[1], 16) if target else None))
    first = min(at)
    out = []
    for i, (op, args, target) in enumerate(code):
        assert not op.startswith(("s_setpc", "s_swappc")), "a branch whose target is not in the text"
        nxt = [] if op in ("s_endpgm", "s_branch") else [i + 1]
        if op.startswith(("s_branch", "s_cbranch")):
            nxt.append(at[first + target])
        out.append((op, args, [n for n in nxt if n < len(code)]))
    return out


@pytest.mark.parametrize("order", [2, 0, 1], ids=["contracted", "separate", "fused scale"])
def test_epilogue_waits_for_the_row_scales(code_object, order):
    flow = control_flow(code_object, KERNEL.format(order=order))
    is_copy = [op == "buffer_load_dword" and args.endswith("lds") for op, args, _ in flow]
    before = [[] for _ in flow]
    for i, (_, _, nxt) in enumerate(flow):
        for n in nxt:
            before[n].append(i)

    def reach(start, edges, stop):
        seen, todo = set(), list(start)
        while todo:
            for n in edges(todo.pop()):
                if n not in seen:
                    seen.add(n)
                    if not stop(n):
                        todo.append(n)
        return seen

    matrix = [i for i, (op, _, _) in enumerate(flow) if op.startswith("v_mfma")]
    k_loop = reach(matrix, lambda i: before[i], lambda n: False) | set(matrix)  # (with the start: all that an MFMA can follow)
    copies = [i for i, c in enumerate(is_copy) if c]
    assert len(copies) >= 5 and matrix  # the first K block's and one in each variant of the K loop
    unmet = reach(copies, lambda i: flow[i][2], lambda n: flow[n][0] == "s_barrier")
    stores = [i for i in unmet if i not in k_loop and flow[i][0].startswith("ds_write")]
    assert any(flow[i][0].startswith("ds_write") for i in range(len(flow)) if i not in k_loop)
    assert not stores, [flow[i][:2] for i in stores[:4]]
