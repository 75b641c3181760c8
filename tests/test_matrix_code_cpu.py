"""The library's own machine code: matrix instructions ignore the mask of active lanes, so none may stand where a kernel
has masked lanes off for a condition.  (Where a whole wave is to skip one, only a branch does that, and the compiler may
leave the branch out: the condition has to be a scalar.)"""
import os
import re
import struct
import subprocess

import pytest

from conftest import load_pkg

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(path):
    """The gfx950 code objects that hipcc put into the library, one per source."""
    with open(path, "rb") as f:
        data = f.read()
    at = data.find(BUNDLE)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + len(BUNDLE))
        pos = at + len(BUNDLE) + 8
        for _ in range(n):
            offset, size, id_len = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + id_len]
            pos += 24 + id_len
            if b"gfx950" in name and size:
                yield data[at + offset:at + offset + size]
        at = data.find(BUNDLE, at + len(BUNDLE))


def masked_matrix_instructions(listing):
    """-> {kernel: matrix instructions between masking lanes off (s_.._saveexec) and restoring the mask}, kernels seen"""
    found, kernels, kernel, masked = {}, set(), None, False
    for line in listing:
        head = re.match(r"^[0-9a-f]+ <(\w+)>:", line)
        if head:
            kernel, masked = head.group(1), False
            continue
        words = line.split()
        if not words:
            continue
        op, dst = words[0], words[1] if len(words) > 1 else ""
        if op.endswith("_saveexec_b64"):
            masked = True
        elif op in ("s_or_b64", "s_mov_b64") and dst == "exec," or op in ("s_branch", "s_endpgm"):
            masked = False
        elif op.startswith("v_mfma"):
            kernels.add(kernel)
            if masked:
                found[kernel] = found.get(kernel, 0) + 1
    return found, kernels


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler here")
def test_no_matrix_instruction_under_a_lane_mask(tmp_path):
    found, kernels = {}, set()
    for i, code in enumerate(code_objects(load_pkg("lib").LIB_PATH)):
        path = tmp_path / f"{i}.co"
        path.write_bytes(code)
        listing = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(path)], capture_output=True,
                                 text=True, check=True).stdout.splitlines()
        bad, seen = masked_matrix_instructions(listing)
        found.update(bad)
        kernels |= seen
    for part in ("router_gemm_kernel", "grouped_gemm_kernel", "few_gemm_kernel", "tall_gemm_kernel", "attn_few_kernel",
                 "attn_few_rope_kernel", "scan_chunk_kernel"):
        assert any(part in k for k in kernels), part      # the listing was read
    assert not found, found


def test_the_scan_sees_a_masked_matrix_instruction():
    listing = ["0000000000001000 <kernel_a>:", "\tv_mfma_f32_16x16x32_bf16 v[0:3], v[4:7], v[8:11], v[0:3]",
               "\ts_and_saveexec_b64 s[4:5], vcc", "\tv_mfma_f32_16x16x32_bf16 v[0:3], v[4:7], v[8:11], v[0:3]",
               "\ts_or_b64 exec, exec, s[4:5]", "\tv_mfma_f32_16x16x32_bf16 v[0:3], v[4:7], v[8:11], v[0:3]"]
    assert masked_matrix_instructions(listing) == ({"kernel_a": 1}, {"kernel_a"})
