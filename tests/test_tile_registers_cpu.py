"""The sums of csrc/tile_gemm.hip live in accumulation registers that asm
statements name and the compiler believes unused between them: in what was
built, nothing but those statements may touch one."""

import re
import shutil
import struct
import subprocess

import pytest

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
OBJDUMP = shutil.which("llvm-objdump") or shutil.which(
    "llvm-objdump", path="/opt/rocm/llvm/bin")


def _code_objects(path):
    """The gfx950 code objects that a module carries."""
    data = open(path, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        pos = at + len(MAGIC)
        count, = struct.unpack_from("<Q", data, pos)
        pos += 8
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", data, pos)
            name = data[pos + 24:pos + 24 + n]
            pos += 24 + n
            if b"gfx950" in name:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, at + 1)


def _misused(lines):
    """(lines that use an accumulation register in another way, counts of
    the allowed ones)."""
    bad, counts = [], {"add": 0, "zero": 0, "get": 0}
    for line in lines:
        ins = line.split("//")[0].strip()
        if not re.search(r"\ba(\d+\b|\[\d)", ins):
            continue
        m = re.fullmatch(r"v_mfma_f32_16x16x32_bf16 a\[(\d+):(\d+)\], "
                         r"v\[[\d:]+\], v\[[\d:]+\], a\[(\d+):(\d+)\]", ins)
        if m and m[1] == m[3] and m[2] == m[4] and int(m[1]) % 4 == 0:
            counts["add"] += 1
        elif re.fullmatch(r"v_accvgpr_write_b32 a\d+, 0", ins):
            counts["zero"] += 1
        elif re.fullmatch(r"v_accvgpr_read_b32 v\d+, a\d+", ins):
            counts["get"] += 1
        else:
            bad.append(ins)
    return bad, counts


def test_what_counts_as_misuse():
    fine = ["v_mfma_f32_16x16x32_bf16 a[4:7], v[0:3], v[8:11], a[4:7] // x",
            "v_accvgpr_write_b32 a255, 0", "v_accvgpr_read_b32 v3, a17",
            "v_add_u32_e32 v1, v2, v3", "s_waitcnt vmcnt(8)"]
    assert _misused(fine) == ([], {"add": 1, "zero": 1, "get": 1})
    for ins in ("v_accvgpr_write_b32 a3, v7", "ds_read_b128 a[0:3], v1",
                "v_accvgpr_mov_b32 a1, a2", "global_load_dword a9, v[0:1], off",
                "v_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[8:11], a[4:7]"):
        assert _misused([ins])[0] == [ins]


@pytest.mark.parametrize("module", ["_kernels", "_kernels_seq"])
def test_built_kernels(module, tmp_path):
    import glob
    import os
    import gllm_amd
    path = glob.glob(os.path.join(os.path.dirname(gllm_amd.__file__),
                                  module + ".cpython*.so"))
    if not path or OBJDUMP is None:
        pytest.skip("not built, or no llvm-objdump")
    kernels = 0
    for code in _code_objects(path[0]):
        if b"tile_gemm_kernel" not in code:
            continue
        obj = tmp_path / "code.o"
        obj.write_bytes(code)
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(obj)],
                              capture_output=True, text=True, check=True)
        for part in re.split(r"\n(?=[0-9a-f]+ <)", text.stdout):
            if "tile_gemm_kernel" not in part.split("\n")[0]:
                continue
            bad, counts = _misused(part.split("\n")[1:])
            assert not bad, bad[:5]
            # 64 and 32 sums of four registers, in both halves of a step
            # (which the compiler may repeat)
            assert counts["zero"] % (4 * 96) == 0 < counts["zero"]
            assert counts["add"] % (2 * 96) == 0 < counts["add"]
            assert counts["get"] % (4 * 96) == 0 < counts["get"]
            kernels += 1
    assert kernels >= 10
