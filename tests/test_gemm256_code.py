"""The products of the 256 x 256 tiles are text to the compiler (gemm256.h): it may neither read nor move a sum between the first product and the wait behind the
last one, because it does not know how long a product takes.  Looked up in the code that was built."""
import os
import shutil
import struct
import subprocess

import pytest

OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data):
    at = data.find(MAGIC)
    while at >= 0:
        (n,), p = struct.unpack_from("<Q", data, at + len(MAGIC)), at + len(MAGIC) + 8
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + length]:
                yield data[at + off:at + off + size]
            p += 24 + length
        at = data.find(MAGIC, at + 1)


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_sums_stay_in_their_registers_between_products(built_libs, tmp_path):
    name = b"mfma_gemm256_kernelILb"
    code = [c for c in _code_objects(open(built_libs[0], "rb").read()) if name in c]
    assert len(code) == 1
    path = tmp_path / "code.elf"
    path.write_bytes(code[0])
    text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", str(path)], stdout=subprocess.PIPE, check=True, text=True).stdout
    kernels = [k for k in text.split("\n\n") if name.decode() in k.lstrip().split("\n")[0]]
    assert len(kernels) == 5
    for k in kernels:
        lines = [line.split("//")[0].strip() for line in k.split("\n")]
        product = [i for i, line in enumerate(lines) if line.startswith("v_mfma_f32_16x16x32_bf16")]
        wait = [i for i, line in enumerate(lines) if line.startswith("s_nop 15")]
        assert len(product) == 512 and wait[-1] > product[-1]
        assert not [line for line in lines[product[0]:wait[-1]] if "accvgpr" in line]
