"""Registers of the built kernels, from the metadata of the library's own code objects: what a kernel keeps over its main loop
fits its registers, and none spills that did not by design."""
import os
import re
import struct
import subprocess
import tempfile

import pytest

from nvllm_amd import capi

READELF = "/opt/rocm/llvm/bin/llvm-readelf"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"

# kernels that fill every register and spill some: at most these many of them
SPILLS = {
    "k_gemm_waves<6, 9, float, OpBf16>": 8,
    "k_gemm_waves<7, 9, float, OpBf16>": 60,
    "k_gemm_prefill<4, 1, 9, float, 2, 4, OpBf16, false, false>": 36,
    "k_window_attn<8, 16, 1, true, 2, false>": 14,
    "k_lightning_out<8>": 131,
}
# and kernels whose next step's operands live in registers across this one's: at most these many registers
REGISTERS = {
    "k_decode_chain<ChainShape<2, 1, 4, 2, 1, 4, 4, 2, 4, 2, 1, 4, 64, __half>>": 192,
    "k_decode_chain<ChainShape<2, 2, 8, 2, 1, 8, 6, 2, 4, 4, 2, 4, 64, __half>>": 240,
}


def kernels():
    """name -> (vector registers, spilled ones, bytes of scratch) of every kernel of the library"""
    with open(capi.HIP_LIB, "rb") as f:
        data = f.read()
    names, values = [], []
    at = data.find(MAGIC)
    while at >= 0:
        entry = at + len(MAGIC) + 8
        for _ in range(struct.unpack_from("<Q", data, at + len(MAGIC))[0]):
            offset, size, length = struct.unpack_from("<QQQ", data, entry)
            target = data[entry + 24:entry + 24 + length].decode()
            entry += 24 + length
            if "gfx950" not in target or not size:
                continue
            with tempfile.NamedTemporaryFile(suffix=".co") as code:
                code.write(data[at + offset:at + offset + size])
                code.flush()
                notes = subprocess.check_output([READELF, "--notes", code.name], text=True)
            for k in re.split(r"\n  - \.agpr_count:", notes)[1:]:
                names.append(re.search(r"\.name: +(\S+)", k)[1])
                values.append(tuple(int(re.search(r"\.%s: +(\d+)" % key, k)[1]) for key in ("vgpr_count", "vgpr_spill_count", "private_segment_fixed_size")))
        at = data.find(MAGIC, at + 1)
    plain = subprocess.run(["c++filt"], input="\n".join(names), capture_output=True, text=True, check=True).stdout.split("\n")
    tidy = [re.sub(r"nvllm::|\(anonymous namespace\)::|^void ", "", n).replace("> >", ">>").split("(")[0] for n in plain]
    return dict(zip(tidy, values))


@pytest.fixture(scope="module")
def usage():
    if not os.path.exists(READELF):
        pytest.skip("no %s here" % READELF)
    return kernels()


def test_no_kernel_spills_that_did_not(usage):
    assert len(usage) > 300
    over = {n: v for n, v in usage.items() if v[1] > SPILLS.get(n, 0) or (v[2] and n not in SPILLS)}
    assert not over


def test_registers_of_the_one_launch_step(usage):
    for name, most in REGISTERS.items():
        assert usage[name][0] <= most, (name, usage[name])
