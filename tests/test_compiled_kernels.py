"""What the instructions of the built kernels have to keep to where inline assembly writes them: the compiler neither counts an access
that such a block makes nor separates it from the instructions in front of it. Read from the library's own gfx950 code objects."""
import glob
import os
import re
import shutil
import subprocess

import pytest

from computelibrary_amd import capi

OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{symbol: [(opcode, operands), ...]}"""
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    d = tmp_path_factory.mktemp("code")
    lib = shutil.copy(capi.LIB_PATH, d)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, stdout=subprocess.DEVNULL)
    out, code = {}, None
    for obj in sorted(glob.glob(lib + ".*gfx950")):
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", obj], check=True, stdout=subprocess.PIPE, text=True).stdout
        for line in text.splitlines():
            line = line.split("//")[0]
            if line.startswith("<"):
                code = out.setdefault(line.strip("<>: \n"), [])
            elif code is not None and line.strip():
                op, _, rest = line.strip().partition(" ")
                code.append((op, [a.strip() for a in rest.split(",")]))
    assert out
    return out


def test_convolutions_wait_for_their_padding_before_they_publish_it(kernels):
    """The convolution's loader writes padding to LDS itself (ds_write_b128); other waves read it behind the next barrier, which waits
    for nothing by itself: between such a write and a barrier stands a wait that leaves no LDS access open."""
    seen = 0
    for name, code in kernels.items():
        if not re.search(r"gemm_ring_kernel.*Li1EEEv", name):  # (the last template argument: RING_CONV)
            continue
        seen += 1
        at = next(i for i, (op, _) in enumerate(code) if op == "s_barrier")
        writes = [i for i in range(at) if code[i][0].startswith("ds_write")]
        assert writes, name
        waits = [i for i in range(writes[-1], at) if code[i][0] == "s_waitcnt" and "lgkmcnt(0)" in " ".join(code[i][1])]
        assert waits and not any(code[i][0].startswith("ds_write") for i in range(waits[-1], at)), name
    assert seen >= 3
