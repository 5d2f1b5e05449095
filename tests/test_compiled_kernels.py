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


KEEP = re.compile(r"^\s*(ds_write|s_barrier|s_waitcnt|global_load_lds|\S+\s+m0,)")


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """{symbol: [(position, opcode, operands), ...]}, the instructions that the tests below ask for"""
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    out = {}
    for which in (capi.LIB_PATH, os.path.join(os.path.dirname(capi.LIB_PATH), "libmi355ceilings.so")):
        lib = shutil.copy(which, tmp_path_factory.mktemp("code"))
        subprocess.run([OBJDUMP, "--offloading", lib], check=True, stdout=subprocess.DEVNULL)
        for obj in sorted(glob.glob(lib + ".*gfx950")):
            text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", obj], check=True, stdout=subprocess.PIPE, text=True).stdout
            code = None
            for at, line in enumerate(text.splitlines()):
                if line.startswith("<"):
                    code = out.setdefault(line.strip("<>: \n"), [])
                elif code is not None and KEEP.match(line):
                    op, _, rest = line.split("//")[0].strip().partition(" ")
                    code.append((at, op, [a.strip() for a in rest.split(",")]))
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
        barrier = next(i for i, (_, op, _) in enumerate(code) if op == "s_barrier")
        writes = [i for i in range(barrier) if code[i][1].startswith("ds_write")]
        assert writes, name
        assert any(op == "s_waitcnt" and "lgkmcnt(0)" in " ".join(args) for _, op, args in code[writes[-1]:barrier]), name
    assert seen >= 3


def test_a_load_to_lds_keeps_its_distance_from_the_write_of_m0(kernels):
    """Loads to LDS take their destination from M0 and need one instruction between its write and themselves."""
    seen = 0
    for name, code in kernels.items():
        for (a, _, args), (b, op, _) in zip(code, code[1:]):
            if op.startswith("global_load_lds"):
                seen += 1
                assert not (args[0] == "m0" and b == a + 1), name
    assert seen > 1000
