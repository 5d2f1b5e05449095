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


KEEP = re.compile(r"^\s*(ds_write|s_barrier|s_waitcnt|s_nop|global_|buffer_|flat_|v_readlane|v_readfirstlane|v_cmp_\S+\s+s\[|\S+\s+m0,)")
MOST = 5  # wait states that a load needs behind a vector instruction which wrote its scalar address


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


def scalars(operand):
    m = re.match(r"s\[(\d+):(\d+)\]$|s(\d+)$", operand.split(" ")[0])
    return set() if m is None else {int(m[3])} if m[3] else set(range(int(m[1]), int(m[2]) + 1))


def test_a_load_keeps_its_distance_from_a_vector_write_of_its_address(kernels):
    """v_readlane (a spilled scalar that comes back), v_readfirstlane and compares write scalar registers; a memory instruction that reads
    one needs five wait states in between (an instruction is one, s_nop n is n + 1)."""
    for name, code in kernels.items():
        written = []  # (position, wait states that s_nop adds up to there, registers)
        nops = 0
        for at, op, args in code:
            if op == "s_nop":
                nops += int(args[0])
            elif op.startswith(("v_read", "v_cmp")):
                written = [w for w in written if at - w[0] <= MOST] + [(at, nops, scalars(args[0]))]
            elif op.startswith(("global_", "buffer_", "flat_")):
                read = set().union(*(scalars(a) for a in args))
                for pos, n, regs in written:
                    assert not (regs & read) or at - pos - 1 + nops - n >= MOST, (name, op, args)
