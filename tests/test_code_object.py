"""What the compiler made of the kernels, from the notes of the built library: no GPU is needed."""
import os
import re
import shutil
import subprocess

import pytest

import abi

LLVM = os.path.join(os.environ.get("ROCM_HOME", "/opt/rocm"), "llvm", "bin")


@pytest.fixture(scope="module")
def code_object(tmp_path_factory):
    """The gfx950 code object of the built library."""
    where = tmp_path_factory.mktemp("code")
    lib = shutil.copy(abi.LIB_PATH, where)
    subprocess.check_call([os.path.join(LLVM, "llvm-objdump"), "--offloading", lib], stdout=subprocess.DEVNULL)
    (found,) = where.glob("*gfx950*")
    return found


@pytest.fixture(scope="module")
def notes(code_object):
    """{kernel: {template arguments: {note: number}}}"""
    text = subprocess.check_output([os.path.join(LLVM, "llvm-readelf"), "--notes", str(code_object)]).decode()
    out = {}
    for part in re.split(r"^ +- \.a", text, flags=re.M)[1:]:  # a kernel's notes begin with .agpr_count
        name = re.search(r"\.name: +_ZN12_GLOBAL__N_1\d+(fmha_\w+?_kernel)I((?:L[ib]\d+E)+)E", part)
        if name:
            key = tuple(int(x) for x in re.findall(r"L[ib](\d+)E", name.group(2)))
            out.setdefault(name.group(1), {})[key] = {k: int(v) for k, v in re.findall(r"\.(\w+): +(\d+)$", part, flags=re.M)}
    return out


def test_last_rows_of_slices_cost_the_128_query_forward_no_registers(notes):
    """The variants with work groups for the last rows of slices spill what those without them spill: nothing at D = 64,
    three vector registers at D = 128."""
    kernels = notes["fmha_fwd_pipe_kernel"]
    assert len(kernels) == 12  # D, causal, odd slots first (without a mask), last rows
    for (d, causal, odd_first, tail), own in kernels.items():
        spilled = {k: own[k] for k in ("sgpr_spill_count", "vgpr_spill_count", "private_segment_fixed_size")}
        assert spilled == {"sgpr_spill_count": 0, "vgpr_spill_count": 3 if d == 128 else 0,
                           "private_segment_fixed_size": 16 if d == 128 else 0}, (d, causal, odd_first, tail)


def test_where_the_loop_of_the_128_query_forward_lies(code_object):
    """The nops in front of its main loop put it where it was timed as the fastest: its first barrier is 16 bytes past a
    32-byte line at D = 128, 8 at D = 64, in every variant without work groups for last rows."""
    text = subprocess.check_output([os.path.join(LLVM, "llvm-objdump"), "-d", "--no-show-raw-insn", str(code_object)]).decode()
    places = {}
    for part in re.split(r"^[0-9a-f]+ <", text, flags=re.M):
        name = re.match(r"_ZN12_GLOBAL__N_120fmha_fwd_pipe_kernelI((?:L[ib]\d+E)+)E", part)
        if not name:
            continue
        d, causal, odd_first, tail = (int(x) for x in re.findall(r"L[ib](\d+)E", name.group(1)))
        code = [(what.strip(), int(at, 16)) for what, at in re.findall(r"^\s+(.*?)\s*// *([0-9A-F]+):", part, flags=re.M)]
        names = " ".join(what.split()[0] + ("0" if what == "s_nop 0" else "") for what, _ in code).split(" ")
        nops = next(i for i in range(len(names)) if names[i:i + 4] == ["s_nop0"] * 4)
        if not tail:
            places[d, causal, odd_first] = code[names.index("s_barrier", nops)][1] % 32
    assert len(places) == 6
    assert places == {key: 16 if key[0] == 128 else 8 for key in places}
