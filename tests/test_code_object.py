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
