"""Where the time loop of the forward kernel with helpers lies against the instruction fetch, in the machine code of the library as built:
its step depends on it (recurrent_fwd_xcd.hpp), and what places it there are five s_nop ahead of code that the compiler writes."""
import os
import subprocess

import pytest

from fastlstm_amd import _lib
from test_mfma_wait_states import OBJDUMP, code_objects, parse

KERNEL = "lstm_fwd_xcd_kernelIDF16%sLi8ELi8ELi1ELi8ELb1EE"


@pytest.mark.parametrize("dtype", ["_", "b"])
def test_time_loop_of_the_forward_kernel_with_helpers(dtype, tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no disassembler")
    name, found = KERNEL % dtype, []
    for blob in code_objects(_lib.LIB_PATH, str(tmp_path)):
        if name.encode() not in blob:
            continue
        path = os.path.join(str(tmp_path), "co")
        open(path, "wb").write(blob)
        text = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", path], check=True, capture_output=True, text=True).stdout
        for fn, code in parse(text.splitlines()).items():
            if name not in fn:
                continue
            start = [code[k + 5][0] for k in range(len(code) - 5) if code[k][0] % 64 == 0 and all(ins[1].strip() == "s_nop 0" for ins in code[k:k + 5])]
            assert len(start) == 1, fn
            loops = [(ins[0] - ins[7], ins[7]) for ins in code if ins[7] is not None and start[0] <= ins[7] <= ins[0]]
            found.append(max(loops)[1] % 32)   # the loop that holds all others
    assert found == [28]
