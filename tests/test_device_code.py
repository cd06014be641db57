"""Properties of the built gfx950 code that the sources rely on and no
numerical test can show (they hold or fail per build)."""
import os
import re

import pytest

from pylops_amd import _lib
from tests import device_code as D

pytestmark = pytest.mark.skipif(not os.path.exists(os.path.join(D.LLVM, "llvm-objdump")),
                                reason="the LLVM binary tools are not installed")


def test_row_broadcasts_carry_their_wait_states(tmp_path):
    """A DPP instruction must not read a register within two wait states of
    the vector instruction that wrote it.  The compiler keeps to it for its
    own instructions and does not look into inline assembly: the half-row
    pairs written there (bank masks 0x3 and 0xc) follow a wait of their own."""
    pairs = 0

    def half(ins):
        return "row_newbcast" in ins and re.search(r"bank_mask:0x[3c]\b", ins)

    for name, code in D.disassemble(_lib.LIBPATH, tmp_path, r"slots_kernel.*Li8E"):
        i = 0
        while i < len(code):
            if "row_newbcast" not in code[i] or "bank_mask:0x3" not in code[i]:
                i += 1
                continue
            # a run of pairs after one wait, none of which writes what a
            # later one broadcasts
            m = re.match(r"s_nop (\d+)", code[i - 1])
            assert m and int(m.group(1)) >= 1, (name, code[i - 3:i + 1])
            written = set()
            while half(code[i]):
                out, src = re.match(r"\S+ (v\d+), (v\d+),", code[i]).groups()
                assert src not in written, (name, code[i])
                written.add(out)
                pairs += "bank_mask:0x3" in code[i]
                i += 1
    assert pairs > 100


def test_batch_gathers_keep_their_values_in_registers(tmp_path):
    """The batch adjoint holds the windowed and the general gather in one
    kernel: with the registers limited for the first, the second kept values
    of every receiver in scratch memory and took twice its time."""
    seen = 0
    for name, md in D.kernel_metadata(_lib.LIBPATH, tmp_path).items():
        if "batch_gather_kernel" in name:
            seen += 1
            assert md["private_segment_fixed_size"] == 0, (name, md)
            assert md["vgpr_spill_count"] == 0, (name, md)
    assert seen > 0
