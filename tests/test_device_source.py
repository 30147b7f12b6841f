"""Rules the device sources keep by themselves, checked on the text."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vai_amd", "csrc")

# Vector instructions in asm without a wait of their own, and what keeps an
# MFMA's result far enough from them.
GUARDED = {
    ("tile_store.h", "v_accvgpr_read_b32 %0, %1"),      # read after the three s_nop 7 of the epilogue
    # O of the last tile: this tile's 32 S^T MFMAs, on other registers, come between
    ("attention.hip", "v_accvgpr_read_b32 %1, %0\\n\\tv_mul_f32 %1, %1, %2\\n\\tv_accvgpr_write_b32 %0, %1"),
}


def test_vector_asm_brings_its_own_wait():
    """The compiler puts wait states between an MFMA and an instruction that
    reads its result only where it places that instruction itself: an asm
    statement that reads values of the kernel either begins with its own s_nop
    or is one of those above."""
    files = sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.h")))
    assert files
    found, bad = set(), []
    for f in files:
        with open(f) as fh:
            text = fh.read()
        for m in re.finditer(r'\basm\s*(?:volatile)?\s*\(\s*((?:"[^"]*"\s*)+)', text):
            body = "".join(re.findall(r'"([^"]*)"', m.group(1)))
            if not re.search(r"\bv_\w+", body):
                continue
            key = (os.path.basename(f), body)
            found.add(key)
            if not body.startswith("s_nop") and key not in GUARDED:
                bad.append(f"{key[0]}:{text.count(chr(10), 0, m.start()) + 1}: {body}")
    assert not bad, bad
    assert GUARDED <= found
