"""Wait states of the hand-written vector-memory instructions (CPU): the compiler's
hazard recognizer does not look inside an asm statement, so a load whose base
address is a scalar register operand must be preceded, within the statement, by
the five wait states a vector instruction's write of that register needs, and one
that takes its LDS address from m0 by one after the write of m0."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dvattention_amd", "csrc")
SGPR_TO_VMEM, M0_TO_LDS_DMA = 5, 1


def statements():
    for path in sorted(glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(CSRC, "*.hip"))):
        for m in re.finditer(r'asm volatile\(\s*((?:"[^"]*"\s*)+)', open(path).read()):
            text = "".join(re.findall(r'"([^"]*)"', m.group(1)))
            yield os.path.basename(path), [i.strip() for i in text.split(r"\n\t")]


def test_wait_states_before_loads():
    scalar_base = 0
    for name, instrs in statements():
        states, since_m0 = 0, None
        for ins in instrs:
            op = ins.split()[0] if ins else ""
            if op.startswith("global_load"):
                if re.match(r"global_load_\w+ %\d+, %\d+", ins):
                    scalar_base += 1
                    assert states >= SGPR_TO_VMEM, (name, instrs)
                if "_lds_" in op:
                    assert since_m0 is not None and since_m0 >= M0_TO_LDS_DMA, (name, instrs)
            n = int(ins.split()[1]) + 1 if op == "s_nop" else 1
            states += n
            since_m0 = 0 if ins.startswith("s_mov_b32 m0") else (None if since_m0 is None else since_m0 + n)
    assert scalar_base == 2
