"""The order of the loads in kernel_prefill_pair.hip, whose waits count them: read off the gfx950 assembly, built with the
library's flags."""
import random
import re
import subprocess

import pytest

from openvino_amd import build
from test_kernel_code import walk


@pytest.fixture(scope="module")
def pair(tmp_path_factory):
    """{kernel: [(block label, loop, instructions)]}; a loop is named after its header"""
    out = tmp_path_factory.mktemp("asm") / "pair.s"
    subprocess.run([build.hipcc_path(), *build.FLAGS, "-S", "--cuda-device-only", f"{build.CSRC}/kernel_prefill_pair.hip",
                    "-o", out], check=True, capture_output=True)
    found = {}
    for name, body in re.findall(r"^(_Z\w+):[^\n]*\n(.*?)^\.Lfunc_end", out.read_text(), re.S | re.M):
        blocks = [["entry", None, []]]
        for line in body.splitlines():
            if label := re.match(r"(?:\.L(BB\d+_\d+):|; (%bb\.\d+):)", line):
                blocks.append([label[1] or label[2], None, []])
            if m := re.search(r";.*(?:in Loop: Header=(BB\d+_\d+)|Inner Loop Header)", line):
                blocks[-1][1] = m[1] or blocks[-1][0]
            ins = line.split(";")[0].strip()
            if ins and not ins.startswith((".", "#")) and not ins.endswith(":"):
                blocks[-1][2].append(ins)
        found[name] = blocks
    return found


def test_activations_have_landed_at_their_barrier(pair):
    """Whichever way a wave goes: at every barrier of a loop over K, the loads of all stages published so far have landed (a
    stage is the loop's loads to LDS over its barriers), and none of the loop's waits drains what was asked for last."""
    assert len(pair) >= 8
    for name, blocks in pair.items():
        main = {}
        for _, loop, code in blocks:
            if loop:
                n = main.setdefault(loop, [0, 0, 0])
                n[0] += sum(i.startswith("s_barrier") for i in code)
                n[1] += sum(i.startswith("buffer_load") and i.endswith("lds") for i in code)
                n[2] += sum(i.startswith("v_mfma") for i in code)
                assert not any(i.startswith("scratch_") for i in code), name
        main = {loop: n[1] // n[0] for loop, n in main.items() if n[2]}
        assert main and all(main.values()), name
        # (label, loop over K that the block belongs to or, for the k-blocks behind it, follows, instructions)
        labels, last = [], None
        for label, loop, code in blocks:
            last = loop if loop in main else last
            behind = loop is None and any(i.startswith("v_mfma") for i in code)
            labels.append((label, (last, True) if loop in main else (last, False) if behind else None, code))
        seen = set()
        for seed in range(60):
            out, landed, trips, first = [], 0, 0, None  # outstanding memory operations, oldest first

            def visit(ins, where):
                nonlocal out, landed, trips, first
                op, (loop, inside) = ins.split()[0], where or (None, False)
                first = first or loop
                if loop != first and loop:
                    out, landed, trips = [], 0, -10 ** 6  # (a way that chance alone takes: two tile heights one after the other)
                if re.match(r"(buffer|global|flat|scratch)_", op):
                    out.append(ins.endswith("lds"))
                if (wait := re.search(r"vmcnt\((\d+)\)", ins)) and op == "s_waitcnt":
                    assert not inside or int(wait[1]) >= main[loop], (name, loop, ins)
                    gone = out[:max(0, len(out) - int(wait[1]))]
                    out, landed = out[len(gone):], landed + sum(gone)
                if op == "s_barrier" and loop:
                    trips += 1
                    assert landed >= main[loop] * trips, (name, loop, f"stage {trips - 1}: {landed} loads have landed")
                    if trips >= 6:
                        seen.add(loop)

            walk(labels, random.Random(seed), visit)
        assert seen, name
