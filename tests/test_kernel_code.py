"""What the compiler makes of kernels whose waits count loads: read off the gfx950 assembly of the sources, built with the
library's flags."""
import os
import random
import re
import shutil
import subprocess

import pytest

from openvino_amd import build


def kernels(source, out):
    """{mangled name: [(block label, in the loop that holds the matrix instructions, instructions)]}"""
    subprocess.run([build.hipcc_path(), *build.FLAGS, "-S", "--cuda-device-only", f"{build.CSRC}/{source}", "-o", out],
                   check=True, capture_output=True)
    found = {}
    for name, body in re.findall(r"^(_Z\w+):[^\n]*\n(.*?)^\.Lfunc_end", out.read_text(), re.S | re.M):
        blocks, loops = [["entry", None, []]], {}
        for line in body.splitlines():
            if label := re.match(r"\.L(BB\d+_\d+):", line):
                blocks.append([label[1], None, []])
            if m := re.search(r";.*(?:in Loop: Header=(BB\d+_\d+)|Inner Loop Header)", line):
                blocks[-1][1] = m[1] or blocks[-1][0]
            ins = line.split(";")[0].strip()
            if ins and not ins.startswith((".", "#")) and not ins.endswith(":"):
                blocks[-1][2].append(ins)
                if ins.startswith("v_mfma"):
                    loops[blocks[-1][1]] = loops.get(blocks[-1][1], 0) + 1
        main = max((loop for loop in loops if loop), key=loops.get, default=None)
        found[name] = [(label, loop is not None and loop == main, code) for label, loop, code in blocks]
    return found


def walk(blocks, rng, visit):
    """One way through the kernel, every branch taken or not by chance."""
    at = {label: i for i, (label, _, _) in enumerate(blocks)}
    i = 0
    while i < len(blocks):
        target = i + 1
        for ins in blocks[i][2]:
            visit(ins, blocks[i][1])
            if ins.startswith("s_endpgm"):
                return
            if ins.startswith("s_branch") or (ins.startswith("s_cbranch") and rng.random() < 0.5):
                target = at[ins.split(".L")[1]]
                break
        i = target


@pytest.fixture(scope="module")
def ragged(tmp_path_factory):
    return kernels("kernel_ragged.hip", tmp_path_factory.mktemp("asm") / "ragged.s")


@pytest.mark.parametrize("bits", [4, 8])
def test_direct_loads_have_landed_at_their_barrier(ragged, bits):
    """fcc_ragged_tile_dma_kernel: whichever way a wave goes, the four activation loads of a k-block are in LDS at the barrier
    of its trip, and no wait of the loop is for anything asked for since the k-block before the last (AL + 8 loads)."""
    blocks = next(b for n, b in ragged.items() if f"fcc_ragged_tile_dma_kernelILi{bits}E" in n)
    longest = 0
    for seed in range(400):
        out, landed, trips = [], 0, 0  # outstanding memory operations, oldest first

        def visit(ins, in_loop):
            nonlocal landed, trips, out
            op = ins.split()[0]
            if re.match(r"(buffer|global|flat|scratch)_", op):
                out.append(ins.endswith("lds"))
            if (wait := re.search(r"vmcnt\((\d+)\)", ins)) and op == "s_waitcnt":
                assert not in_loop or int(wait[1]) >= 12, ins
                gone = out[:max(0, len(out) - int(wait[1]))]
                out, landed = out[len(gone):], landed + sum(gone)
            if op == "s_barrier" and in_loop:
                trips += 1
                assert landed >= 4 * trips, f"k-block {trips - 1}: {landed} loads have landed"

        walk(blocks, random.Random(seed), visit)
        longest = max(longest, trips)
    assert longest >= 6


# Registers that the compiler may spill, all of them outside the loops over k-blocks: around the 128-row kernel's (six more
# inside, reloaded with every second k-block, took a tenth of its time with zero-points), and where the integer kernel adds
# parked sums.
SPILLS = {"fcc_prefill_async_kernel": 2, "fcc_prefill_async_grouped_kernel": 2, "fcc_prefill_big_kernel": 0,
          "fcc_prefill_i8_big_kernel": 8, "fcc_ragged_tile_dma_kernel": 0}


def test_no_more_registers_are_spilled_than_were_looked_at(tmp_path):
    """Read off the built library's notes."""
    shutil.copy(build.LIB, tmp_path / "lib.so")
    tools = f"{os.path.dirname(os.path.realpath(build.hipcc_path()))}/../llvm/bin"
    subprocess.run([f"{tools}/llvm-objdump", "--offloading", "lib.so"], cwd=tmp_path, check=True, capture_output=True)
    seen = {}
    for obj in tmp_path.glob("*gfx950"):
        notes = subprocess.run([f"{tools}/llvm-readelf", "--notes", str(obj)], check=True, capture_output=True, text=True).stdout
        for name, spilled in re.findall(r"\.name: +(_Z\w+)\n(?:(?! +\.name:).*\n)*? +\.vgpr_spill_count: +(\d+)", notes):
            kernel = re.match(r"_ZN5ovfcc\d+(fcc_[a-z0-9_]+_kernel)", name)
            if kernel and kernel[1] in SPILLS:
                seen.setdefault(kernel[1], []).append(int(spilled))
                assert int(spilled) <= SPILLS[kernel[1]], name
    assert seen.keys() == SPILLS.keys() and len(seen["fcc_prefill_async_kernel"]) >= 12, seen
