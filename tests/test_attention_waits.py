"""Every barrier of the attention kernels' block loop stands behind a wait for the wave's own global -> LDS loads: a wave hands
its part of a block to the others there, also one that left the block before without reading it (a window mask: its queries
see no key of that block)."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from pipelink_amd.pipec.pack import LLVM_BIN
from pipelink_amd.stages.attention import build as fa_build

pytestmark = pytest.mark.skipif(shutil.which("hipcc") is None and not Path("/opt/rocm/bin/hipcc").exists(), reason="needs the ROCm toolchain")


def _unwaited_barriers(text: str) -> list[str]:
    """Barriers a path through the kernel reaches with a load into LDS in flight (blocks and branches followed to a fixed point)."""
    lines = [m.groups() for m in re.finditer(r"^\s+([a-z]\w*)([^\n]*?)//\s*([0-9A-F]+):[^\n]*$", text, re.M)]
    at = {int(a, 16): i for i, (_, _, a) in enumerate(lines)}
    base = int(lines[0][2], 16)
    targets = [re.search(r"<pipelink_kernel\+0x([0-9a-f]+)>", l) for l in re.findall(r"^\s+[a-z]\w*[^\n]*$", text, re.M)]
    state: list[set] = [set() for _ in lines]
    state[0].add(False)
    work, bad = [(0, False)], []
    while work:
        i, flying = work.pop()
        op, args, addr = lines[i]
        if op == "s_barrier" and flying:
            bad.append(addr)
        if op.startswith("buffer_load") and "lds" in args:
            flying = True
        if op == "s_waitcnt" and re.search(r"vmcnt\(0\)", args):
            flying = False
        follow = []
        if op == "s_endpgm":
            continue
        if op in ("s_branch",) or op.startswith("s_cbranch"):
            follow.append(at[base + int(targets[i].group(1), 16)])
        if op != "s_branch":
            follow.append(i + 1)
        for j in follow:
            if flying not in state[j]:
                state[j].add(flying)
                work.append((j, flying))
    return bad


@pytest.mark.parametrize("image", ["linked", "window_linked", "half_linked", "window_half_linked", "one_unit"])
def test_no_barrier_is_reached_with_a_load_into_lds_in_flight(image):
    text = subprocess.run([str(LLVM_BIN / "llvm-objdump"), "-d", str(fa_build.images()[image])], capture_output=True, text=True, check=True).stdout
    text = text[text.index("<pipelink_kernel>:"):]
    assert len(re.findall(r"buffer_load_dwordx4[^\n]* lds", text)) >= 16
    assert _unwaited_barriers(text) == []


@pytest.mark.parametrize("image", ["linked", "window_linked", "half_linked", "window_half_linked", "one_unit"])
def test_reads_of_v_wait_for_no_load(image):
    """The next block's keys and values fly while this one's are read: the compiler puts no wait for them in front of the transposing
    reads (it does where it knows nothing of what these may alias)."""
    text = subprocess.run([str(LLVM_BIN / "llvm-objdump"), "-d", str(fa_build.images()[image])], capture_output=True, text=True, check=True).stdout
    reads, flying, waited = 0, False, False   # loads into LDS issued behind the last barrier; a wait for loads behind those
    for line in text[text.index("<pipelink_kernel>:"):].splitlines():
        if re.match(r"\s+s_barrier", line):
            flying = waited = False
        elif re.match(r"\s+buffer_load_dwordx4.* lds", line):
            flying, waited = True, False
        elif re.match(r"\s+s_waitcnt.*vmcnt", line):
            waited = True
        elif re.match(r"\s+ds_read_b64_tr_b16", line):
            reads += 1
            assert not (flying and waited), line
    assert reads >= 32
