"""Order of the batched decode kernel's loads, from the assembly of this
build.  Its waits are counts of loads (s_waitcnt vmcnt) that stand for whole
stages of the ring, so every stage's loads have to be issued together and in
turn; a load that moved behind later stages' would be waited for by draining
them, or, if a copy to LDS, be read before it lands."""
import os
import re
import shutil
import subprocess

import pytest

from conftest import PKG

RING, PIECES = 4, 3      # kRing, kPieces


@pytest.fixture(scope="module")
def asm(tmp_path_factory):
    import build
    if not (shutil.which(build.HIPCC) or os.path.exists(build.HIPCC)):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("asm") / "gemv_batch.s")
    subprocess.run([build.HIPCC, *build.DEVICE_FLAGS, *build.COMMON_FLAGS, "--cuda-device-only", "-S", "-o", out,
                    os.path.join(PKG, "csrc", "gemv_batch.hip")], check=True, capture_output=True)
    return open(out).read()


def events(asm, tile, stream):
    """A kernel's LDS copies (L), weight loads (W), barriers (B) and vmcnt
    waits (numbers), in order."""
    name = "_ZN5q35mm17gemv_batch_kernelILj%dELb%dEEEvNS_11BatchParamsE" % (tile, stream)
    body = asm[asm.index("\n%s:" % name):]
    ev = []
    for ln in body[:body.index("s_endpgm")].splitlines():
        op = ln.split()[0] if ln.split() else ""
        if op.startswith("buffer_load") and ln.rstrip().endswith("lds"):
            ev.append("L")
        elif op == "global_load_dwordx4":
            ev.append("W")
        elif op == "s_barrier":
            ev.append("B")
        elif op == "s_waitcnt" and "vmcnt" in ln:
            ev.append(int(re.search(r"vmcnt\((\d+)\)", ln).group(1)))
    return ev


@pytest.mark.parametrize("tile,stream", [(16, 1), (32, 0), (32, 1)])
def test_stages_are_issued_and_awaited_in_turn(asm, tile, stream):
    chunks = 64 // tile                         # weight loads of a stage
    stage = PIECES + chunks
    ev = events(asm, tile, stream)
    first = ev.index("L")
    pro = ev[first:first + RING * stage]
    for d in range(RING):
        got = sorted(pro[d * stage:(d + 1) * stage])
        assert got == ["L"] * PIECES + ["W"] * chunks, (d, pro)
    rest = ev[first + RING * stage:]
    waits = [v for v in rest[:-1 - rest[::-1].index("L")] if isinstance(v, int)]
    # until the last copy is issued nothing waits for the two newest stages
    assert waits and min(waits) >= (RING - 2) * stage, waits
