"""What a kernel's correctness needs of the instructions that the compiler makes of it, read from their listing (no GPU)."""
import os
import re
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gradients.c_amd", "csrc")


def _listing(source, tmp_path):
    """gfx950 instructions and labels per kernel of a source, compiled with the library's own flags."""
    make = ["make", "-s", "-C", CSRC, "--no-print-directory", "--eval", "print-flags:;@echo $(HIPCC) $(HIPFLAGS)", "print-flags"]
    out = str(tmp_path / "kernels.s")
    command = subprocess.run(make, check=True, capture_output=True, text=True).stdout.split()
    subprocess.run(command + ["-S", "--cuda-device-only", "-o", out, os.path.join(CSRC, source)], check=True, capture_output=True)
    kernels, name = {}, None
    for line in open(out):
        line = line.split(";")[0].strip()
        if re.match(r"_Z\w+:$", line):
            name = line[:-1]
            kernels[name] = []
        elif line.startswith(".section") or line.startswith(".end_amdhsa"):
            name = None
        elif name and line and (not line.startswith(".") or line.endswith(":")):
            kernels[name].append(line)
    return kernels


@pytest.mark.parametrize("source", ["ops/sdpa_decode/hip/sdpa_decode_pieces.hip"])
def test_partials_have_left_before_their_piece_is_counted_in(source, tmp_path):
    """The workgroup that counts the last piece of a row reads what the others stored: in front of the barrier that precedes
    the counting add, every wavefront waits for its own stores, with no way round the wait."""
    kernels = _listing(source, tmp_path)
    assert len(kernels) == 36  # 12 head shapes x (prefix, streaming, plain)
    for name, code in kernels.items():
        adds = [i for i, line in enumerate(code) if line.startswith("global_atomic_add")]
        assert len(adds) == 1, name
        barrier = max(i for i, line in enumerate(code[:adds[0]]) if line.startswith("s_barrier"))
        stores = [i for i, line in enumerate(code[:adds[0]]) if line.startswith("global_store") and line.endswith("sc1")]
        assert stores and stores[-1] < barrier, name
        before = barrier - 1
        while not re.match(r"s_waitcnt vmcnt\(0\)", code[before]):
            assert not re.match(r"(\.?\w+:|s_c?branch|global_|flat_|buffer_)", code[before]), (name, code[before])
            before -= 1
