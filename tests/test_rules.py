"""The conditions of csrc/rules.h, compiled for the CPU: what a path is
chosen by, checked against what the path does with the sizes."""
import ctypes as C
import re
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "lemonade-burn_amd" / "csrc"

SHIM = """
#include "rules.h"
extern "C" {
int lean_offsets_fit(long m, long ld, long tok0, long tokens, long rows) {
    return lbt::lean_offsets_fit(m, ld, tok0, tokens, rows);
}
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "shim.cpp").write_text(SHIM)
    so = d / "rules.so"
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", f"-I{CSRC}",
                        str(d / "shim.cpp"), "-o", str(so)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    lib = C.CDLL(str(so))
    lib.lean_offsets_fit.argtypes = [C.c_long] * 5
    return lib


# outputs whose last value lies just below and above 2^30 values, by the rows
# of a token (one, a vocabulary, many) and the tokens of the last block
@pytest.mark.parametrize("ld", [1, 3, 64, 2560, 6912, 65536, 128256, 9_000_000, 1 << 29])
def test_lean_epilogue_offsets_never_wrap_into_the_output(rules, ld):
    # a wavefront block's tokens and rows in the pipelined GEMMs' tilings
    blocks = [(32, 32), (64, 64), (128, 32), (32, 64)]
    top = (1 << 30) // ld
    ms = {m for d in (0, 1, 2, 31, 33, 63, 65, 100, 127, 129) for m in (top - d, top + d) if m > 0}
    for m in sorted(ms | {33, 100, 301, 8371, 16383, 155344}):
        for tokens, rows in blocks:
            for tok0 in {0, (m - 1) // tokens * tokens, max(0, (m - 1) // tokens * tokens - tokens)}:
                if not rules.lean_offsets_fit(m, ld, tok0, tokens, rows):
                    continue
                # the offsets of the block's tokens past m stay past the end of
                # the buffer of m ld values, those below m inside it
                assert m * ld * 4 < 1 << 32
                for tok in {tok0, min(m, tok0 + tokens - 1), tok0 + tokens - 1}:
                    for row in (0, min(ld, rows) - 1, ld - 1):
                        off = (tok * ld + row) * 4 % (1 << 32)
                        assert (off < m * ld * 4) == (tok < m), (m, tok0, tokens, tok, row)


def test_lean_epilogue_keeps_the_blocks_it_can_address(rules):
    # whole and ragged blocks of ordinary outputs, up to the last that fits
    for m, ld in ((33, 3840), (301, 1706), (3000, 13824), (2048, 2560), (8000, 128256)):
        for tok0 in range(0, m, 64):
            assert rules.lean_offsets_fit(m, ld, tok0, 64, 64)


def test_no_launch_keeps_per_process_state():
    # A kernel's LDS limit belongs to the device the context is on: a flag set
    # once per process leaves a second device without it, and races between
    # threads.  Launch code holds no writable function-level statics.
    for src in sorted(CSRC.glob("*.hip")) + sorted(CSRC.glob("*.cpp")):
        for n, line in enumerate(src.read_text().splitlines(), 1):
            assert not re.match(r"\s+static (?!const|inline|_)", line), f"{src.name}:{n}: {line.strip()}"
