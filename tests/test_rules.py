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
int head_tiled(long rows, long m, long cus) { return lbt::head_tiled(rows, m, cus); }
int head_row_by_row(long rows, long cols, long m, int q8, long cus) {
    return lbt::head_row_by_row(rows, cols, m, q8 != 0, cus);
}
int attn_tiles_pay(long m, long pos0, long nh, long kvh, long splits, long keys) {
    return lbt::attn_tiles_pay(m, pos0, nh, kvh, splits, keys);
}
int gemm_128_tiles(long t128, long t64, int long_epilogue) {
    return lbt::gemm_128_tiles(t128, t64, long_epilogue != 0);
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
    lib.head_tiled.argtypes = [C.c_long] * 3
    lib.head_row_by_row.argtypes = [C.c_long] * 3 + [C.c_int, C.c_long]
    lib.attn_tiles_pay.argtypes = [C.c_long] * 6
    lib.gemm_128_tiles.argtypes = [C.c_long, C.c_long, C.c_int]
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


# us on an MI355X, row by row and with the several-row kernels
@pytest.mark.parametrize("q8,cols,rows,m,one,several", [
    (0, 2560, 16, 64, 4.5, 9.9), (0, 2560, 64, 24, 6.0, 10.2), (0, 2560, 1000, 2, 7.1, 10.8), (0, 2560, 1000, 8, 7.2, 10.7),
    (0, 2560, 1000, 16, 9.0, 11.5),
    (0, 2560, 1000, 48, 18.0, 12.8), (0, 2560, 1500, 5, 8.7, 11.3), (0, 2560, 2000, 4, 8.9, 11.2), (0, 2560, 4000, 2, 8.9, 12.0), (0, 2560, 4000, 5, 18.6, 12.1),
    (0, 2560, 4000, 16, 46.7, 13.0), (0, 2560, 40000, 8, 230.3, 46.0), (0, 2048, 12000, 4, 31.6, 16.5), (0, 1280, 12000, 2, 12.1, 16.8),
    (0, 1000, 16000, 3, 20.2, 14.2), (0, 512, 4000, 8, 9.4, 4.8), (0, 64, 40000, 64, 453.1, 40.6), (1, 64, 16, 9, 4.4, 5.9),
    (1, 2560, 300, 16, 7.3, 15.2), (1, 2560, 1000, 16, 9.1, 15.6), (1, 2560, 1000, 64, 21.4, 16.4), (1, 2560, 4000, 2, 8.2, 11.3),
    (1, 2560, 4000, 8, 16.0, 11.0), (1, 2560, 16000, 2, 15.9, 19.6), (1, 2560, 16000, 4, 27.8, 19.6), (1, 1000, 1000, 8, 7.8, 6.2),
    (1, 1000, 300, 9, 7.2, 8.4), (1, 512, 40000, 24, 176.7, 23.5),
])
def test_several_row_linears_take_the_faster_kernel(rules, q8, cols, rows, m, one, several):
    assert min(one, several) * 1.05 >= (one if rules.head_row_by_row(rows, cols, m, q8, 256) else several)


def test_more_rows_than_a_grid_holds_stay_on_the_several_row_kernels(rules):
    for rows in (1, 16, 32, 33, 1000):
        for cols in (8, 64, 2560):
            assert not any(rules.head_row_by_row(rows, cols, m, q8, 256) for m in (65536, 70000, 1 << 30)
                           for q8 in (0, 1))


# us of the other kernels and of the 16-row tiles
@pytest.mark.parametrize("heads,kv,pos0,m,other,tiles", [
    (20, 5, 0, 64, 7.9, 13.1), (20, 5, 0, 100, 10.5, 13.0), (20, 5, 0, 160, 14.9, 13.1), (20, 5, 0, 512, 55.7, 35.8),
    (20, 5, 700, 24, 14.4, 12.2), (20, 5, 2000, 17, 18.1, 19.6), (20, 5, 2000, 50, 34.3, 32.3), (20, 5, 3500, 17, 24.9, 33.2),
    (20, 5, 3500, 64, 83.8, 48.2), (8, 8, 0, 100, 6.7, 12.9), (8, 8, 0, 160, 9.3, 13.2), (8, 8, 0, 200, 20.0, 13.1),
    (8, 8, 700, 17, 7.4, 12.2), (8, 8, 700, 50, 16.7, 12.3), (8, 8, 2000, 17, 13.3, 19.1), (8, 8, 2000, 50, 35.4, 21.4),
    (8, 8, 3500, 17, 24.4, 31.7), (4, 4, 0, 160, 6.5, 12.8), (4, 4, 700, 33, 7.6, 12.2), (4, 4, 2000, 100, 42.8, 22.9),
    (32, 32, 0, 50, 7.0, 12.0), (32, 32, 0, 100, 20.6, 12.8), (8, 1, 2000, 17, 13.1, 19.1), (8, 1, 2000, 128, 90.0, 23.4),
    (24, 12, 0, 50, 6.3, 12.3), (24, 12, 300, 64, 25.2, 13.4), (16, 2, 700, 9, 8.0, 12.0), (6, 2, 0, 200, 17.2, 13.0),
])
def test_prefill_attention_takes_the_faster_kernel(rules, heads, kv, pos0, m, other, tiles):
    vis = pos0 + m
    keys = max(64, -(-vis // 16))
    pick = rules.attn_tiles_pay(m, pos0, heads, kv, -(-vis // keys), keys)
    assert min(other, tiles) * 1.05 >= (tiles if pick else other)


# us with 64 x 64 and 128 x 128 tiles
@pytest.mark.parametrize("rows,m,small,large", [
    ((1503, 203), 1250, 12.2, 13.6), ((1000, 1000, 1000), 700, 8.6, 10.6), ((1000, 1000, 1000), 1000, 24.7, 27.6),
    ((2560,), 850, 26.6, 22.5), ((2560,), 768, 18.7, 22.4)])
def test_prefill_gemms_take_the_faster_tile(rules, rows, m, small, large):
    total, ends = sum(rows), [sum(rows[:i + 1]) for i in range(len(rows) - 1)]
    t128, t64 = -(-total // 128) * -(-m // 128), -(-total // 64) * -(-m // 64)
    pick = rules.gemm_128_tiles(t128, t64, int(any(e % 64 for e in ends)))
    assert pick == (large < small)
