"""Several-row bf16 and int8 heads on the f32 matrix cores: every row's sums
equal the one-row head's bit for bit, over ragged rows, columns past a chain's
last chunk, token groups, unaligned inputs and sums whose products underflow."""
import ctypes as C

import numpy as np
import pytest

import lbt_hip
import lbt_oracle as orc
from conftest import announce

pytestmark = pytest.mark.gpu


def linear_dev(ctx, fn, h, x, rows, offset=0):
    """fn over device buffers, x at `offset` floats into its allocation."""
    m, cols = x.shape
    lib = ctx.lib
    dx, do = C.c_void_p(), C.c_void_p()
    ctx.check(lib.lbt_dev_alloc(ctx.h, (m * cols + offset) * 4, C.byref(dx)))
    ctx.check(lib.lbt_dev_alloc(ctx.h, m * rows * 4, C.byref(do)))
    xp = C.c_void_p(dx.value + 4 * offset)
    out = np.zeros((m, rows), np.float32)
    try:
        ctx.check(lib.lbt_memcpy_h2d(ctx.h, xp, x.ctypes.data, x.nbytes))
        ctx.check(fn(ctx.h, h, xp, m, do))
        ctx.check(lib.lbt_memcpy_d2h(ctx.h, out.ctypes.data, do, out.nbytes))
    finally:
        lib.lbt_dev_free(ctx.h, dx)
        lib.lbt_dev_free(ctx.h, do)
    return out


# rows: whole and ragged 16-row tiles, few and many a CU, an odd and an even
# number a workgroup; cols: one to five chunks a chain, whole and cut; first
# matrices that stay on the older kernels
@pytest.mark.parametrize("rows,cols", [(300, 8), (1001, 648), (4000, 2560), (16401, 8), (16409, 128),
                                       (17345, 512), (16399, 520), (18000, 1000),
                                       (16500, 1536), (16807, 2040), (16392, 2552), (16400, 2560), (24577, 2560)])
@pytest.mark.parametrize("q8", [False, True])
def test_several_rows_equal_one_row(ctx, rows, cols, q8):
    rng = np.random.default_rng(rows + cols)
    w = (rng.standard_normal((rows, cols)) * 0.05).astype(np.float32)
    w[::97] *= 1e-30
    w[3::101] = 0.0
    wb = orc.f32_to_bf16(w).reshape(rows, cols)
    b = ctx.bf16_upload(wb)
    h = ctx.q8head_from_bf16(b) if q8 else b
    fn = ctx.lib.lbt_q8head_linear_dev if q8 else ctx.lib.lbt_bf16_linear_dev
    x = rng.standard_normal((50, cols)).astype(np.float32)
    x[5] *= 1e-20  # with the small rows: products below the denormals
    x[7] = 0.0
    one = np.concatenate([linear_dev(ctx, fn, h.h, x[i:i + 1], rows) for i in range(50)])
    for m, offset in ((2, 0), (4, 1), (5, 0), (8, 0), (9, 0), (12, 1), (13, 0), (16, 1), (17, 0), (24, 2), (33, 3), (50, 0)):
        announce(f"head rows={rows} cols={cols} q8={q8} m={m} offset={offset}")
        got = linear_dev(ctx, fn, h.h, x[:m], rows, offset)
        assert np.array_equal(got.view(np.uint32), one[:m].view(np.uint32)), m
    if q8:
        h.free()
    b.free()
