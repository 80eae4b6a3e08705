"""The pipelined GEMMs' lean epilogues on ragged blocks (tokens past the last
one, rows past a matrix's end, gate/up and q/k/v outputs): equal to the
few-token kernel's general epilogue bit for bit, through every tiling."""
import numpy as np
import pytest

import lbt_hip
import lbt_oracle as orc
from conftest import announce

pytestmark = pytest.mark.gpu

MODES = ["4", "5", "7", "8"]


# tokens around a block's 32 and a tile's 64 / 128; an FFN that is no multiple
# of a row tile; head_dim 64 and 128
@pytest.mark.parametrize("heads,kv,hidden,ffn", [(4, 1, 512, 1000), (8, 2, 512, 336)])
@pytest.mark.parametrize("n", [33, 63, 65, 129, 200])
def test_model_epilogues_on_ragged_prompts(ctx_with, heads, kv, hidden, ffn, n):
    cfg = lbt_hip.make_config(hidden=hidden, intermediate=ffn, heads=heads, kv_heads=kv, layers=2, vocab=300,
                              max_pos=512)
    toks = np.random.default_rng(n).integers(0, 300, n).astype(np.uint32)
    want = None
    for mode in ["6"] + MODES:
        announce(f"ragged epilogues heads={heads} ffn={ffn} n={n} mode={mode}")
        m = lbt_hip.Model.synthetic(ctx_with(LBT_GEMM_MODE=mode), cfg, 41)
        c = m.new_cache()
        m.forward(toks[:5], c)  # rows start at position 5
        out = (m.forward(toks[5:], c, all_logits=True), c.read(1, False), c.read(1, True), m.read_hidden(n - 5))
        c.free()
        m.free()
        want = want or out
        for x, y in zip(out, want):
            assert np.array_equal(x, y), mode


@pytest.mark.parametrize("rows", [(33,), (70, 95), (1503, 203), (64, 1, 130)])
@pytest.mark.parametrize("m", [33, 95, 301])
def test_linear_epilogues_on_ragged_rows(ctx_with, rows, m):
    cols = 300
    rng = np.random.default_rng(m + len(rows))
    x = rng.standard_normal((m, cols)).astype(np.float32)
    w = [rng.integers(-1, 2, (r, cols)).astype(np.int8) for r in rows]
    want = None
    for mode in ["6"] + MODES:
        announce(f"ragged linear rows={rows} m={m} mode={mode}")
        ctx = ctx_with(LBT_GEMM_MODE=mode)
        ws = [ctx.upload(orc.pack(t), t.shape[0], cols, 11.0 + i) for i, t in enumerate(w)]
        out = ctx.ternary_linear(ws, x)
        q, s, su = ctx.quantize_acts(x)
        ints = ctx.gemm_i32(ws[0], q, su)
        assert np.array_equal(ints, q[:, :cols].astype(np.int64) @ w[0].astype(np.int64).T)
        want = want or out
        for a, b in zip(out, want):
            assert np.array_equal(a, b), mode
        for h in ws:
            h.free()
