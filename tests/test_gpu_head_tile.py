"""Several-row bf16 and int8 heads on the f32 matrix cores: every row's sums
equal the one-row head's bit for bit, over ragged rows, columns past a chain's
last chunk, token groups, unaligned inputs and sums whose products underflow;
and the greedy tokens they pick are the first largest logit's."""
import ctypes as C
import json

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
# matrices that stay on the older kernels, or (2560 x 4000 at 2 rows, 1001 x 648
# at 2 to 50 of int8) go row by row
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


# Greedy tokens (the argmax keys of the several-row kernels): vocabularies above
# their line, whole and ragged 16-row tiles; every token group (4, 8, 12 and 16
# rows, one and two of them); every embedding row twice, so that each largest
# logit is a tie of two rows that different workgroups hold.
@pytest.mark.parametrize("vocab", [34000, 34009])
def test_greedy_tokens_are_the_first_largest_logit(ctx, tmp_path, vocab):
    import torch
    from safetensors.torch import save_file

    H, I, half = 640, 256, vocab // 2
    rng = np.random.default_rng(vocab)
    t = {}
    names = ["self_attn.q_proj", "self_attn.k_proj", "self_attn.v_proj", "self_attn.o_proj", "mlp.gate_proj",
             "mlp.up_proj", "mlp.down_proj"]
    for n, (r, c) in zip(names, [(H, H), (128, H), (128, H), (H, H), (I, H), (I, H), (H, I)]):
        w = rng.integers(-1, 2, (r, c)).astype(np.int8)
        t[f"model.layers.0.{n}.qweight"] = torch.from_numpy(np.ascontiguousarray(orc.pack(w)))
        t[f"model.layers.0.{n}.wscale"] = torch.from_numpy(np.array([20.0], np.float32))
    for n, k in (("input_layernorm", H), ("post_attention_layernorm", H), ("self_attn.attn_sub_norm", H),
                 ("mlp.ffn_sub_norm", I)):
        t[f"model.layers.0.{n}.weight"] = torch.ones(k)
    t["model.norm.weight"] = torch.ones(H)
    emb = rng.uniform(-1, 1, (vocab, H)).astype(np.float32)
    emb[half:2 * half] = emb[:half]
    t["model.embed_tokens.weight"] = torch.from_numpy(emb).to(torch.bfloat16)
    save_file(t, str(tmp_path / "model.lbt.safetensors"), metadata={"format": "lemonade-burn-ternary", "version": "1"})
    (tmp_path / "config.json").write_text(json.dumps({
        "hidden_size": H, "intermediate_size": I, "num_attention_heads": 5, "num_key_value_heads": 1,
        "num_hidden_layers": 1, "vocab_size": vocab, "rms_norm_eps": 1e-5, "rope_theta": 1e4,
        "max_position_embeddings": 64, "hidden_act": "relu2", "tie_word_embeddings": True, "bos_token_id": 1}))
    m = lbt_hip.Model.load(ctx, tmp_path)
    for kind in (0, 1):
        m.set_head(kind)
        for nseq in (2, 6, 11, 16, 20, 30):
            announce(f"greedy tokens of the several-row head, vocab={vocab} kind={kind} nseq={nseq}")
            toks = rng.integers(0, vocab, nseq).astype(np.uint32)
            for want in (True, False):
                b = m.new_batch(nseq, 64)
                b.fill_synthetic(9, 4)
                logits, nxt = b.forward(toks, want)
                b.free()
                if want:
                    first = logits.argmax(1)
                    assert (first < half).any()
                    assert (np.ptp(np.sort(logits, 1)[:, -2:], axis=1) == 0)[first < half].all()
                assert np.array_equal(nxt, first)
    m.free()
