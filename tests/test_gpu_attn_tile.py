"""Prefill attention in 16-row tiles on the f32 matrix cores
(LBT_ATTN_TILE): the same logits and KV cache, bit for bit, as the workgroup
kernels over tile edges, split edges, chunked prompts and head groupings, and
non-finite V values kept out of the rows that do not see them."""
import json

import numpy as np
import pytest

import lbt_hip
import lbt_oracle as orc
from conftest import announce

pytestmark = pytest.mark.gpu


def run(ctx, cfg, pos0, toks):
    m = lbt_hip.Model.synthetic(ctx, cfg, 23)
    c = m.new_cache()
    if pos0:
        m.forward(toks[:pos0], c)
    out = (m.forward(toks[pos0:], c, all_logits=True), c.read(1, False), c.read(1, True))
    c.free()
    m.free()
    return out


# (heads, kv heads) with head_dim 128; (positions before, tokens): tiles of
# fewer than 16 rows at either end, 64-key splits and their edges, 65..256-key
# splits (past 1024 keys), the longest split the kernel takes (4096 keys), one
# more (the other kernels serve it)
@pytest.mark.parametrize("heads", [(4, 1), (2, 2), (5, 1), (6, 3)])
@pytest.mark.parametrize("pos0,n", [(0, 2), (0, 17), (0, 65), (7, 9), (15, 2), (63, 40), (1000, 30), (1031, 33),
                                    (2040, 20), (0, 1100), (4070, 26), (4080, 30)])
def test_attention_tiles_equal_workgroup_kernels(ctx_with, heads, pos0, n):
    nh, kvh = heads
    cfg = lbt_hip.make_config(hidden=128 * nh, intermediate=256, heads=nh, kv_heads=kvh, layers=2, vocab=300,
                              max_pos=4224)
    announce(f"attention tiles heads={heads} pos0={pos0} n={n}")
    toks = np.random.default_rng(n + pos0).integers(0, 300, pos0 + n).astype(np.uint32)
    a = run(ctx_with(LBT_ATTN_TILE="1"), cfg, pos0, toks)
    b = run(ctx_with(LBT_ATTN_TILE="0"), cfg, pos0, toks)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


def test_attention_tiles_keep_nonfinite_values_from_earlier_rows(ctx_with, tmp_path):
    # Token 1 has a channel whose norm gain makes its V row infinite or NaN.
    # Rows before it in the same 16-row tile do not see that key: their logits
    # stay finite, and every row equals the workgroup kernel's.
    import torch
    from safetensors.torch import save_file

    H, I, KV, V = 512, 256, 128, 300
    rng = np.random.default_rng(3)
    t = {}
    names = ["self_attn.q_proj", "self_attn.k_proj", "self_attn.v_proj", "self_attn.o_proj", "mlp.gate_proj",
             "mlp.up_proj", "mlp.down_proj"]
    for n, (r, c) in zip(names, [(H, H), (KV, H), (KV, H), (H, H), (I, H), (I, H), (H, I)]):
        w = rng.integers(-1, 2, (r, c)).astype(np.int8)
        t[f"model.layers.0.{n}.qweight"] = torch.from_numpy(np.ascontiguousarray(orc.pack(w)))
        scale = 1e-12 if n == "self_attn.v_proj" else 20.0
        t[f"model.layers.0.{n}.wscale"] = torch.from_numpy(np.array([scale], np.float32))
    gain = np.ones(H, np.float32)
    gain[300] = 1e30
    for n, k in (("input_layernorm", H), ("post_attention_layernorm", H), ("self_attn.attn_sub_norm", H),
                 ("mlp.ffn_sub_norm", I)):
        t[f"model.layers.0.{n}.weight"] = torch.from_numpy(gain if n == "input_layernorm" else np.ones(k, np.float32))
    t["model.norm.weight"] = torch.from_numpy(np.ones(H, np.float32))
    emb = rng.uniform(-1, 1, (V, H)).astype(np.float32)
    emb[:, 300] = 0.0
    emb[1, 300] = 1.0
    t["model.embed_tokens.weight"] = torch.from_numpy(emb).to(torch.bfloat16)
    save_file(t, str(tmp_path / "model.lbt.safetensors"), metadata={"format": "lemonade-burn-ternary", "version": "1"})
    (tmp_path / "config.json").write_text(json.dumps({
        "hidden_size": H, "intermediate_size": I, "num_attention_heads": 4, "num_key_value_heads": 1,
        "num_hidden_layers": 1, "vocab_size": V, "rms_norm_eps": 1e-5, "rope_theta": 1e4,
        "max_position_embeddings": 512, "hidden_act": "relu2", "tie_word_embeddings": True, "bos_token_id": 1}))
    announce("attention tiles, a non-finite V row at position 74 of 90")
    toks = rng.integers(2, V, 90).astype(np.uint32)
    toks[74] = 1
    outs = []
    for env in ("1", "0"):
        m = lbt_hip.Model.load(ctx_with(LBT_ATTN_TILE=env), tmp_path)
        c = m.new_cache()
        logits = m.forward(toks, c, all_logits=True)
        v = orc.bf16_to_f32(c.read(0, True))
        outs.append((logits, m.read_hidden(90)))
        c.free()
        m.free()
    assert np.isfinite(v[:, :74]).all() and not np.isfinite(v[:, 74]).any()
    for a, b in zip(*outs):
        assert np.isfinite(a[:74]).all()
        assert np.array_equal(a, b, equal_nan=True)
