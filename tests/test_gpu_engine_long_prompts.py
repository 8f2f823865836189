"""Prompts so long that the many-row attention runs without a key split and writes the
o projection's input by itself, the GEMM's padding rows included (more than 2048 rows
at head dim 256, more than 4096 at 512, with 8 heads).  The plain prefill is held to
the diagnostic one, which stores every stage and prepares each GEMM's input from it."""
import numpy as np
import pytest

import synthetic as syn

pytestmark = pytest.mark.gpu

H, HEADS, P, V, INTER, RPS = 128, 8, 32, 512, 256, 64


def engine(g4, hd, max_seq):
    """Two layers with caches of their own, a sliding and a global one, both of head dim hd."""
    c = g4.GemmaConfig()
    c.hidden, c.heads, c.ple_dim, c.vocab = H, HEADS, P, V
    c.layers, c.max_seq, c.window, c.eps, c.softcap = 2, max_seq, 512, 1e-6, 30.0
    for i in range(2):
        c.head_dim[i], c.intermediate[i], c.full[i], c.kv_source[i] = hd, INTER, i, -1
        c.rope_base[i], c.rope_prop[i] = 1e4, 1.0
    rng = np.random.default_rng(hd)
    m = g4.Gemma(c)
    m.set_embedding(g4.Buffer.from_array(
        syn.bf16_rne(rng.standard_normal((V, H)).astype(np.float32) * np.float32(0.05))))
    t = g4.PleTable(V, 2 * P, 32, RPS)
    for s in range(V // RPS):
        t.upload_shard(s, syn.ple_shard(7, s, RPS, 2 * P))
    m.set_ple(t)
    seed = [hd]

    def lin(layer, name, n, k):
        seed[0] += 1
        m.set_linear(layer, name, g4.W4Linear(*syn.w4_weights(seed[0], n, k)[:2]))

    lin(-1, "top", 2 * P, H)
    m.set_norm(-1, "ple_projection", rng.uniform(0.8, 1.2, P).astype(np.float32))
    m.set_norm(-1, "final", rng.uniform(0.8, 1.2, H).astype(np.float32))
    for i in range(2):
        for name, n, k in (("q", HEADS * hd, H), ("k", hd, H), ("v", hd, H), ("o", H, HEADS * hd),
                           ("gate", INTER, H), ("up", INTER, H), ("down", H, INTER),
                           ("ple_gate", P, H), ("ple_proj", H, P)):
            lin(i, name, n, k)
        for name in ("input", "post_attn", "pre_ffw", "post_ffw", "post_ple"):
            m.set_norm(i, name, rng.uniform(0.8, 1.2, H).astype(np.float32))
        for name in ("q", "k"):
            m.set_norm(i, name, rng.uniform(0.2, 0.4, hd).astype(np.float32))
        m.set_layer_scalar(i, 1.0)
    return m


def rel(a, b):
    return np.linalg.norm(a.astype(np.float64) - b) / np.linalg.norm(b)


# one live row, a half and a whole one in the last 64-row block, and padding after it
@pytest.mark.parametrize("hd,rows", [(256, 2049), (256, 2053), (256, 2056), (256, 2112),
                                     (512, 4097), (512, 4131)])
def test_unsplit_attention_hands_over_its_rows(g4, hd, rows):
    m = engine(g4, hd, rows + 32)
    ids = syn.token_ids(rows, rows + 6, V)
    got = {}
    for kind in ("plain", "diagnostic"):
        m.reset()
        last, after = g4.Buffer(H * 4), g4.Buffer(H * 4)
        if kind == "plain":
            m.forward(ids[:rows], 0, last)
        else:
            m.forward_diag(ids[:rows], 0, last, None, None, None)
        # six more rows see what both layers' caches hold of every row before them
        layers = g4.Buffer(2 * 6 * H * 4)
        m.forward_diag(ids[rows:], rows, after, None, None, layers)
        got[kind] = [b.download(np.float32) for b in (last, after, layers)]
    m.free()
    for a, b in zip(got["plain"], got["diagnostic"]):
        assert np.all(np.isfinite(a)) and rel(a, b) < 1e-5, (hd, rows, rel(a, b))
