"""Seeded random shapes through the W4 linear, dequant and PLE entry points.

A linear case draws a row count (the GEMV sizes 1-4 and the GEMM sizes
above), an output width that is rarely a tile multiple, an input width (a
multiple of the 32-value group), an activation dtype and an output dtype, and
checks the result against the binary64 product x . dequant(W)^T (max
relative L2 error per row); BF16 outputs must be the round-to-nearest-even of
the FP32 outputs of the same call.  Dequant and PLE cases draw shapes, row
ranges, table geometry and ids, and must match the oracle bit for bit.
"""
import numpy as np
import pytest

import synthetic as syn

pytestmark = pytest.mark.gpu

ROWS = [1, 2, 3, 4, 5, 8, 33, 100, 257]


def dense(q, scales):
    return q.astype(np.float64) * np.repeat(syn.bf16_to_f32(scales).astype(np.float64), 32, axis=1)


def rel_l2_rows(y, ref):
    num = np.linalg.norm(np.asarray(y, np.float64) - ref, axis=-1)
    den = np.maximum(np.linalg.norm(ref, axis=-1), 1e-300)
    return float((num / den).max())


def draw(seed):
    rng = np.random.default_rng(1000 + seed)
    rows = int(rng.choice(ROWS))
    n = int(rng.integers(1, 700))
    k = 32 * int(rng.integers(1, 129))  # 32 .. 4096
    f32x = bool(rng.integers(0, 2))
    return rng, rows, n, k, f32x


def activations(g4, rng, rows, k, f32x):
    x = rng.standard_normal((rows, k)).astype(np.float32)
    if f32x:
        return g4.Buffer.from_array(x), x, g4.F32
    bits = syn.bf16_rne(x)
    return g4.Buffer.from_array(bits), syn.bf16_to_f32(bits).reshape(rows, k), g4.BF16


@pytest.mark.parametrize("seed", range(48))
def test_random_linear(g4, seed):
    rng, rows, n, k, f32x = draw(seed)
    packed, scales, q = syn.w4_weights(500 + seed, n, k)
    lin = g4.W4Linear(packed, scales)
    xb, x, xd = activations(g4, rng, rows, k, f32x)
    y32 = g4.Buffer(rows * n * 4)
    y16 = g4.Buffer(rows * n * 2)
    lin.linear(xb.ptr, xd, rows, y32.ptr, g4.F32)
    lin.linear(xb.ptr, xd, rows, y16.ptr, g4.BF16)
    got = y32.download(np.float32).reshape(rows, n)
    ref = x.astype(np.float64) @ dense(q, scales).T
    assert rel_l2_rows(got, ref) <= 1e-4, (rows, n, k, f32x)
    assert np.array_equal(y16.download(np.uint16).reshape(rows, n),
                          syn.bf16_rne(got).reshape(rows, n)), (rows, n, k, f32x)


# The few-row kernel at its edges: one to 257 stages of 64 inputs (idle waves, a
# last slice that is short, 8 slices, one stage too many for it), row tiles of
# 16 and 32 and several of them, ragged and tiny widths, and what it leaves to
# the prefill GEMM and the GEMV beside it.  A wrong stage, row or column changes
# whole elements.
@pytest.mark.parametrize("k", [64, 128, 1536, 1600, 2048, 2112, 6144, 16384, 16448])
@pytest.mark.parametrize("rows,n", [(2, 1), (3, 257), (4, 100), (5, 16), (16, 47), (17, 100),
                                    (32, 33), (33, 15), (70, 240), (130, 17)])
@pytest.mark.parametrize("f32x", [False, True])
def test_few_rows_edges(g4, k, rows, n, f32x):
    rng = np.random.default_rng([k, rows, n])
    packed, scales, q = syn.w4_weights(k + 7 * rows + n, n, k)
    lin = g4.W4Linear(packed, scales)
    x = rng.standard_normal((rows, k)).astype(np.float32)
    x *= (10.0 ** rng.uniform(-6, 6, (rows, 1))).astype(np.float32)
    x[rows // 2] = 0.0
    if f32x:
        xb = g4.Buffer.from_array(x)
    else:
        bits = syn.bf16_rne(x)
        xb, x = g4.Buffer.from_array(bits), syn.bf16_to_f32(bits).reshape(rows, k)
    xd = g4.F32 if f32x else g4.BF16
    ref = x.astype(np.float64) @ dense(q, scales).T
    y32, y16 = g4.Buffer(rows * n * 4), g4.Buffer(rows * n * 2)
    lin.linear(xb.ptr, xd, rows, y32.ptr, g4.F32)
    lin.linear(xb.ptr, xd, rows, y16.ptr, g4.BF16)
    got = y32.download(np.float32).reshape(rows, n)
    # FP32 x to 2^-22, and one rounding (2^-24 of a partial sum, within four
    # standard deviations 4 size) per matrix step (two per 32 inputs with FP32 x)
    # and per slice added; up to four rows may run the GEMV, with x in two BF16
    # parts (2^-17 per product) and as many roundings as inputs per lane
    bound = 2.0 ** -22 + (2 * k / 32 + 16) * 2.0 ** -24
    if rows <= 4:
        bound += 2.0 ** -15
    size = np.sqrt(((np.abs(x).astype(np.float64) ** 2) @ (dense(q, scales).T ** 2)))
    assert np.all(np.abs(got - ref) <= bound * size * 4 + 1e-30), (k, rows, n, f32x)
    assert not np.any(got[rows // 2])
    assert np.array_equal(y16.download(np.uint16).reshape(rows, n),
                          syn.bf16_rne(got).reshape(rows, n))


@pytest.mark.parametrize("rows,k,widths", [(3, 1536, (70, 16)), (23, 1536, (100, 257, 16)),
                                           (40, 2048, (64, 33)), (9, 6144, (48, 48))])
def test_few_rows_several_weights_and_recorded(g4, rows, k, widths):
    # several weights in one launch (one slice of K) or one by one (three slices
    # and a sum), bit-identical to single calls and to every replay of a recording
    lins = [g4.W4Linear(*syn.w4_weights(k + w, w, k)[:2]) for w in widths]
    rng = np.random.default_rng(rows)
    xb = g4.Buffer.from_array(rng.standard_normal((rows, k)).astype(np.float32))
    one, many = ([g4.Buffer(rows * w * 4) for w in widths] for _ in range(2))
    for lin, y in zip(lins, one):
        lin.linear(xb.ptr, g4.F32, rows, y.ptr, g4.F32)
    want = [y.download(np.float32) for y in one]
    g4.W4Linear.linear_multi(lins, xb.ptr, g4.F32, rows, [y.ptr for y in many], g4.F32)
    for y, w in zip(many, want):
        np.testing.assert_array_equal(y.download(np.float32), w)
    with g4.Encoder() as enc:
        g4.W4Linear.linear_multi(lins, xb.ptr, g4.F32, rows, [y.ptr for y in many], g4.F32)
        lins[0].linear(xb.ptr, g4.F32, rows, one[0].ptr, g4.F32)
    for _ in range(3):
        for y in many + one[:1]:
            y.upload(np.zeros(y.nbytes // 4, np.float32))
        enc.cmdbuf.submit()
        for y, w in zip(many + one[:1], want + want[:1]):
            np.testing.assert_array_equal(y.download(np.float32), w)


@pytest.mark.parametrize("rows,widths", [(290, (2048, 256, 256)), (389, (2047, 250, 33)),
                                         (640, (1536, 640)), (1000, (600, 1001))])
@pytest.mark.parametrize("bf16_out", [False, True])
def test_several_weights_with_a_summed_split(g4, rows, widths, bf16_out):
    # joint launches whose K split is summed into each weight's output, at row
    # counts and widths whose products are and are not multiples of four
    k = 1536
    rng = np.random.default_rng([rows, len(widths)])
    x = rng.standard_normal((rows, k)).astype(np.float32)
    xb = g4.Buffer.from_array(x)
    lins, refs = [], []
    for n in widths:
        packed, scales, q = syn.w4_weights(n, n, k)
        lins.append(g4.W4Linear(packed, scales))
        refs.append(x.astype(np.float64) @ dense(q, scales).T)
    size = 2 if bf16_out else 4
    ys = [g4.Buffer(rows * n * size) for n in widths]
    g4.W4Linear.linear_multi(lins, xb.ptr, g4.F32, rows, [y.ptr for y in ys],
                             g4.BF16 if bf16_out else g4.F32)
    for y, n, ref in zip(ys, widths, refs):
        if bf16_out:
            got = syn.bf16_to_f32(y.download(np.uint16)).reshape(rows, n)
        else:
            got = y.download(np.float32).reshape(rows, n)
        # 22-bit x and FP32 sums; BF16 has 8 significant bits: half an ulp is at
        # most 2^-8 of each value
        assert rel_l2_rows(got, ref) <= 2e-6 + (2.0 ** -8 if bf16_out else 0)


@pytest.mark.parametrize("k", [16384, 32768])
@pytest.mark.parametrize("rows", [1, 3, 40])
@pytest.mark.parametrize("f32x", [False, True])
def test_long_in_dim_linear(g4, k, rows, f32x):
    # in_dims whose activation row no longer fits the GEMVs' LDS staging
    # (32768 BF16, 16384 and 32768 FP32) take the GEMM at every row count;
    # the reference's GPUOps.w4 takes any inDim
    rng = np.random.default_rng([k, rows, f32x])
    n = 300
    packed, scales, q = syn.w4_weights(k + rows, n, k)
    lin = g4.W4Linear(packed, scales)
    xb, x, xd = activations(g4, rng, rows, k, f32x)
    y32 = g4.Buffer(rows * n * 4)
    lin.linear(xb.ptr, xd, rows, y32.ptr, g4.F32)
    ref = x.astype(np.float64) @ dense(q, scales).T
    assert rel_l2_rows(y32.download(np.float32).reshape(rows, n), ref) <= 1e-4
    ys = [g4.Buffer(rows * w * 4) for w in (64, 200)]
    lins = [g4.W4Linear(*syn.w4_weights(k + w, w, k)[:2]) for w in (64, 200)]
    g4.W4Linear.linear_multi(lins, xb.ptr, xd, rows, [b.ptr for b in ys], g4.F32)
    for w, lw, yb in zip((64, 200), lins, ys):
        _, sc, qq = syn.w4_weights(k + w, w, k)
        r = x.astype(np.float64) @ dense(qq, sc).T
        assert rel_l2_rows(yb.download(np.float32).reshape(rows, w), r) <= 1e-4


@pytest.mark.parametrize("seed", range(16))
def test_random_linear_multi(g4, seed):
    rng, rows, _, k, f32x = draw(100 + seed)
    widths = [int(v) for v in rng.integers(1, 700, size=int(rng.integers(2, 4)))]
    lins, refs = [], []
    xb, x, xd = activations(g4, rng, rows, k, f32x)
    for i, n in enumerate(widths):
        packed, scales, q = syn.w4_weights(600 + 4 * seed + i, n, k)
        lins.append(g4.W4Linear(packed, scales))
        refs.append(x.astype(np.float64) @ dense(q, scales).T)
    ys = [g4.Buffer(rows * n * 4) for n in widths]
    g4.W4Linear.linear_multi(lins, xb.ptr, xd, rows, [y.ptr for y in ys], g4.F32)
    for y, n, ref in zip(ys, widths, refs):
        got = y.download(np.float32).reshape(rows, n)
        assert rel_l2_rows(got, ref) <= 1e-4, (rows, widths, k, f32x)


@pytest.mark.parametrize("seed", range(8))
def test_random_ple_geometry(g4, oracle, seed):
    # Random table geometry (vocab, width, rows per shard, a short last
    # shard) and ids with the edges: rows bit-exact against the oracle's
    # readRows restatement, BF16 the round-to-nearest-even of FP32.
    rng = np.random.default_rng(2000 + seed)
    width = 32 * int(rng.integers(1, 129))
    rps = 8 * int(rng.integers(1, 65))
    vocab = int(rng.integers(1, 5000))
    shards = syn.ple_table(300 + seed, vocab, width, rps, threads=4)
    t = g4.PleTable(vocab, width, 32, rps)
    for i, s in enumerate(shards):
        t.upload_shard(i, s)
    host = np.concatenate(shards)
    ids = rng.integers(0, vocab, size=int(rng.integers(1, 300))).astype(np.int32)
    ids[: min(3, len(ids))] = [0, vocab - 1, min(rps, vocab - 1)][: min(3, len(ids))]
    want = oracle.ple_gather(host, vocab, width, rps, ids)
    out = g4.Buffer(len(ids) * width * 4)
    t.gather(ids, out.ptr, g4.F32)
    assert np.array_equal(out.download(np.uint32).reshape(-1), want.view(np.uint32).reshape(-1))
    out16 = g4.Buffer(len(ids) * width * 2)
    t.gather(ids, out16.ptr, g4.BF16)
    assert np.array_equal(out16.download(np.uint16).reshape(-1), oracle.f32_to_bf16_array(want))
    t.free()


@pytest.mark.parametrize("seed", range(8))
def test_random_dequant(g4, oracle, seed):
    # dequantizeOfficialW4A16Rows over random shapes and row ranges, bit-exact.
    rng = np.random.default_rng(3000 + seed)
    n, k = int(rng.integers(1, 600)), 32 * int(rng.integers(1, 129))
    packed, scales, _ = syn.w4_weights(700 + seed, n, k)
    lin = g4.W4Linear(packed, scales)
    r0 = int(rng.integers(0, n))
    rc = int(rng.integers(0, n - r0 + 1))
    want_rc, want = oracle.w4_dequant_rows(packed, syn.bf16_to_f32(scales), n, k, r0, rc)
    assert want_rc == 0
    if rc == 0:
        return
    out = g4.Buffer(rc * k * 4)
    lin.dequant(r0, rc, out.ptr, g4.F32)
    assert np.array_equal(out.download(np.uint32).reshape(-1), want.view(np.uint32).reshape(-1))
