"""What the ops hold in scratch, and what a recording does with the scratch it finds.
Scratch only grows, so each case runs in a process of its own."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def fresh(body):
    """Runs `body` in a new process with the library initialised; its stdout."""
    head = ("import sys; sys.path[:0] = %r\n"
            "import ctypes, numpy as np, g4hip as g4, layer_oracle as lo, synthetic as syn\n"
            "g4.init(0)\n"
            % [os.path.join(ROOT, "gemma4-js_amd"), os.path.join(ROOT, "oracle")])
    p = subprocess.run([sys.executable, "-c", head + body], stdout=subprocess.PIPE,
                       stderr=subprocess.PIPE, text=True, timeout=100)
    assert p.returncode == 0, p.stderr[-2000:]
    return p.stdout


@pytest.mark.parametrize("k", [1536, 6144, 12288])
@pytest.mark.parametrize("rows", [2, 3, 4])
def test_two_to_four_rows_use_no_scratch(k, rows):
    # recorded before anything has made scratch, from the static array's entry point
    # too, and eager: the same bits (in_dim 6144 and 12288 would split K over planes)
    fresh("""
k, rows = %d, %d
rng = np.random.default_rng(5)
pair = [g4.W4Linear(*syn.w4_weights(k + n, n, k)[:2]) for n in (1536, 48)]
x = g4.Buffer.from_array(rng.standard_normal((rows, k)).astype(np.float32))
ys = [g4.Buffer(rows * n * 4) for n in (1536, 1536, 1536, 48)]
def calls():
    pair[0].linear(x.ptr, g4.F32, rows, ys[0].ptr, g4.F32)
    pair[0].linear_noalloc(x.ptr, g4.F32, rows, ys[1].ptr, g4.F32)
    g4.W4Linear.linear_multi(pair, x.ptr, g4.F32, rows, [ys[2].ptr, ys[3].ptr], g4.F32)
with g4.Encoder() as enc:
    calls()
enc.cmdbuf.submit()
first = [y.download(np.uint32) for y in ys]
calls()
again = [y.download(np.uint32) for y in ys]
assert all(np.array_equal(a, b) for a, b in zip(first, again))
assert np.array_equal(first[0], first[1]) and np.array_equal(first[0], first[2])
""" % (k, rows))


def test_one_row_attention_holds_its_partials_only():
    # one row over 16384 keys at head dim 512: 1024 splits of 8 x 514 floats, 17 MB
    out = fresh("""
hip = ctypes.CDLL("libamdhip64.so")
def free():
    a, b = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
    return a.value
keys, hd = 16384, 512
q, y = g4.Buffer(8 * hd * 4), g4.Buffer(8 * hd * 4)
k, v = g4.Buffer(keys * hd * 4), g4.Buffer(keys * hd * 4)
g4.attention(q, k, v, 1, 8, hd, 64, 63, False, 0, y)
g4.sync()
before = free()
g4.attention(q, k, v, 1, 8, hd, keys, keys - 1, False, 0, y)
g4.sync()
print(before - free())
""")
    assert int(out) < 24 << 20, out


# The scratch that is there holds the FP32 split kernel's partials alone (60 rows), or
# also the many-row kernel's tiles but not all of its planes (100 rows).
@pytest.mark.parametrize("first_rows", [60, 100])
def test_attention_recorded_with_less_scratch_than_an_eager_call_takes(first_rows):
    fresh("""
first, rows, heads, hd, keys = %d, 6, 8, 512, 3000
rng = np.random.default_rng(6)
def buf(*shape):
    a = rng.standard_normal(shape).astype(np.float32)
    return a, g4.Buffer.from_array(a)
_, q0 = buf(first, heads * 64)
_, kv0 = buf(keys, 64)
y0 = g4.Buffer(first * heads * 64 * 4)
g4.attention(q0, kv0, kv0, first, heads, 64, keys, keys - first, False, 0, y0)
(q, qb), (k, kb), (v, vb) = buf(rows, heads * hd), buf(keys, hd), buf(keys, hd)
q *= np.float32(hd ** -0.5)
qb = g4.Buffer.from_array(q)
y = g4.Buffer(rows * heads * hd * 4)
call = lambda: g4.attention(qb, kb, vb, rows, heads, hd, keys, keys - rows, False, 0, y)
with g4.Encoder() as enc:
    call()
want = lo.attention(q, k, v, rows, heads, hd, keys, keys - rows, False, 0)
got = []
for _ in range(3):
    enc.cmdbuf.submit()
    got.append(y.download(np.float32).reshape(want.shape))
call()
eager = y.download(np.float32).reshape(want.shape)
for g in got + [eager]:
    np.testing.assert_allclose(g, want, rtol=2e-5, atol=1e-5)
    assert np.array_equal(g, got[0]) or g is eager
assert not np.array_equal(eager, got[0])  # another kernel or another key split
""" % first_rows)


def test_several_weights_recorded_with_less_scratch_than_an_eager_call_takes():
    # the scratch of the weights one by one does not hold the planes of all of them:
    # the recording takes one launch without a K split
    fresh("""
rows, k, widths = 389, 1536, (2048, 256, 256)
rng = np.random.default_rng(7)
x = rng.standard_normal((rows, k)).astype(np.float32)
xb = g4.Buffer.from_array(x)
lins, refs = [], []
for n in widths:
    packed, scales, q = syn.w4_weights(n, n, k)
    lins.append(g4.W4Linear(packed, scales))
    w = q.astype(np.float64) * np.repeat(syn.bf16_to_f32(scales).astype(np.float64), 32, axis=1)
    refs.append(x.astype(np.float64) @ w.T)
ys = [g4.Buffer(rows * n * 4) for n in widths]
for lin, y in zip(lins, ys):
    lin.linear(xb.ptr, g4.F32, rows, y.ptr, g4.F32)
def call():
    g4.W4Linear.linear_multi(lins, xb.ptr, g4.F32, rows, [y.ptr for y in ys], g4.F32)
def result():
    return [y.download(np.float32).reshape(rows, n) for y, n in zip(ys, widths)]
with g4.Encoder() as enc:
    call()
enc.cmdbuf.submit()
first = result()
call()
eager = result()
enc.cmdbuf.submit()
for got in (first, eager, result()):
    for g, ref in zip(got, refs):
        assert np.linalg.norm(g - ref) <= 2e-6 * np.linalg.norm(ref)
assert not all(np.array_equal(a, b) for a, b in zip(first, eager))
""")
