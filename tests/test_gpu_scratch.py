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
