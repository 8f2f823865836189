"""Values far apart in size within one call: what a small value contributes must not
depend on the large ones beside it, as with FP32 operands."""
import numpy as np
import pytest

import layer_oracle as lo

pytestmark = pytest.mark.gpu


def attend(g4, q, k, v, qrows, heads, hd, keylen, qpos0):
    y = g4.Buffer(qrows * heads * hd * 4)
    b = [g4.Buffer.from_array(np.ascontiguousarray(a, np.float32)) for a in (q, k, v)]
    g4.attention(b[0], b[1], b[2], qrows, heads, hd, keylen, qpos0, False, 0, y)
    return y.download(np.float32).reshape(qrows, heads * hd)


def attention_case(hd, seed, qrows=12, heads=8, keylen=600):
    """q, k and v of many rows over a long cache (the split-operand kernel)."""
    rng = np.random.default_rng([seed, hd])
    q = rng.standard_normal((qrows, heads * hd)).astype(np.float32) * np.float32(hd ** -0.25)
    k = rng.standard_normal((keylen, hd)).astype(np.float32) * np.float32(hd ** -0.25)
    v = rng.standard_normal((keylen, hd)).astype(np.float32)
    return q, k, v, qrows, heads, hd, keylen, keylen - qrows


def assert_small_values_kept(g4, case, bound):
    # every element against its own sum p |v|, whatever stands in the other dims
    q, k, v = case[:3]
    got = attend(g4, *case)
    want = lo.attention(q, k, v, *case[3:], False, 0)
    size = lo.attention(q, k, np.abs(v), *case[3:], False, 0)
    bad = np.abs(got - want) > bound * size
    assert not bad.any(), (int(bad.sum()), float((np.abs(got - want) / np.maximum(size, 1e-38)).max()))


# Bound: p carries its score's rounding (2^-24 |s|, |s| < 8, a few of them) and the
# outputs a few roundings of 2^-24: below 2^-19 of sum p |v|.
@pytest.mark.parametrize("hd", [256, 512])
@pytest.mark.parametrize("big", [1e6, 1e12, 1e30])
@pytest.mark.parametrize("where", ["a dim of every key", "an element of one key"])
def test_attention_keeps_small_values_beside_large_ones(g4, hd, big, where):
    case = attention_case(hd, 31)
    v = case[2]
    if where == "a dim of every key":
        v[:, 5] *= np.float32(big)
    else:
        v[77, 5] = big
    assert_small_values_kept(g4, case, 2.0 ** -19)


@pytest.mark.parametrize("hd", [256, 512])
def test_attention_keeps_small_weights_beside_large_ones(g4, hd):
    # keys with weights near e^-28 of the others' stand alone in half of the dims
    # (|s| < 40, so their weights are good to a few times 40 2^-24: 2^-17)
    case = attention_case(hd, 32)
    q, k, v = case[:3]
    few = np.arange(3, 588, 13)
    q.reshape(-1, hd)[:, 0] = 4.0
    k[:, 0] = 0.0
    k[few, 0] = -7.0
    alone = v[few, hd // 2:].copy()
    v[:, hd // 2:] = 0.0
    v[few, hd // 2:] = alone
    assert_small_values_kept(g4, case, 2.0 ** -17)


@pytest.mark.parametrize("hd", [256, 512])
def test_attention_keeps_tiny_values(g4, hd):
    # down to where FP32 itself ends: full precision while the values and their
    # 24 bits are normal numbers
    case = attention_case(hd, 33)
    case[2][:, ::3] *= np.float32(1e-28)
    case[2][:, 1::3] *= np.float32(1e-33)
    assert_small_values_kept(g4, case, 2.0 ** -19)


@pytest.mark.parametrize("hd", [256, 512])
@pytest.mark.parametrize("top,other", [(3e38, 2.9e38), (-8e29, -9e29)])
def test_attention_scores_at_the_ends_of_their_range(g4, hd, top, other):
    # all weight on key 40's and 41's equal maxima, up to FP32's largest scores and
    # down to the shader's masked logit of -1e30
    case = attention_case(hd, 34)
    q, k, v = case[:3]
    q[:] = 0.0
    q.reshape(-1, hd)[:, 0] = 1.5e19
    k[:, 0] = other / 1.5e19
    k[40:42, 0] = top / 1.5e19
    got = attend(g4, *case)
    want = np.tile(0.5 * (v[40] + v[41]), (case[3], case[4]))
    np.testing.assert_allclose(got, want, rtol=1e-6, atol=1e-6)
