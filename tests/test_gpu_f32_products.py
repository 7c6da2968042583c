"""The four-wave f32 kernel's products, each f32 operand the sum of three bf16 parts: errors at the
level of f32 sums over magnitudes from 2^-112 to 2^112, tile and row remainders in both K layouts,
operands without such parts (infinite, huge, or tiny, alone or beside ordinary ones), weights down
to the smallest f32 holds, and masked keys of any value."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from ffai_amd import _lib as L
from ffai_amd import flash_attn as fa
from tests.helpers import randn

pytestmark = pytest.mark.gpu


@pytest.fixture
def split_override():
    prev = L.get_fwd_split_override()
    yield L.set_fwd_split_override
    L.set_fwd_split_override(*prev)


def _run(gpu, q, k, v, k_transposed, scale, **kw):
    kd = np.ascontiguousarray(np.swapaxes(k, 2, 3)) if k_transposed else k
    # (a fresh tensor: an axis of one key may carry any stride in numpy)
    q, kd, v = (torch.empty(x.shape, device=gpu).copy_(torch.from_numpy(x)) for x in (q, kd, v))
    out = torch.empty(q.shape, device=gpu)
    kw.update(k_transposed=k_transposed, scale=scale)
    assert fa.plan(q, kd, v, out, **kw)["shape"] == "wave4"
    assert fa.attention(q, kd, v, out=out, **kw) is not None
    return out.cpu().numpy().astype(np.float64)


def _exact(q, k, v, scale):
    q, k, v = (x.astype(np.float64) for x in (q, k, v))
    s = np.matmul(q, np.swapaxes(k, 2, 3)) * scale
    w = np.exp(s - s.max(-1, keepdims=True))
    return np.matmul(w / w.sum(-1, keepdims=True), v)


@pytest.mark.parametrize("k_transposed", [True, False])
@pytest.mark.parametrize("queries,keys", [(33, 1), (33, 3), (64, 63), (129, 64), (100, 65),
                                          (128, 127), (257, 1037), (64, 4098)])
def test_remainders(gpu, queries, keys, k_transposed):
    """Relative error in the 2-norm at most 1e-6: scores of 64 products (sqrt(64) / 2 steps of 2^-24
    of a score of ~1, so ~2.4e-7 of a weight), as many again from v_exp_f32 and the weighted sum."""
    rng = np.random.default_rng(queries * 5000 + keys)
    q, k, v = (randn(rng, (2, 3, n, 64)) for n in (queries, keys, keys))
    want = _exact(q, k, v, 0.125)
    got = _run(gpu, q, k, v, k_transposed, 0.125)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"{queries} x {keys} kt={k_transposed}: {err:.2e}")
    assert err < 1e-6


@pytest.mark.parametrize("e", [-100, -60, -20, 20, 60, 100])
def test_magnitudes(gpu, e):
    """Keys and values 2^e times wider (queries 2^-e), and values spread over 2^+-12 within a row: no
    magnitude loses bits (elements outside 2^-40 .. 2^30 send their workgroup to the f32 MFMA)."""
    rng = np.random.default_rng(600 + e)
    q, k, v = (randn(rng, (1, 2, n, 64)) for n in (96, 200, 200))
    v *= np.exp2(rng.integers(-12, 13, size=v.shape)).astype(np.float32)
    q, k, v = np.ldexp(q, -e), np.ldexp(k, e), np.ldexp(v, e)
    want = _exact(q, k, v, 0.125)
    got = _run(gpu, q, k, v, True, 0.125)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"2^{e}: {err:.2e}")
    assert err < 1e-6


@pytest.mark.parametrize("k_transposed", [True, False])
@pytest.mark.parametrize("e", [-28, -14, 14, 22])
def test_magnitudes_in_bf16_parts(gpu, e, k_transposed):
    """As above with every element from 2^-38 to 2^30, so that the products stay on bf16 parts, at
    either end of their range; queries and keys up to both ends as well."""
    rng = np.random.default_rng(630 + e)

    def draw(n, spread):
        x = randn(rng, (1, 2, n, 64))
        x = np.copysign(np.clip(np.abs(x), 2.0 ** -6, 8.0), x)
        return np.ldexp(x, rng.integers(-spread, spread + 1, size=x.shape)).astype(np.float32)

    q, k, v = np.ldexp(draw(96, 0), -e), np.ldexp(draw(200, 0), e), np.ldexp(draw(200, 4), e)
    for x in (q, k, v):
        assert np.abs(x).min() >= 2.0 ** -38 and np.abs(x).max() <= 2.0 ** 31
    v = np.clip(v, -2.0 ** 30, 2.0 ** 30)
    want = _exact(q, k, v, 0.125)
    got = _run(gpu, q, k, v, k_transposed, 0.125)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"2^{e}: {err:.2e}")
    assert err < 1e-6


@pytest.mark.parametrize("k_transposed", [True, False])
def test_infinite_and_largest_elements(gpu, k_transposed):
    """An infinite value reaches its column only, values near the largest f32 stay finite, and keys
    at -inf score -inf and weigh nothing, in the first tile, a later one and the tail."""
    rng = np.random.default_rng(620)
    q, k, v = (randn(rng, (1, 3, n, 64)) for n in (130, 200, 200))
    q[..., 5] = np.abs(q[..., 5]) + 0.1
    gone = [3, 100, 199]
    k[0, 0, gone, 5] = -np.inf          # head 0: three keys at -inf
    v[0, 1, 70, 9] = np.inf             # head 1: column 9 infinite
    v[0, 2, 198, 11] = 3.4e38           # head 2: column 11 huge
    kept = [j for j in range(200) if j not in gone]
    got = _run(gpu, q, k, v, k_transposed, 0.125)
    want0 = _exact(q[:, :1], k[:, :1, kept], v[:, :1, kept], 0.125)
    assert np.linalg.norm(got[:, :1] - want0) / np.linalg.norm(want0) < 1e-6
    cols = [d for d in range(64) if d != 9]
    want1 = _exact(q[:, 1:2], k[:, 1:2], v[:, 1:2][..., cols], 0.125)
    assert np.all(np.isposinf(got[:, 1, :, 9]))
    assert np.linalg.norm(got[:, 1:2][..., cols] - want1) / np.linalg.norm(want1) < 1e-6
    want2 = _exact(q[:, 2:], k[:, 2:], v[:, 2:], 0.125)
    err = np.abs(got[:, 2:] - want2) / np.abs(want2).max((2,), keepdims=True)
    assert err.max() < 4e-6


def test_a_tiny_column_beside_others(gpu):
    """A column of V at 2^-118 beside columns at 1 keeps its own relative precision."""
    rng = np.random.default_rng(640)
    q, k, v = (randn(rng, (1, 2, n, 64)) for n in (70, 150, 150))
    v[0, 1, :, 20] = np.ldexp(v[0, 1, :, 20], -118)
    want = _exact(q, k, v, 0.125)
    got = _run(gpu, q, k, v, False, 0.125)
    err = np.linalg.norm(got - want, axis=2) / np.linalg.norm(want, axis=2)
    assert err.max() < 1.2e-6


@pytest.mark.parametrize("tiny", [2.0 ** -92, 1.0e-36, 1.2345e-39])
@pytest.mark.parametrize("k_transposed", [True, False])
def test_a_tiny_value_beside_others(gpu, tiny, k_transposed):
    """One tiny value (the last a subnormal) among keys and columns at 1: a causal row that sees its
    key alone returns it (weight 1, so to the rounding of 1 / l), and every row keeps its error."""
    rng = np.random.default_rng(650)
    q, k, v = (randn(rng, (1, 2, n, 64)) for n in (70, 150, 150))
    v[0, 1, 0, 20] = np.float32(tiny)
    v[0, 1, 1, 20] = 1.0
    got = _run(gpu, q, k, v, k_transposed, 0.125, causal=True)
    want0 = v[:, :, 0].astype(np.float64)
    assert np.max(np.abs(got[:, :, 0] - want0) / np.abs(want0)) < 3e-7
    for row in (1, 2, 69):
        want = _exact(q[:, :, row:row + 1], k[:, :, :row + 1], v[:, :, :row + 1], 0.125)
        assert np.linalg.norm(got[:, :, row:row + 1] - want) / np.linalg.norm(want) < 1e-6, row


@pytest.mark.parametrize("k_transposed", [True, False])
@pytest.mark.parametrize("tiny,large", [(1.0e-36, 1.0e36), (1.2345e-39, 1.0e38)])
def test_a_tiny_key_element_against_a_large_query_one(gpu, tiny, large, k_transposed):
    """Scores that rest on one dimension, tiny in every key and large in every query, the other
    dimensions ordinary (a subnormal of ~20 bits: its parts are exact, its products f32's)."""
    rng = np.random.default_rng(660)
    q, k, v = (randn(rng, (1, 2, n, 64)) for n in (70, 150, 150))
    q[..., 6] = np.float32(large) * np.sign(q[..., 6])
    k[..., 6] *= np.float32(tiny)
    want = _exact(q, k, v, 0.125)
    got = _run(gpu, q, k, v, k_transposed, 0.125)
    assert np.linalg.norm(got - want) / np.linalg.norm(want) < 1e-6


@pytest.mark.parametrize("keys,at,pieces", [(64, 9, 1), (200, 9, 1), (200, 150, 1), (200, 150, 4)])
@pytest.mark.parametrize("log2_weight", [-90, -107, -113, -119, -124])
def test_small_weights_keep_their_bits(gpu, split_override, log2_weight, keys, at, pieces):
    """A column whose only nonzero value stands behind a small weight, in the first tile or a later
    one, the item whole or in pieces: the output is that weight. Its score, ~|log2_weight| in base
    2, carries 2^-24 of itself from each of the score, scale and exponent roundings, so the weight 3
    |log2_weight| 2^-24 ln 2 of itself; twice that allowed, and the step of the subnormals."""
    split_override(-1, pieces)
    rng = np.random.default_rng(670)
    q, k, v = (randn(rng, (1, 2, n, 64)) for n in (70, keys, keys))
    q[...], k[...] = 0.0, 0.0
    q[..., 0] = 1.0 + rng.random((1, 2, 70), dtype=np.float32) / 64
    k[..., at, 0] = log2_weight * np.log(2.0)
    v[..., 33] = 0.0
    v[..., at, 33] = 1.0
    want = _exact(q, k, v, 1.0)[..., 33]
    got = _run(gpu, q, k, v, True, 1.0)[..., 33]
    kept = want * keys > 2.0 ** -126  # (exp2 flushes a smaller weight)
    assert kept.any()
    err = np.max(((np.abs(got - want) - 2.0 ** -149) / want)[kept])
    print(f"weight 2^{log2_weight}: {err:.2e}")
    assert err < 6 * abs(log2_weight) * 1.02 * 2.0 ** -24 * np.log(2.0)


@pytest.mark.parametrize("k_transposed", [True, False])
def test_scores_below_the_f32_range_weigh_nothing(gpu, k_transposed):
    """Finite elements whose products pass -3.4e38, by so much that the products of their parts do
    too, with either sign: the score is -inf in f32, its weight 0."""
    rng = np.random.default_rng(680)
    q, k, v = (randn(rng, (1, 3, n, 64)) for n in (130, 200, 200))
    q[..., 5] = np.float32(3e21) * (1 + rng.random((1, 3, 130), dtype=np.float32))
    k[..., 5] = 0.0
    gone = [3, 64, 100, 199]
    k[:, :, gone, 5] = np.float32(-3e21) * (1 + rng.random((1, 3, 4), dtype=np.float32))
    kept = [j for j in range(200) if j not in gone]
    got = _run(gpu, q, k, v, k_transposed, 0.125)
    want = _exact(q, k[:, :, kept], v[:, :, kept], 0.125)
    assert np.linalg.norm(got - want) / np.linalg.norm(want) < 1e-6


@pytest.mark.parametrize("k_transposed", [True, False])
@pytest.mark.parametrize("lens", [1, 62, 130, 190])
def test_masked_keys_change_nothing(gpu, lens, k_transposed):
    """Keys and values past a window's length, whatever they hold (infinite, huge, tiny, subnormal),
    leave every bit of the result as zeros there do."""
    rng = np.random.default_rng(690 + lens)
    q, k, v = (randn(rng, (1, 2, n, 64)) for n in (70, 201, 201))
    n = torch.tensor([lens], dtype=torch.int32, device=gpu)
    k[:, :, lens:], v[:, :, lens:] = 0.0, 0.0
    want = _run(gpu, q, k, v, k_transposed, 0.125, kv_lens=n)
    assert np.linalg.norm(want - _exact(q, k[:, :, :lens], v[:, :, :lens], 0.125)) / \
        np.linalg.norm(want) < 1e-6
    for x in (np.inf, 3e38, 1e-30, 1e-40):
        k[:, :, lens:], v[:, :, lens:] = x, x
        assert np.array_equal(_run(gpu, q, k, v, k_transposed, 0.125, kv_lens=n), want), x
