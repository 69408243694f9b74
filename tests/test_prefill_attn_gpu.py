"""The matrix-core prefill attention (head sizes 128 and 256) against the causal
attention of customlib/runtime/custom_model.cpp:840-951 in 64 bits, at the edges
of its tiles: 32- and 64-column blocks (tokens x query heads of a kv head), the
128- and 256-key chunks split over a block's waves, the last partial key tile.

Bound: q and the probabilities carry about 22 bits (fp16 hi + lo), so a score of
|q| |k| / sqrt(hd) <= 16 is off by at most 16 x 2^-22 and a probability by 4e-6
of itself; the output, a convex combination of |v| <= 6, by 3e-5."""
import ctypes

import numpy as np
import pytest

import xqbind as xb
from test_decode_ops_gpu import dev

pytestmark = pytest.mark.gpu
ATOL = 3e-5


def want64(q, gate, kc, vc, pos0):
    T, nq, hd = q.shape
    q, gate, kc, vc = (a.astype(np.float64) for a in (q, gate, kc, vc))
    group = nq // kc.shape[1]
    late = np.arange(pos0 + T)[None, :] > pos0 + np.arange(T)[:, None]
    out = np.empty_like(q)
    for h in range(nq):
        s = q[:, h] @ kc[:, h // group].T / np.sqrt(hd)
        s[late] = -np.inf
        p = np.exp(s - s.max(-1, keepdims=True))
        out[:, h] = p @ vc[:, h // group] / p.sum(-1, keepdims=True)
    return out / (1 + np.exp(-gate))


@pytest.mark.parametrize("q_scale", [1.0, 2.0**17])
@pytest.mark.parametrize("nq,nkv,hd,T,pos0", [
    (32, 8, 128, 512, 0), (32, 8, 128, 497, 15), (32, 8, 128, 1, 0), (32, 8, 128, 9, 255), (32, 8, 128, 16, 256),
    (16, 4, 128, 33, 1000), (3, 1, 128, 65, 31), (8, 8, 128, 40, 5), (14, 2, 128, 11, 127), (16, 2, 128, 8, 129),
    (16, 4, 256, 512, 1), (16, 4, 256, 17, 127), (16, 4, 256, 1, 700), (6, 2, 256, 50, 63), (16, 2, 256, 512, 0)])
def test_matches_64_bit_attention(nq, nkv, hd, T, pos0, q_scale):
    """q_scale 2^17 with keys of 2^-17: queries beyond fp16's range, the same scores."""
    rng = np.random.default_rng(T + pos0 + hd)
    kc = rng.normal(0, 1, (pos0 + T, nkv, hd)).astype(np.float16)
    if q_scale != 1.0:
        kc = (np.round(kc.astype(np.float32) * 64) / 64 / q_scale).astype(np.float16)  # subnormal, exact to 2^-6 of one
    vc = rng.normal(0, 1, kc.shape).astype(np.float16)
    q = (rng.normal(0, 1, (T, nq, hd)) * q_scale).astype(np.float32)
    gate = rng.normal(0, 1, q.shape).astype(np.float32)
    # rows past the context hold NaN: no key after a token's own may reach its output
    pad = np.full((70, nkv, hd), np.nan, np.float16)
    stride, n = nq * hd + 8, nq * hd
    row = lambda a: np.concatenate([a.reshape(T, n), np.full((T, 8), np.nan, np.float32)], 1)  # noqa: E731
    out = dev(np.full((T, stride), 7.0, np.float32))
    xb.ck(xb.hip().xqhip_prefill_attention(dev(row(q)).ptr, dev(row(gate)).ptr, dev(np.concatenate([kc, pad])).ptr,
                                           dev(np.concatenate([vc, pad])).ptr, nq, nkv, hd, T, stride,
                                           dev(np.array([pos0], np.int32)).ptr, out.ptr, stride, None))
    got = out.download(np.float32, T * stride).reshape(T, stride)
    assert (got[:, n:] == 7.0).all()
    err = np.abs(got[:, :n].reshape(q.shape) - want64(q, gate, kc, vc, pos0))
    assert err.max() <= ATOL, err.max()


def test_rows_off_16_bytes_take_the_general_kernel():
    nq, nkv, hd, T, pos0 = 8, 2, 128, 5, 3
    rng = np.random.default_rng(0)
    kc, vc = (rng.normal(0, 1, (pos0 + T, nkv, hd)).astype(np.float16) for _ in range(2))
    q, gate = (rng.normal(0, 1, (T, nq, hd)).astype(np.float32) for _ in range(2))
    stride = nq * hd + 1
    row = lambda a: np.concatenate([a.reshape(T, -1), np.zeros((T, 1), np.float32)], 1)  # noqa: E731
    out = xb.DeviceBuffer(T * stride * 4)
    xb.ck(xb.hip().xqhip_prefill_attention(dev(row(q)).ptr, dev(row(gate)).ptr, dev(kc).ptr, dev(vc).ptr, nq, nkv, hd,
                                           T, stride, dev(np.array([pos0], np.int32)).ptr, out.ptr, stride, None))
    got = out.download(np.float32, T * stride).reshape(T, stride)[:, :nq * hd].reshape(q.shape)
    assert np.abs(got - want64(q, gate, kc, vc, pos0)).max() <= ATOL


@pytest.mark.parametrize("nq,nkv,hd,T,pos0", [
    (32, 8, 128, 2, 0), (32, 8, 128, 8, 24), (32, 8, 128, 8, 25), (32, 8, 128, 12, 200), (8, 8, 128, 64, 0),
    (5, 1, 128, 30, 2), (32, 8, 128, 260, 0), (16, 4, 256, 2, 0), (16, 4, 256, 8, 24), (16, 4, 256, 8, 56),
    (16, 4, 256, 3, 110), (4, 4, 256, 64, 1)])
def test_short_contexts(nq, nkv, hd, T, pos0):
    """One to a few key tiles: the waves without a key are left out of the merge (edges of 32 keys, of a chunk, of the
    tokens and heads of a block)."""
    test_matches_64_bit_attention(nq, nkv, hd, T, pos0, 1.0)


@pytest.mark.parametrize("nq,nkv,hd", [(8, 2, 128), (8, 2, 256)])
@pytest.mark.parametrize("shift", [1, 2, 4])
def test_caches_off_16_bytes(nq, nkv, hd, shift):
    """Caches that start 2, 4 or 8 bytes into an allocation."""
    T, pos0 = 19, 41
    rng = np.random.default_rng(shift)
    kc, vc = (rng.normal(0, 1, (pos0 + T, nkv, hd)).astype(np.float16) for _ in range(2))
    q, gate = (rng.normal(0, 1, (T, nq, hd)).astype(np.float32) for _ in range(2))
    k, v = (dev(np.concatenate([np.zeros(shift, np.float16), a.reshape(-1)])) for a in (kc, vc))
    at = lambda b: ctypes.c_void_p(b.ptr.value + 2 * shift)  # noqa: E731
    out = xb.DeviceBuffer(q.nbytes)
    xb.ck(xb.hip().xqhip_prefill_attention(dev(q).ptr, dev(gate).ptr, at(k), at(v), nq, nkv, hd, T, nq * hd,
                                           dev(np.array([pos0], np.int32)).ptr, out.ptr, nq * hd, None))
    got = out.download(np.float32, q.size).reshape(q.shape)
    assert np.abs(got - want64(q, gate, kc, vc, pos0)).max() <= ATOL


SHAPES = [(16, 4, 256, 40, 3), (4, 4, 256, 9, 130), (32, 8, 128, 512, 0), (3, 1, 128, 33, 60), (16, 2, 128, 21, 300)]


def attend(q, gate, kc, vc, pos0):
    T, nq, hd = q.shape
    out = dev(np.full((T, nq * hd), 7.0, np.float32))
    # (the buffers live until the download: the launch does not wait)
    args = [dev(a) for a in (q, gate, kc, vc, np.array([pos0], np.int32))]
    xb.ck(xb.hip().xqhip_prefill_attention(args[0].ptr, args[1].ptr, args[2].ptr, args[3].ptr, nq, kc.shape[1], hd, T,
                                           nq * hd, args[4].ptr, out.ptr, nq * hd, None))
    return out.download(np.float32, T * nq * hd).reshape(q.shape)


@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("nq,nkv,hd,T,pos0", SHAPES)
def test_a_value_that_is_not_finite_reaches_its_own_and_later_tokens_only(nq, nkv, hd, T, pos0, value):
    """A value beyond fp16's range is an infinity in the cache: tokens before it are as if it were not there, its own
    and later ones get it in that dim."""
    rng = np.random.default_rng(T + pos0)
    kc, vc = (rng.normal(0, 1, (pos0 + T, nkv, hd)).astype(np.float16) for _ in range(2))
    q, gate = (rng.normal(0, 1, (T, nq, hd)).astype(np.float32) for _ in range(2))
    want = want64(q, gate, kc, vc, pos0)
    t, kh, d = T - 3, nkv - 1, hd - 5
    vc[pos0 + t, kh, d] = value
    got = attend(q, gate, kc, vc, pos0)
    heads, group = slice(kh * nq // nkv, None), nq // nkv
    assert group == got[:, heads].shape[1]
    np.testing.assert_array_equal(got[t:, heads, d], np.full((T - t, group), value, np.float32))
    want[t:, heads, d] = got[t:, heads, d] = 0.0
    assert np.abs(got - want).max() <= ATOL


@pytest.mark.parametrize("nq,nkv,hd,T,pos0", SHAPES)
def test_scores_near_the_lowest_value(nq, nkv, hd, T, pos0):
    """All scores -1e30 sqrt(hd), as a mask of large negative queries gives: the mean of the values."""
    rng = np.random.default_rng(T + pos0)
    vc = rng.normal(0, 1, (pos0 + T, nkv, hd)).astype(np.float16)
    q, gate = np.full((T, nq, hd), -1e30, np.float32), np.zeros((T, nq, hd), np.float32)
    got = attend(q, gate, np.ones_like(vc), vc, pos0)
    assert np.abs(got - want64(q, gate, np.ones_like(vc), vc, pos0)).max() <= ATOL
