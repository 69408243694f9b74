"""Decode attention over 256-dim heads (xqhip_attn_decode: up to 32 context
splits per query head, passes of 256 positions, then the merge) against the
attention of customlib/runtime/custom_model.cpp:740-951 in 64 bits, at empty
splits, one position, sub-pass and pass edges and several passes.

Bound: scores and values in fp32 over hd products of size <= 8 (2^-24 each, rounding
errors of either sign): exp arguments within 1e-5, outputs (convex in |v| <= 6) within 1e-4."""
import numpy as np
import pytest

import xqbind as xb
from test_decode_ops_gpu import attn_layer_inputs, dev
from test_prefill_attn_gpu import want64

pytestmark = pytest.mark.gpu
HD, EPS = 256, 1e-6


@pytest.mark.parametrize("nq,nkv,rd,pos,gated", [
    (16, 4, 64, 0, True), (16, 4, 64, 1, True), (16, 4, 256, 15, False), (16, 4, 64, 17, True), (16, 4, 64, 2048, True),
    (16, 4, 64, 2049, True), (16, 4, 64, 4096, True), (16, 4, 64, 4200, False), (16, 4, 0, 9000, True),
    (8, 1, 64, 4000, True), (4, 4, 128, 1500, True), (40, 8, 64, 700, True), (300, 60, 64, 300, True)])
def test_matches_64_bit_attention(nq, nkv, rd, pos, gated):
    qsrc, k, v, qn, kn, kc, vc = attn_layer_inputs(nq, nkv, HD, pos, seed=pos + nq, gated=gated)
    tab = np.zeros(max(1, (pos + 1) * rd), np.float32)
    if rd:
        xb.ck(xb.hip().xqhip_rope_table(1e7, rd, pos + 1, xb.ptr(tab)))
    grow = lambda a: np.concatenate([a.reshape(pos, nkv, HD), np.full((40, nkv, HD), np.nan, np.float16)])  # noqa: E731
    kd, vd = dev(grow(kc)), dev(grow(vc))
    out = xb.DeviceBuffer(nq * HD * 4)
    ws = dev(np.full(xb.hip().xqhip_gqa_workspace_bytes(nq, nkv, HD) // 4, np.nan, np.float32))
    xb.ck(xb.hip().xqhip_attn_decode(dev(qsrc).ptr, dev(k).ptr, dev(v).ptr, int(gated), nq, nkv, HD, rd, dev(qn).ptr,
                                     dev(kn).ptr, EPS, dev(tab).ptr, dev(np.array([pos], np.int32)).ptr, kd.ptr, vd.ptr,
                                     pos + 40, out.ptr, ws.ptr, None))
    rows = qsrc.astype(np.float64).reshape(nq, -1)
    norm = lambda x, w: x / np.sqrt((x * x).mean(-1, keepdims=True) + EPS) * w.astype(np.float64)  # noqa: E731
    q, kk = norm(rows[:, :HD], qn), norm(k.astype(np.float64).reshape(nkv, HD), kn)
    if rd:
        cs = tab.astype(np.float64).reshape(-1, rd // 2, 2)[pos]
        for x in (q, kk):
            a, b = x[:, :rd // 2].copy(), x[:, rd // 2:rd].copy()
            x[:, :rd // 2], x[:, rd // 2:rd] = a * cs[:, 0] - b * cs[:, 1], b * cs[:, 0] + a * cs[:, 1]
    got_k = kd.download(np.float16, (pos + 40) * nkv * HD).reshape(pos + 40, nkv, HD)
    got_v = vd.download(np.float16, (pos + 40) * nkv * HD).reshape(pos + 40, nkv, HD)
    assert np.array_equal(got_v[pos].reshape(-1), v.astype(np.float16))
    assert np.abs(got_k[pos].astype(np.float64) - kk).max() <= 2.0**-10 * np.abs(kk).max()
    assert np.array_equal(got_k[:pos].reshape(-1), kc.reshape(-1)) and np.isnan(got_k[pos + 1:]).all()
    gate = rows[:, HD:] if gated else np.zeros((nq, HD))
    want = want64(q[None], gate[None], got_k[:pos + 1], got_v[:pos + 1], pos)[0]
    err = np.abs(out.download(np.float32, nq * HD).reshape(nq, HD) - want)
    assert err.max() <= 1e-4, err.max()
