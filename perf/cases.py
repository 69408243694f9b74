"""The calls whose time counts: one decode token's and one prompt's work through
the C ABIs (include/xqhip.h per kernel family and layer, include/xqwen35.h for a
whole session), over the shapes of the 9B-shaped benchmark model, the head
layouts of the tests and odd sizes between them.

  listed()            the cases by name
  draw(rng)           one more case of the same ranges
  prepare(case, seed) inputs, weights, workspaces and captured graphs on the GPU
  run(state)          one pass, its outputs
  work, tolerance, exact   the bytes and operations of a pass, the error another
                      correct implementation may show, the result in 64 bits
"""
import ctypes
import json
import math
import os
import shutil
import struct
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "yingjie-work-trial-mnn-custom-inference-library_amd", "python"))
import xqbind as xb  # noqa: E402

GROUP, EPS, THETA, KSIZE = 64, 1e-6, 1e7, 4
F64 = torch.float64

# The session's model: the 9B-shaped model's layer pattern and head sizes at
# half its hidden size, four layers, so that it is written in about a second.
SESSION = dict(hidden_size=2048, intermediate_size=8192, vocab_size=16384, num_layers=4, num_attention_heads=16,
               num_key_value_heads=4, head_dim=128, linear_key_head_dim=128, linear_value_head_dim=128,
               linear_num_key_heads=8, linear_num_value_heads=16)


def listed():
    return [
        # one projection on its own, fp16 in and out: the smallest call a program makes
        dict(name="gemv_4096", kind="gemv", rows=4096, cols=4096, bits=4, meta="sym", pro="none", epi="store", f16=True),
        # a linear-attention layer of the 9B shape for one token, as a captured graph
        # (three of four layers; five dependent launches)
        dict(name="layer_linear", kind="layer", full=False, hidden=4096, inter=12288, n_a=16, n_b=32, hd=128, pos=540,
             meta="sym"),
        # a full-attention layer for one token after a 512-token prompt, with the
        # metadata the packer's default (asymmetric) quantiser writes
        dict(name="layer_full_asym", kind="layer", full=True, hidden=4096, inter=12288, n_a=32, n_b=8, hd=128, pos=540,
             meta="asym"),
        # final norm, lm_head and greedy sampling: the largest matrix of a step
        dict(name="lm_head", kind="lm_head", rows=248320, cols=4096, meta="sym"),
        # decode attention in a long conversation
        dict(name="attn_decode_8k", kind="attn_decode", nq=32, nkv=8, hd=128, pos=8100),
        # the same step with 256-wide heads
        dict(name="attn_decode_256", kind="attn_decode", nq=16, nkv=4, hd=256, pos=2000),
        # gate/up projection of a whole 512-token prompt chunk: where a prefill's time goes
        dict(name="gemm_512", kind="gemm", rows=24576, cols=4096, m=512, meta="sym", pro="rms", epi="silu"),
        # input projection of a one-sentence prompt
        dict(name="gemm_21", kind="gemm", rows=12352, cols=4096, m=21, meta="sym", pro="rms", epi="store"),
        # the eighth 512-token chunk of a long prompt
        dict(name="attn_prefill_3584", kind="attn_prefill", nq=32, nkv=8, hd=128, tokens=512, pos0=3584),
        # 256-wide heads, a ragged second chunk
        dict(name="attn_prefill_256", kind="attn_prefill", nq=16, nkv=4, hd=256, tokens=333, pos0=512),
        # linear attention over a prompt chunk, the last 64-token block partial
        dict(name="scan_500", kind="scan", lk=16, lv=32, tokens=500),
        # a whole request: 300-token prompt, 16 greedy tokens
        dict(name="session_300_16", kind="session", prompt=300, new=16, asym=False),
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of `step` between lo and hi, spread over the logarithm."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi + 0.999)))
    return max(lo, min(hi, int(v / step) * step))


def draw(rng):
    kind = rng.choice(["gemv", "layer", "attn_decode", "gemm", "gemm", "attn_prefill", "scan", "session"])
    if kind == "gemv":
        pro = rng.choice(["none", "rms"])
        epi = rng.choice(["store", "add", "silu"])
        bits = rng.choice([4, 4, 4, 3, 2])
        return dict(kind=kind, rows=_log(rng, 64, 24576) // 2 * 2, cols=_log(rng, 512, 12288, GROUP), bits=bits,
                    meta=rng.choice(["sym", "asym"]) if bits == 4 else "pair", pro=pro, epi=epi, f16=epi == "store" and
                    rng.random() < 0.3)
    if kind == "layer":
        hidden = _log(rng, 1024, 4096, GROUP)
        full = rng.random() < 0.4
        n_b = rng.choice([2, 4, 8]) if full else rng.choice([8, 16, 32])
        return dict(kind=kind, full=full, hidden=hidden, inter=_log(rng, hidden, 12288, GROUP),
                    n_a=4 * n_b if full else n_b // 2, n_b=n_b, hd=128, pos=_log(rng, 1, 6000),
                    meta=rng.choice(["sym", "asym"]))
    if kind == "attn_decode":
        nq, nkv, hd = rng.choice([(32, 8, 128), (32, 8, 128), (16, 4, 128), (16, 4, 256)])
        return dict(kind=kind, nq=nq, nkv=nkv, hd=hd, pos=_log(rng, 1, 16000))
    if kind == "gemm":
        epi = rng.choice(["store", "add", "silu"])
        return dict(kind=kind, rows=_log(rng, 512, 24576) // 2 * 2, cols=_log(rng, 1024, 12288, GROUP),
                    m=_log(rng, 2, 512), meta=rng.choice(["sym", "sym", "asym"]), pro=rng.choice(["none", "rms"]),
                    epi=epi)
    if kind == "attn_prefill":
        nq, nkv, hd = rng.choice([(32, 8, 128), (32, 8, 128), (16, 4, 128), (16, 4, 256)])
        return dict(kind=kind, nq=nq, nkv=nkv, hd=hd, tokens=_log(rng, 2, 512), pos0=rng.choice([0, _log(rng, 1, 6000)]))
    if kind == "scan":
        lk = rng.choice([8, 16])
        return dict(kind=kind, lk=lk, lv=2 * lk, tokens=_log(rng, 2, 512))
    return dict(kind=kind, prompt=_log(rng, 2, 700), new=_log(rng, 2, 32), asym=rng.random() < 0.5)


# ---- inputs ------------------------------------------------------------------
class _Rand:
    """Seeded values on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0):
        return torch.randn(*shape, generator=self.g, device="cuda") * std + mean

    def matrix(self, rows, cols, meta, bits=4):
        """Packed codes, fp32 scales and zeros of a group-64 matrix: uniform codes,
        scales |N(0, 0.02)|; `sym`: fp16 scales, zero at the middle code; `asym`:
        fp32 scales and integer zeros; `pair`: fp16 scales and zeros."""
        n = rows * cols // GROUP
        packed = torch.randint(0, 256, (rows * cols * bits // 8,), generator=self.g, device="cuda", dtype=torch.uint8)
        scales = self.normal(n, std=0.02).abs()
        if meta == "sym":
            return packed, scales.half().float(), torch.full((n,), 8.0, device="cuda"), bits
        mid = (1 << bits) / 2 - 0.5
        zeros = (self.normal(n) + mid).round().clamp(0, (1 << bits) - 1)
        return packed, scales.half().float() if meta == "pair" else scales, zeros, bits


def _inputs(case, seed):
    r = _Rand(seed)
    k = case["kind"]
    if k in ("gemv", "gemm", "lm_head"):
        rows, cols = case["rows"], case["cols"]
        m = case.get("m", 1)
        d = dict(w=r.matrix(rows, cols, case["meta"], case.get("bits", 4)), x=r.normal(m, cols),
                 norm=r.normal(cols, std=0.1, mean=1.0))
        if case.get("f16"):
            d["x"] = d["x"].half()
        if k == "lm_head":
            d["table"] = (r.normal(rows, cols) * 0.02).bfloat16()
        elif case["epi"] != "silu":
            d["y0"] = r.normal(m, rows) if case["epi"] == "add" else torch.zeros(m, rows, device="cuda")
        return d
    if k == "layer":
        h, i, na, nb, hd = case["hidden"], case["inter"], case["n_a"], case["n_b"], case["hd"]
        width = (na if case["full"] else nb) * hd
        n_in = 2 * na * hd + 2 * nb * hd if case["full"] else 2 * na * hd + 2 * nb * hd + 2 * nb
        d = dict(w_in=r.matrix(n_in, h, case["meta"]), w_out=r.matrix(h, width, case["meta"]),
                 w_gu=r.matrix(2 * i, h, case["meta"]), w_down=r.matrix(h, i, case["meta"]), x=r.normal(1, h),
                 n1=r.normal(h, std=0.1, mean=1.0), n2=r.normal(h, std=0.1, mean=1.0))
        d.update(_attn_inputs(r, na, nb, hd, case["pos"], 1) if case["full"] else _linear_inputs(r, na, nb))
        if not case["full"]:
            d["lin_norm"] = r.normal(hd, std=0.1, mean=1.0)
        return d
    if k == "attn_decode":
        d = _attn_inputs(r, case["nq"], case["nkv"], case["hd"], case["pos"], 1)
        d["proj"] = r.normal(1, 2 * (case["nq"] + case["nkv"]) * case["hd"])
        return d
    if k == "attn_prefill":
        n = case["nq"] * case["hd"]
        d = _attn_inputs(r, case["nq"], case["nkv"], case["hd"], case["pos0"], case["tokens"])
        d.update(q=r.normal(case["tokens"], n), gate=r.normal(case["tokens"], n))
        return d
    d = _linear_inputs(r, case["lk"], case["lv"])  # scan
    d["proj"] = r.normal(case["tokens"], 128 * (2 * case["lk"] + case["lv"]) + 2 * case["lv"])
    return d


def _attn_inputs(r, nq, nkv, hd, pos, new):
    """Caches of `pos` tokens with room for `new`, head norms and the rotary table."""
    ctx = pos + new
    return dict(kc=r.normal(ctx, nkv, hd).half(), vc=r.normal(ctx, nkv, hd).half(),
                qn=r.normal(hd, std=0.1, mean=1.0), kn=r.normal(hd, std=0.1, mean=1.0),
                rope=torch.from_numpy(_rope_table(ctx, hd // 4)).cuda())


def _linear_inputs(r, lk, lv):
    cd = 128 * (2 * lk + lv)
    return dict(conv=r.normal(cd, KSIZE, std=0.3), hist=r.normal(2, cd, KSIZE - 1), a_log=r.normal(lv, std=0.5),
                dt=r.normal(lv, std=0.5), S=r.normal(lv, 128, 128, std=0.1))


def _rope_table(n, rot):
    """(cos, sin) [n][rot / 2] in the float32 steps of the host's libm."""
    libm = ctypes.CDLL("libm.so.6")
    libm.powf.restype, libm.powf.argtypes = ctypes.c_float, [ctypes.c_float, ctypes.c_float]
    f = np.array([libm.powf(THETA, np.float32(-2 * i) / np.float32(rot)) for i in range(rot // 2)], np.float32)
    ang = (np.arange(n, dtype=np.float32)[:, None] * f).astype(np.float64)
    return np.stack([np.cos(ang), np.sin(ang)], -1).astype(np.float32)


# ---- what a program holds before the call, and the call ----------------------------
def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _upload(w, rows, cols):
    packed, scales, zeros, bits = w
    return xb.DeviceW4(packed.cpu().numpy(), scales.cpu().numpy(), zeros.cpu().numpy(), rows, cols, bits=bits)


def _pro(mode, weight=None, gate=None, head_dim=0):
    return xb.Prologue(mode, head_dim, _p(weight) if weight is not None else None,
                       _p(gate) if gate is not None else None, EPS)


def _ref(pro):
    return ctypes.byref(pro) if pro is not None else None


def _zeros(*shape, dtype=torch.float32):
    return torch.zeros(*shape, device="cuda", dtype=dtype)


EPI = dict(store=xb.EPI_STORE, add=xb.EPI_ADD, silu=xb.EPI_SILU_PAIR)


class _State:
    """The tensors and handles of a case, and the calls of one pass."""

    def __init__(self, case):
        self.case, self.calls, self.graph, self.outputs, self.slot = case, [], None, None, None

    def call(self, name, *args):
        self.calls.append((getattr(xb.hip(), name), args))

    def launch(self):
        for fn, args in self.calls:
            xb.ck(fn(*args))

    def capture(self):
        """The calls as one graph, as the session's decode step runs them."""
        L, stream, g = xb.hip(), ctypes.c_void_p(), ctypes.c_void_p()
        torch.cuda.synchronize()
        xb.ck(L.xqhip_stream_create(ctypes.byref(stream)))
        self.calls = [(fn, args[:-1] + (stream,)) for fn, args in self.calls]
        xb.ck(L.xqhip_graph_begin(stream))
        self.launch()
        xb.ck(L.xqhip_graph_end(stream, ctypes.byref(g)))
        xb.ck(L.xqhip_stream_destroy(stream))
        self.graph, self.calls = g, [(L.xqhip_graph_launch, (g, None))]

    def __del__(self):
        if self.graph:
            xb.hip().xqhip_graph_destroy(self.graph)
        if self.slot:
            xb.hip().xqhip_host_free(self.slot)


def prepare(case, seed):
    if case["kind"] == "session":
        return _prepare_session(case, seed)
    s, L, k = _State(case), xb.hip(), case["kind"]
    s.d = d = _inputs(case, seed)
    if k in ("gemv", "gemm", "lm_head"):
        rows, cols = case["rows"], case["cols"]
        s.w = _upload(d.pop("w"), rows, cols)
        s.pro = None if case.get("pro") == "none" else _pro(xb.PRO_RMS, d["norm"])
        if k == "lm_head":
            s.ws = _zeros(L.xqhip_argmax_workspace_bytes(rows), dtype=torch.uint8)
            s.idx, s.pos = _zeros(1, dtype=torch.int32), _zeros(1, dtype=torch.int32)
            s.val, s.emb, s.slot = _zeros(1), _zeros(cols), ctypes.c_void_p()
            xb.ck(L.xqhip_host_alloc_coherent(ctypes.byref(s.slot), 8))
            s.call("xqhip_gemv_w4a16_argmax_publish_embed", s.w.ref, _p(d["x"]), xb.F32, _ref(s.pro), _p(s.ws),
                   _p(s.idx), _p(s.val), _p(s.pos), s.slot, _p(d["table"]), rows, cols, _p(s.emb), None)
            s.outputs = dict(index=s.idx, value=s.val, row=s.emb)
            return s
        m, n = case.get("m", 1), rows // 2 if case["epi"] == "silu" else rows
        y = d["y0"] if "y0" in d else _zeros(m, n)
        if k == "gemv":
            y = y.half() if case["f16"] else y
            t = xb.F16 if case["f16"] else xb.F32
            s.call("xqhip_gemv_w4a16", s.w.ref, _p(d["x"]), t, _ref(s.pro), _p(y), t, EPI[case["epi"]], None)
        else:
            s.ws = _zeros(L.xqhip_gemm_workspace_bytes(m, cols, rows), dtype=torch.uint8)
            s.call("xqhip_gemm_w4a16", s.w.ref, _p(d["x"]), m, cols, _ref(s.pro), 0, _p(y), n, EPI[case["epi"]],
                   _p(s.ws), s.ws.numel(), None)
        s.outputs = dict(y=y)
    elif k == "layer":
        h, i, na, nb, hd = case["hidden"], case["inter"], case["n_a"], case["n_b"], case["hd"]
        width, n_in = (na if case["full"] else nb) * hd, len(d["w_in"][1]) * GROUP // h
        s.w = [_upload(d.pop("w_in"), n_in, h), _upload(d.pop("w_out"), h, width), _upload(d.pop("w_gu"), 2 * i, h),
               _upload(d.pop("w_down"), h, i)]
        s.proj, s.attn, s.ffn = _zeros(n_in), _zeros(width), _zeros(i)
        s.pos = torch.tensor([case["pos"]], dtype=torch.int32, device="cuda")
        z = s.proj[128 * (2 * na + nb) + 2 * nb:]
        s.pro = [_pro(xb.PRO_RMS, d["n1"]), _pro(xb.PRO_RMS, d["n2"]),
                 None if case["full"] else _pro(xb.PRO_GATED_HEAD_ACT, d["lin_norm"], z, hd)]
        gemv = lambda w, x, pro, y, epi: s.call("xqhip_gemv_w4a16", w.ref, _p(x), xb.F32, _ref(pro), _p(y),  # noqa: E731
                                                xb.F32, epi, None)
        gemv(s.w[0], d["x"], s.pro[0], s.proj, xb.EPI_STORE)
        if case["full"]:
            _decode_attention(s, d, s.proj, na, nb, hd, s.attn)
            s.outputs = dict(x=d["x"], kc=d["kc"], vc=d["vc"])
        else:
            cd = 128 * (2 * na + nb)
            s.call("xqhip_linear_attn_step_act", _p(s.proj), _p(d["hist"]), _p(d["conv"]), _p(s.proj[cd:]),
                   _p(s.proj[cd + nb:]), _p(d["a_log"]), _p(d["dt"]), _p(d["S"]), na, hd, nb, hd, KSIZE, _p(s.pos),
                   _p(s.attn), _p(z), None)
            s.outputs = dict(x=d["x"], S=d["S"], hist=d["hist"][(case["pos"] + 1) & 1])  # as the next position reads it
        gemv(s.w[1], s.attn, s.pro[2], d["x"], xb.EPI_ADD)
        gemv(s.w[2], d["x"], s.pro[1], s.ffn, xb.EPI_SILU_PAIR)
        gemv(s.w[3], s.ffn, None, d["x"], xb.EPI_ADD)
        s.capture()
    elif k == "attn_decode":
        s.pos = torch.tensor([case["pos"]], dtype=torch.int32, device="cuda")
        s.out = _zeros(case["nq"] * case["hd"])
        _decode_attention(s, d, d["proj"].reshape(-1), case["nq"], case["nkv"], case["hd"], s.out)
        s.outputs = dict(out=s.out, kc=d["kc"], vc=d["vc"])
    elif k == "attn_prefill":
        n, t = case["nq"] * case["hd"], case["tokens"]
        s.pos, s.out = torch.tensor([case["pos0"]], dtype=torch.int32, device="cuda"), _zeros(t, n)
        s.call("xqhip_prefill_attention", _p(d["q"]), _p(d["gate"]), _p(d["kc"]), _p(d["vc"]), case["nq"], case["nkv"],
               case["hd"], t, n, _p(s.pos), _p(s.out), n, None)
        s.outputs = dict(out=s.out)
    else:  # scan
        lk, lv, t = case["lk"], case["lv"], case["tokens"]
        cd, stride = 128 * (2 * lk + lv), d["proj"].shape[1]
        s.out = _zeros(t, lv * 128)
        s.ws = _zeros(L.xqhip_linear_scan_workspace_bytes(t, lk, 128, lv, 128), dtype=torch.uint8)
        a, b = d["proj"].reshape(-1)[cd:], d["proj"].reshape(-1)[cd + lv:]
        s.call("xqhip_linear_attn_scan_ws", _p(d["proj"]), _p(a), _p(b), stride, _p(d["hist"]), 0, _p(d["conv"]),
               _p(d["a_log"]), _p(d["dt"]), _p(d["S"]), lk, 128, lv, 128, KSIZE, t, _p(s.out), lv * 128, _p(s.ws), None)
        s.outputs = dict(out=s.out, S=d["S"], hist=d["hist"][t & 1])  # the copy the next position reads
    return s


def _decode_attention(s, d, proj, nq, nkv, hd, out):
    """The decode attention call the session makes for this head size and context."""
    L, k_src, v_src = xb.hip(), proj[2 * nq * hd:], proj[(2 * nq + nkv) * hd:]
    args = [_p(proj), _p(k_src), _p(v_src), 1, nq, nkv, hd, hd // 4, _p(d["qn"]), _p(d["kn"]), EPS, _p(d["rope"]),
            _p(s.pos), _p(d["kc"]), _p(d["vc"])]
    if hd != 128:
        s.attn_ws = _zeros(L.xqhip_gqa_workspace_bytes(nq, nkv, hd), dtype=torch.uint8)
        s.call("xqhip_attn_decode", *args, d["kc"].shape[0], _p(out), _p(s.attn_ws), None)
    elif d["kc"].shape[0] < 400:
        s.call("xqhip_attn_decode_head", *args, _p(out), None)
    else:
        s.attn_ws = _zeros(L.xqhip_attn_split_workspace_bytes(nq), dtype=torch.uint8)
        s.call("xqhip_attn_decode_split", *args, 8, _p(s.attn_ws), _p(out), None)


def _write_model(case, seed):
    where = tempfile.mkdtemp(prefix="xq_")
    xb.write_synth_model(where, seed=seed, asymmetric=int(case["asym"]), **SESSION)
    return where


def _prompt(case, seed):
    return np.random.default_rng(seed).integers(0, SESSION["vocab_size"], case["prompt"]).astype(np.int32)


def _prepare_session(case, seed):
    s = _State(case)
    where = _write_model(case, seed)
    try:
        s.session = xb.Session(where, xb.options(max_context=1024))
    finally:
        shutil.rmtree(where, ignore_errors=True)
    if not s.session.ok():
        raise RuntimeError("xq_create: %d" % s.session.status)
    s.tokens = _prompt(case, seed)
    return s


def run(s):
    if s.case["kind"] == "session":
        status, ids, _ = s.session.generate(s.tokens, s.case["new"])
        hidden_status, hidden, _ = s.session.hidden()
        debug_status, text = s.session.json("xq_get_debug_json", 1 << 14)
        if status or hidden_status or debug_status:
            raise RuntimeError("session: %d, %d, %d" % (status, hidden_status, debug_status))
        top = json.loads(text)["lm_head_topk"]
        return dict(tokens=ids, hidden=hidden, ids=np.array([t["token"] for t in top], np.int64),
                    logits=np.array([t["logit"] for t in top], np.float32))
    s.launch()
    return s.outputs


# ---- bytes and operations, tolerances ------------------------------------------------
def _matrix_bytes(rows, cols, meta, bits=4):
    return rows * cols * bits / 8 + rows * (cols // GROUP) * {"sym": 2, "asym": 4.5, "pair": 4}[meta]


def work(case):
    k = case["kind"]
    if k in ("gemv", "gemm", "lm_head"):
        rows, cols, m = case["rows"], case["cols"], case.get("m", 1)
        out = {"silu": rows // 2, "add": 2 * rows, "store": rows}[case["epi"]] if k != "lm_head" else 1.5 * cols / m
        one = 2 if case.get("f16") else 4
        return dict(bytes=_matrix_bytes(rows, cols, case["meta"], case.get("bits", 4)) + one * m * (cols + out),
                    flops=2.0 * rows * cols * m)
    if k == "layer":
        h, i, na, nb, hd = case["hidden"], case["inter"], case["n_a"], case["n_b"], case["hd"]
        n_in = 2 * na * hd + 2 * nb * hd + (0 if case["full"] else 2 * nb)
        width = (na if case["full"] else nb) * hd
        total = sum(_matrix_bytes(a, b, case["meta"]) for a, b in ((n_in, h), (h, width), (2 * i, h), (h, i)))
        extra = 4 * case["pos"] * nb * hd if case["full"] else 8 * nb * hd * hd
        return dict(bytes=total + extra + 12 * h, flops=2.0 * (n_in * h + h * width + 3 * i * h))
    if k == "attn_decode":
        n = case["pos"] * case["hd"]
        return dict(bytes=4.0 * n * case["nkv"] + 12 * case["nq"] * case["hd"], flops=4.0 * n * case["nq"])
    if k == "attn_prefill":
        t, p, hd = case["tokens"], case["pos0"], case["hd"]
        return dict(bytes=4.0 * (p + t) * case["nkv"] * hd + 12.0 * t * case["nq"] * hd,
                    flops=4.0 * case["nq"] * hd * (t * p + t * (t + 1) / 2))
    if k == "scan":
        t, lk, lv = case["tokens"], case["lk"], case["lv"]
        return dict(bytes=4.0 * t * 128 * (2 * lk + 2 * lv) + 8.0 * lv * 128 * 128, flops=6.0 * t * lv * 128 * 128)
    c = SESSION
    h, i = c["hidden_size"], c["intermediate_size"]
    width = c["num_attention_heads"] * 128
    in_full = 2 * width + 2 * c["num_key_value_heads"] * 128
    in_lin = 2 * width + 2 * c["linear_num_key_heads"] * 128 + 2 * c["linear_num_value_heads"]
    params = c["num_layers"] * (3 * h * i + h * width) + h * (in_full + 3 * in_lin)
    per = 0.5 + (4.5 if case["asym"] else 2.0) / GROUP
    steps, head = case["new"] + 1, c["vocab_size"] * h
    return dict(bytes=per * (params + head) * steps, flops=2.0 * (params * (case["prompt"] + case["new"]) + head * steps))


def tolerance(case):
    """About four times the error against exact() that the paths show; where a new key
    and value are rounded to fp16 in the cache, a last bit that turns out otherwise
    (2^-10 of the value) in a few of a short cache's values."""
    k = case["kind"]
    if k == "gemv":
        return dict(rel=1e-3 if case["f16"] else 2e-6)
    return dict(lm_head=dict(rel=2e-6, differ=0.0), layer=dict(rel=3e-5, max=2e-3),
                gemm=dict(rel=2e-6), attn_decode=dict(rel=2e-5, max=2e-3), attn_prefill=dict(rel=4e-6), scan=dict(rel=4e-6),
                session=dict(rel=1e-5, differ=0.0))[k]


# ---- the same in 64 bits ------------------------------------------------------------
def _dense(w, rows, cols):
    """The dequantised matrix in 64 bits."""
    packed, scales, zeros, bits = w
    if bits == 4:
        q = torch.stack([packed & 15, packed >> 4], -1)
    else:  # an LSB-first bit stream
        b = (packed[:, None] >> torch.arange(8, device=packed.device, dtype=torch.uint8)) & 1
        q = (b.reshape(-1, bits) << torch.arange(bits, device=packed.device, dtype=torch.uint8)).sum(-1)
    q = q.reshape(rows, cols // GROUP, GROUP).to(F64)
    return ((q - zeros.to(F64).reshape(rows, -1, 1)) * scales.to(F64).reshape(rows, -1, 1)).reshape(rows, cols)


def _product(w, rows, cols, x):
    """x W^T in 64 bits, a slab of rows at a time."""
    packed, scales, zeros, bits = w
    out, step = [], max(8, (1 << 26) // cols // 8 * 8)
    for a in range(0, rows, step):
        n = min(step, rows - a)
        part = (packed[a * cols * bits // 8:(a + n) * cols * bits // 8],
                *(t[a * cols // GROUP:(a + n) * cols // GROUP] for t in (scales, zeros)), bits)
        out.append(x @ _dense(part, n, cols).T)
    return torch.cat(out, -1)


def _norm(x, weight):
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * weight.to(F64)


def _silu_pair(y):
    return torch.nn.functional.silu(y[..., 0::2]) * y[..., 1::2]


def _rotate(x, cs):
    """Rotates the first dims of x [T][heads][hd] by the table rows cs [T][pairs][2]."""
    n = cs.shape[1]
    c, s = cs[:, None, :, 0].to(F64), cs[:, None, :, 1].to(F64)
    a, b = x[..., :n], x[..., n:2 * n]
    return torch.cat([a * c - b * s, b * c + a * s, x[..., 2 * n:]], -1)


def _attend(q, gate, kc, vc, pos0):
    """Gated causal attention of q [T][nq][hd] at pos0 .. over caches [ctx][nkv][hd]."""
    T, nq, hd = q.shape
    ctx, g = pos0 + T, nq // kc.shape[1]
    k, v = (t[:ctx].to(F64).transpose(0, 1).contiguous() for t in (kc, vc))
    late = torch.arange(ctx, device=q.device)[None, :] > pos0 + torch.arange(T, device=q.device)[:, None]
    out = torch.empty_like(q)
    for h in range(nq):
        p = (q[:, h] @ k[h // g].T / math.sqrt(hd)).masked_fill(late, -math.inf).softmax(-1)
        out[:, h] = p @ v[h // g]
    return out * torch.sigmoid(gate)


def _split_heads(proj, nq, nkv, hd, d, cs):
    """q, gate, k, v [T][heads][hd] of a projection row, q and k normed and rotated."""
    T = proj.shape[0]
    qg = proj[:, :2 * nq * hd].reshape(T, nq, 2 * hd)
    k, v = (t.reshape(T, nkv, hd) for t in proj[:, 2 * nq * hd:2 * (nq + nkv) * hd].chunk(2, -1))
    return _rotate(_norm(qg[..., :hd], d["qn"]), cs), qg[..., hd:], _rotate(_norm(k, d["kn"]), cs), v


def _scan(proj, hist, S, lk, lv, d):
    """The gated delta rule over the rows of proj: outputs, state and conv history after."""
    T, cd = proj.shape[0], 128 * (2 * lk + lv)
    x = torch.cat([hist.to(F64).T, proj[:, :cd]])
    y = torch.nn.functional.silu(sum(x[i:i + T] * d["conv"][:, i].to(F64) for i in range(KSIZE)))
    unit = lambda t: t / (t.square().sum(-1, keepdim=True) + 1e-6).sqrt()  # noqa: E731
    q, k = (unit(t.reshape(T, lk, 128)).repeat_interleave(lv // lk, 1) for t in y[:, :256 * lk].chunk(2, -1))
    v = y[:, 256 * lk:].reshape(T, lv, 128)
    beta = torch.sigmoid(proj[:, cd + lv:cd + 2 * lv])
    decay = (-d["a_log"].to(F64).exp() * torch.nn.functional.softplus(proj[:, cd:cd + lv] + d["dt"].to(F64),
                                                                         threshold=100.0)).exp()
    S, out = S.to(F64).clone(), torch.empty_like(v)
    for t in range(T):
        S *= decay[t][:, None, None]
        delta = beta[t][:, None] * (v[t] - torch.einsum("hij,hi->hj", S, k[t]))
        S += k[t][:, :, None] * delta[:, None, :]
        out[t] = torch.einsum("hij,hi->hj", S, q[t]) / math.sqrt(128)
    return out, S, x[-(KSIZE - 1):].T


def _layer(x, full, mats, na, nb, hd, d, cache, pos0, cs):
    """One layer on rows x [T][hidden]; mats: the four products; cache: (K, V) or (history, state)."""
    T = x.shape[0]
    proj = mats[0](_norm(x, d["n1"]))
    if full:
        q, gate, k, v = _split_heads(proj, na, nb, hd, d, cs)
        cache[0][pos0:pos0 + T], cache[1][pos0:pos0 + T] = k.half(), v.half()
        a = _attend(q, gate, cache[0], cache[1], pos0)
    else:
        a, cache[1], cache[0] = _scan(proj, cache[0], cache[1], na, nb, d)
        z = proj[:, -nb * hd:].reshape(T, nb, hd)
        a = _norm(a, d["lin_norm"]) * torch.nn.functional.silu(z)
    x = x + mats[1](a.reshape(T, -1))
    return x + mats[3](_silu_pair(mats[2](_norm(x, d["n2"]))))


def exact(case, seed):
    k = case["kind"]
    if k == "session":
        return _exact_session(case, seed)
    d = _inputs(case, seed)
    if k in ("gemv", "gemm", "lm_head"):
        rows, cols = case["rows"], case["cols"]
        x = d["x"].to(F64)
        y = _product(d["w"], rows, cols, x if case.get("pro") == "none" else _norm(x, d["norm"]))
        if k == "lm_head":
            i = y.argmax(-1)
            return dict(index=i.int(), value=y.amax(-1), row=d["table"][i[0]].to(F64))
        return dict(y=_silu_pair(y) if case["epi"] == "silu" else d["y0"].to(F64) + y)
    if k == "layer":
        h, i, na, nb, hd = case["hidden"], case["inter"], case["n_a"], case["n_b"], case["hd"]
        width, n_in = (na if case["full"] else nb) * hd, len(d["w_in"][1]) * GROUP // h
        mats = [lambda v, w=d[n], a=a, b=b: _product(w, a, b, v)
                for n, a, b in (("w_in", n_in, h), ("w_out", h, width), ("w_gu", 2 * i, h), ("w_down", h, i))]
        parity = case["pos"] & 1
        cache = [d["kc"], d["vc"]] if case["full"] else [d["hist"][parity], d["S"]]
        cs = d["rope"][case["pos"]:] if case["full"] else None
        x = _layer(d["x"].to(F64), case["full"], mats, na, nb, hd, d, cache, case["pos"], cs)
        if case["full"]:
            return dict(x=x, kc=cache[0].to(F64), vc=cache[1].to(F64))
        return dict(x=x, S=cache[1], hist=cache[0])
    if k == "attn_decode":
        q, gate, kn, vn = _split_heads(d["proj"].to(F64), case["nq"], case["nkv"], case["hd"], d, d["rope"][case["pos"]:])
        d["kc"][case["pos"]], d["vc"][case["pos"]] = kn[0].half(), vn[0].half()
        return dict(out=_attend(q, gate, d["kc"], d["vc"], case["pos"]).reshape(-1), kc=d["kc"].to(F64),
                    vc=d["vc"].to(F64))
    if k == "attn_prefill":
        q, gate = (d[n].to(F64).reshape(case["tokens"], case["nq"], case["hd"]) for n in ("q", "gate"))
        return dict(out=_attend(q, gate, d["kc"], d["vc"], case["pos0"]).reshape(case["tokens"], -1))
    out, S, new = _scan(d["proj"].to(F64), d["hist"][0], d["S"], case["lk"], case["lv"], d)
    return dict(out=out.reshape(case["tokens"], -1), S=S, hist=new)


def _exact_session(case, seed):
    where = _write_model(case, seed)
    try:
        return _forward(case, seed, where)
    finally:
        shutil.rmtree(where, ignore_errors=True)


def _forward(case, seed, where):
    c = SESSION

    def vector(name, plus=0.0):
        return torch.from_numpy(np.fromfile(os.path.join(where, name + ".f32"), np.float32)).cuda() + plus

    def matrix(name):
        with open(os.path.join(where, name + ".xq4"), "rb") as f:
            head = f.read(52)
            rows, cols = struct.unpack("<II", head[12:20])
            sizes = struct.unpack("<QQQ", head[28:52])
            packed = torch.from_numpy(np.fromfile(f, np.uint8, sizes[0])).cuda()
            scales, zeros = (torch.from_numpy(np.fromfile(f, np.float32, n)).cuda() for n in sizes[1:])
        return _dense((packed, scales, zeros, 4), rows, cols)

    def layer(i):
        p = "layers_%d_" % i
        full = i % 4 == 3
        d = dict(n1=vector(p + "input_layernorm_weight", 1.0), n2=vector(p + "post_attention_layernorm_weight", 1.0))
        if full:
            names, out = ["self_attn_%s_proj" % n for n in "qkv"], "self_attn_o_proj"
            d.update(qn=vector(p + "self_attn_q_norm_weight", 1.0), kn=vector(p + "self_attn_k_norm_weight", 1.0))
        else:
            names, out = ["linear_attn_in_proj_" + n for n in ("qkv", "a", "b", "z")], "linear_attn_out_proj"
            d.update(lin_norm=vector(p + "linear_attn_norm_weight"), a_log=vector(p + "linear_attn_A_log"),
                     dt=vector(p + "linear_attn_dt_bias"),
                     conv=vector(p + "linear_attn_conv1d_weight").reshape(-1, KSIZE))
        gate_up = torch.stack([matrix(p + "mlp_gate_proj_weight"), matrix(p + "mlp_up_proj_weight")], 1).flatten(0, 1)
        mats = [torch.cat([matrix(p + n + "_weight") for n in names]), matrix(p + out + "_weight"), gate_up,
                matrix(p + "mlp_down_proj_weight")]
        mats = [lambda v, w=w: v @ w.T for w in mats]
        if full:
            cache = [_zeros(case["prompt"] + case["new"], c["num_key_value_heads"], 128, dtype=torch.half) for _ in "kv"]
            return full, mats, c["num_attention_heads"], c["num_key_value_heads"], 128, d, cache
        lk, lv = c["linear_num_key_heads"], c["linear_num_value_heads"]
        return full, mats, lk, lv, 128, d, [_zeros(128 * (2 * lk + lv), KSIZE - 1), _zeros(lv, 128, 128)]

    layers = [layer(i) for i in range(c["num_layers"])]
    head, last = matrix("lm_head_weight"), vector("norm_weight", 1.0)
    raw = np.fromfile(os.path.join(where, "embeddings_bf16.bin"), np.int16).reshape(-1, c["hidden_size"])
    table = torch.from_numpy(raw).cuda().view(torch.bfloat16)
    cs = torch.from_numpy(_rope_table(case["prompt"] + case["new"], 32)).cuda()

    def forward(ids, pos0):
        x = table[torch.as_tensor(ids, device="cuda").long()].to(F64)
        for ly in layers:
            x = _layer(x, *ly, pos0, cs[pos0:pos0 + len(ids)])
        return _norm(x[-1], last)

    h, ids = forward(_prompt(case, seed), 0), []
    for t in range(case["new"]):
        ids.append(int((head @ h).argmax()))
        h = forward(ids[-1:], case["prompt"] + t)
    top = (head @ h).topk(10)
    return dict(tokens=np.array(ids, np.int32), hidden=h, ids=top.indices, logits=top.values)
