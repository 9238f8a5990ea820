"""The work that programs have this library do, as timed cases.

  gemv      one quantised matrix times 1..8 activation rows (qgpu_gemv_batch), on device pointers
  attn      the gated attention of a forward of 1..8 tokens over a KV cache (qgpu_attn_fused)
  gdn       the Gated-DeltaNet conv + recurrence of 1..8 tokens with state snapshots (qgpu_gdn_fused)
  sample    one draw of the sampler over a vocabulary's logits (qgpu_sample)
  generate  a whole request to the model: model_reset, model_spec_begin (the prompt),
            model_spec_run (speculative or plain greedy cycles), as model_generate_spec chains them

The matrices, heads and states have the sizes of the 27B hybrid (qwen_synth_spec_27b) and of its
checkpoint's format mix.  The generate cases run eight of its layers (six Gated-DeltaNet, two
attention) and its MTP layer over a vocabulary of 32768, so that the head weighs against the layers
about as it does in the whole model and a case loads in a second.
"""
import ctypes
import importlib.util
import math
import os
import sys

import numpy as np
import torch

E, FF, VOCAB, NH, NKV, HD, ROPE, NK, NV, HK = 5120, 17408, 248320, 24, 4, 256, 64, 16, 48, 128
CONV, INNER, NSLOT, EPS, THETA = 2 * NK * HK + NV * HK, NV * HK, 9, 1e-6, 1e7
MODEL_VOCAB, MODEL_LAYERS = 32768, 8
TYPES = {"IQ4_XS": 23, "Q4_K": 12, "Q5_K": 13, "Q6_K": 14, "Q8_0": 8}
BLOCK = {23: (256, 136), 12: (256, 144), 13: (256, 176), 14: (256, 210), 8: (32, 34)}
IQ4NL = (-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113)
F32P, U32P, I32P = (ctypes.POINTER(t) for t in (ctypes.c_float, ctypes.c_uint32, ctypes.c_int))


def _pyqwen():
    if "pyqwen" not in sys.modules:
        path = os.path.join(os.getcwd(), "qwen3.8-27b-in-c_amd", "pyqwen.py")
        spec = importlib.util.spec_from_file_location("pyqwen", path)
        sys.modules["pyqwen"] = mod = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(mod)
    return sys.modules["pyqwen"]


# ---------------------------------------------------------------------------- the cases
def listed():
    return [
        # the k or v projection of one decoded token: the smallest call, where launches count
        {"name": "gemv_kv_b1", "kind": "gemv", "type": "IQ4_XS", "ne0": E, "ne1": NKV * HD, "n": 1},
        # the FFN gate or up projection of a verify of three drafts, the benchmark's matrix
        {"name": "gemv_ffn_b4", "kind": "gemv", "type": "IQ4_XS", "ne0": E, "ne1": FF, "n": 4},
        # attn_qkv of the checkpoint's format mix for a ragged batch of seven
        {"name": "gemv_qkv_q5k_b7", "kind": "gemv", "type": "Q5_K", "ne0": E, "ne1": CONV, "n": 7},
        # the lm_head of the format mix for one decoded token: the largest matrix
        {"name": "gemv_head_q6k_b1", "kind": "gemv", "type": "Q6_K", "ne0": E, "ne1": VOCAB, "n": 1},
        # attention of a verify of three drafts in an ordinary chat context
        {"name": "attn_b4_800", "kind": "attn", "B": 4, "pos": 800, "n_ctx": 1024},
        # attention of the deepest verify (seven drafts) at the end of a long context
        {"name": "attn_b8_8184", "kind": "attn", "B": 8, "pos": 8184, "n_ctx": 8192},
        # one Gated-DeltaNet layer's recurrence in a verify of three drafts
        {"name": "gdn_b4", "kind": "gdn", "B": 4, "nk": NK, "nv": NV, "cur": 5},
        # a sampled token with the command line's usual settings
        {"name": "sample_k40", "kind": "sample", "vocab": VOCAB, "temp": 0.8, "top_p": 0.9, "top_k": 40,
         "penalty": 1.1, "window": 64},
        # the benchmark's prompt, then one speculative cycle: time to first tokens
        {"name": "prompt_512", "kind": "generate", "mix": 0, "n_prompt": 512, "k": 3, "cycles": 1},
        # a long prompt of odd length on the checkpoint's format mix: a document
        {"name": "prompt_1999_mix", "kind": "generate", "mix": 1, "n_prompt": 1999, "k": 3, "cycles": 1},
        # a short question and 48 speculative cycles: decode dominates
        {"name": "chat_spec_k3", "kind": "generate", "mix": 0, "n_prompt": 33, "k": 3, "cycles": 48},
        # a short question and 48 plain greedy tokens (no drafts): batch-1 decode
        {"name": "chat_greedy", "kind": "generate", "mix": 0, "n_prompt": 17, "k": 0, "cycles": 48},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "gemv", "attn", "gdn", "sample", "generate", "generate", "generate"])
    if kind == "gemv":
        t = rng.choice(["IQ4_XS", "IQ4_XS", "IQ4_XS", "Q4_K", "Q5_K", "Q6_K", "Q8_0"])
        ne0 = 256 * rng.choice([4, 8, 20, 20, 20, 24, 40, 68, rng.randint(1, 68)])
        ne1 = _log_int(rng, 48, min(VOCAB, int(1.2e9 / ne0)))
        return {"kind": kind, "type": t, "ne0": ne0, "ne1": ne1, "n": rng.randint(1, 8)}
    if kind == "attn":
        n_ctx = rng.choice([512, 1024, 2048, 4096, 8192])
        b = rng.randint(1, 8)
        return {"kind": kind, "B": b, "pos": min(n_ctx - b, _log_int(rng, 1, n_ctx)), "n_ctx": n_ctx}
    if kind == "gdn":
        nk, nv = rng.choice([(NK, NV), (NK, NV), (16, 32), (8, 24), (2, 4)])
        return {"kind": kind, "B": rng.randint(1, 8), "nk": nk, "nv": nv, "cur": rng.randrange(NSLOT)}
    if kind == "sample":
        return {"kind": kind, "vocab": rng.choice([VOCAB, _log_int(rng, 1000, VOCAB)]),
                "temp": rng.choice([0.0, 0.6, 0.8, 1.0]), "top_p": rng.choice([0.9, 0.95, 1.0]),
                "top_k": rng.choice([20, 40, 100, 256]), "penalty": rng.choice([1.0, 1.1]),
                "window": rng.randint(0, 64)}
    n = _log_int(rng, 1, 1900)
    return {"kind": kind, "mix": rng.randint(0, 1), "n_prompt": n, "k": rng.choice([0, 1, 2, 3, 3, 5, 7]),
            "cycles": 1 if n > 400 else rng.choice([1, 8, 24])}


# ---------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32)


def _activations(g, rows, n):
    """rows as a norm leaves them: normal, channels of unequal strength and a few strong ones"""
    scale = torch.exp(0.4 * _normal(g, n))
    scale[torch.randint(0, n, (max(1, n // 512),), generator=g, device="cuda")] *= 8.0
    return (_normal(g, rows, n) * scale).contiguous()


def _weight_bytes(g, t, ne0, ne1):
    """rows of quantised blocks, random codes and scales, of unit output for unit input"""
    be, bs = BLOCK[t]
    b = torch.randint(0, 256, (ne1, ne0 // be, bs), generator=g, device="cuda", dtype=torch.uint8)
    unit = {23: 67.44 * 18.48, 12: 36.5 * 8.8, 13: 36.5 * 18.0, 14: 73.9 * 18.5, 8: 73.9}[t] * math.sqrt(ne0)

    def half(at, sigma):
        d = (_normal(g, ne1, ne0 // be).abs() * sigma).to(torch.float16)
        b[:, :, at:at + 2] = d.contiguous().view(torch.uint8).view(ne1, ne0 // be, 2)
    half({14: 208}.get(t, 0), 1.0 / unit)
    if t in (12, 13):
        half(2, 4.0 / unit)
    return b


def _dequant(t, b):
    """[rows, blocks, bytes] -> [rows, columns] in 64 bits (the published ggml block formats)"""
    rows, nb = b.shape[0], b.shape[1]

    def half(at):
        return b[:, :, at:at + 2].contiguous().view(torch.float16).double()          # [rows, nb, 1]
    i = b.to(torch.int32)
    if t == 8:
        w = half(0) * b[:, :, 2:34].contiguous().view(torch.int8).double()
    elif t == 23:
        ib = torch.arange(8, device=b.device)
        sh = i[:, :, 2:3] | (i[:, :, 3:4] << 8)
        lo = (i[:, :, 4:8].repeat_interleave(2, 2) >> (4 * (ib % 2))) & 15
        dl = half(0) * ((lo | (((sh >> (2 * ib)) & 3) << 4)) - 32).double()
        q = i[:, :, 8:136].view(rows, nb, 8, 16)
        code = torch.tensor(IQ4NL, device=b.device, dtype=torch.float64)
        w = torch.cat([code[(q & 15).long()], code[(q >> 4).long()]], 3) * dl[..., None]
    elif t in (12, 13):
        s = i[:, :, 4:16]
        sc = torch.cat([s[:, :, 0:4] & 63, (s[:, :, 8:12] & 15) | ((s[:, :, 0:4] >> 6) << 4)], 2).double()
        mn = torch.cat([s[:, :, 4:8] & 63, (s[:, :, 8:12] >> 4) | ((s[:, :, 4:8] >> 6) << 4)], 2).double()
        qs = i[:, :, (16 if t == 12 else 48):].view(rows, nb, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 3).view(rows, nb, 8, 32)
        if t == 13:
            sh = torch.arange(8, device=b.device)[:, None]
            q = q + (((i[:, :, None, 16:48] >> sh) & 1) << 4)
        w = (half(0) * sc)[..., None] * q.double() - (half(2) * mn)[..., None]
    else:
        ql, qh = i[:, :, :128].view(rows, nb, 2, 2, 32), i[:, :, 128:192].view(rows, nb, 2, 1, 32)
        two = torch.cat([(qh >> (2 * j)) & 3 for j in range(4)], 3)
        q = (torch.cat([ql & 15, ql >> 4], 3) | (two << 4)) - 32                      # [rows, nb, 2, 4, 32]
        sc = b[:, :, 192:208].contiguous().view(torch.int8).double().view(rows, nb, 2, 4, 2)
        w = half(208)[..., None, None] * q.double() * sc.repeat_interleave(16, 4)
    return w.reshape(rows, -1)


def _p(t, typ=F32P):
    return ctypes.cast(ctypes.c_void_p(t.data_ptr()), typ)


def _rope_tables(n):
    """the model's tables: float angles and their float cosines and sines"""
    i = np.arange(ROPE // 2, dtype=np.float32)
    freq = np.power(np.float32(THETA), (np.float32(-2.0) * i / np.float32(ROPE)).astype(np.float32)).astype(np.float32)
    ang = (np.arange(n, dtype=np.float32)[:, None] * freq[None]).astype(np.float32)
    return np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)


def _gemv_inputs(case, seed):
    g = _gen(seed)
    t = TYPES[case["type"]]
    return t, _weight_bytes(g, t, case["ne0"], case["ne1"]), _activations(g, case["n"], case["ne0"])


def _attn_inputs(case, seed):
    g, B, n_ctx = _gen(seed), case["B"], case["n_ctx"]
    s = {"q": 2.0 * _normal(g, B, NH * 2 * HD), "k": _normal(g, B, NKV * HD), "v": _normal(g, B, NKV * HD),
         "qw": 1 + 0.1 * _normal(g, HD), "kw": 1 + 0.1 * _normal(g, HD)}
    s["kc"] = torch.zeros(n_ctx, NKV * HD, device="cuda")
    s["vc"] = torch.zeros(n_ctx, NKV * HD, device="cuda")
    s["kc"][:case["pos"]] = _normal(g, case["pos"], NKV * HD)
    s["vc"][:case["pos"]] = _normal(g, case["pos"], NKV * HD)
    s["cos"], s["sin"] = (torch.from_numpy(a).cuda() for a in _rope_tables(n_ctx))
    return s


def _gdn_inputs(case, seed):
    g, B, nv, at = _gen(seed), case["B"], case["nv"], case["cur"]
    chan = (2 * case["nk"] + nv) * HK
    s = {"x": _normal(g, B, chan), "beta": _normal(g, B, nv), "alpha": _normal(g, B, nv),
         "cw": 0.5 * _normal(g, chan, 4), "dtb": 0.5 * _normal(g, nv), "a": -(0.3 + 0.7 * _normal(g, nv).abs()),
         "conv": torch.zeros(NSLOT, chan, 4, device="cuda"), "ssm": torch.zeros(NSLOT, nv, HK, HK, device="cuda")}
    s["conv"][at] = 0.5 * _normal(g, chan, 4)
    s["ssm"][at] = 0.05 * _normal(g, nv, HK, HK)
    return s


def _sample_inputs(case, seed):
    g, V = _gen(seed), case["vocab"]
    logits = 2.5 * _normal(g, V)
    return logits, torch.randint(0, V, (max(1, case["window"]),), generator=g, device="cuda").to(torch.int32)


def _spec(case, seed):
    host = _pyqwen().host_lib()
    s = (host.spec_27b_mix if case["mix"] else host.spec_27b)(1000 + int(seed))
    s.n_layer, s.vocab = MODEL_LAYERS, MODEL_VOCAB
    return s


def _prompt(case, seed):
    return np.random.RandomState(int(seed) % 2**31).randint(0, MODEL_VOCAB, case["n_prompt"]).astype(np.uint32)


def prepare(case, seed):
    py, kind = _pyqwen(), case["kind"]
    gpu = py.gpu_lib()
    s = {"kind": kind, "L": gpu.L, "ok": gpu.ok}
    if kind == "gemv":
        t, b, x = _gemv_inputs(case, seed)
        torch.cuda.synchronize()
        h = ctypes.c_void_p()
        gpu.ok(gpu.L.qgpu_tensor_from_device(ctypes.c_void_p(b.data_ptr()), t, case["ne0"], case["ne1"],
                                             ctypes.byref(h)))
        gpu.sync()
        s["W"], s["x"] = py.Tensor(gpu, h, t, case["ne0"], case["ne1"]), x
        s["out"] = torch.empty(case["n"], case["ne1"], device="cuda")
        s["args"] = (h, _p(x), case["ne0"], case["n"], _p(s["out"]), case["ne1"], 0)
    elif kind == "attn":
        s.update(_attn_inputs(case, seed))
        s["out"] = torch.empty(case["B"], NH * HD, device="cuda")
        s["pos"] = torch.tensor([case["pos"]], dtype=torch.int32, device="cuda")
        gpu.ok(gpu.L.qgpu_attn_reserve(case["n_ctx"], NKV))
        s["args"] = (_p(s["q"]), NH * 2 * HD, _p(s["k"]), _p(s["v"]), NKV * HD, _p(s["qw"]), _p(s["kw"]),
                     _p(s["kc"]), _p(s["vc"]), _p(s["cos"]), _p(s["sin"]), ROPE, _p(s["pos"], I32P), case["n_ctx"],
                     case["B"], NH, NKV, HD, EPS, _p(s["out"]), NH * HD)
    elif kind == "gdn":
        s.update(_gdn_inputs(case, seed))
        nk, nv, chan = case["nk"], case["nv"], s["x"].shape[1]
        s["out"] = torch.empty(case["B"], nv * HK, device="cuda")
        s["at"] = torch.tensor([case["cur"]], dtype=torch.int32, device="cuda")
        s["args"] = (_p(s["x"]), chan, case["B"], chan, _p(s["cw"]), _p(s["conv"]), chan * 4, _p(s["beta"]),
                     _p(s["alpha"]), nv, _p(s["dtb"]), _p(s["a"]), _p(s["ssm"]), nv * HK * HK, NSLOT,
                     _p(s["at"], I32P), nk, nv, HK, EPS, _p(s["out"]), nv * HK)
    elif kind == "sample":
        s["fresh"], s["window"] = _sample_inputs(case, seed)
        V = case["vocab"]
        s["logits"] = torch.empty((V + 3) // 4 * 4, device="cuda")       # room for whole 16-byte copies
        s["source"] = torch.zeros_like(s["logits"])
        s["source"][:V] = s["fresh"]
        s["rng"] = torch.tensor([0x9E3779B9 + int(seed)], dtype=torch.int64, device="cuda")
        s["token"] = torch.zeros(1, dtype=torch.int32, device="cuda")
        s["shown"] = s["logits"][:V]
        s["copy"] = (ctypes.c_void_p(s["logits"].data_ptr()), ctypes.c_void_p(s["source"].data_ptr()),
                     s["logits"].numel() * 4)
        s["args"] = (_p(s["logits"]), V, _p(s["window"], U32P), case["window"], case["temp"], case["top_p"],
                     case["top_k"], case["penalty"], 64, _p(s["rng"], ctypes.POINTER(ctypes.c_uint64)),
                     _p(s["token"], U32P))
    else:
        n_ctx = -(-(case["n_prompt"] + 8 * case["cycles"] + 16) // 256) * 256
        s["m"] = py.Model(spec=_spec(case, seed), n_ctx=n_ctx)
        s["case"], s["prompt"] = dict(case), _prompt(case, seed)
    return s


# ---------------------------------------------------------------------------- one pass
def run(state):
    L, ok, kind = state["L"], state["ok"], state["kind"]
    if kind == "gemv":
        ok(L.qgpu_gemv_batch(*state["args"]))
        return state["out"]
    if kind == "attn":
        ok(L.qgpu_attn_fused(*state["args"]))
        return {"out": state["out"], "kc": state["kc"], "vc": state["vc"]}
    if kind == "gdn":
        ok(L.qgpu_gdn_fused(*state["args"]))
        return {"out": state["out"], "conv": state["conv"], "ssm": state["ssm"]}
    if kind == "sample":
        ok(L.qgpu_copy(*state["copy"]))                    # the logits of this token
        ok(L.qgpu_sample(*state["args"]))
        return {"logits": state["shown"], "token": state["token"], "rng": state["rng"]}
    m, c = state["m"], state["case"]
    m.reset()
    m.spec_begin(state["prompt"], c["k"])
    first = m.field("logits", m.V)
    tokens, depth, _ = m.spec_run(c["k"], c["cycles"])
    rows = c["k"] + 1
    return {"logits": first, "tokens": tokens.astype(np.int64), "depth": depth.astype(np.int64),
            "logits_b": m.field("logits_b", rows * m.V), "h": m.field("h_save", rows * m.E),
            "mtp_h": m.field("mtp_h", m.E)}


# ---------------------------------------------------------------------------- what a pass needs
def _layer_weights():
    ffn = 3 * E * FF
    gdn = E * (CONV + INNER + 2 * NV) + INNER * E + ffn
    att = E * (2 * NH * HD + 2 * NKV * HD) + NH * HD * E + ffn
    return gdn, att


def work(case):
    kind = case["kind"]
    if kind == "gemv":
        be, bs = BLOCK[TYPES[case["type"]]]
        n, a, b = case["n"], case["ne0"], case["ne1"]
        return {"bytes": a // be * bs * b + 4 * n * (a + b), "flops": 2.0 * n * a * b}
    if kind == "attn":
        B, seen = case["B"], case["pos"] + case["B"]
        return {"bytes": 4 * (2 * seen * NKV * HD + B * (2 * NH * HD + 4 * NKV * HD + NH * HD)),
                "flops": 4.0 * B * NH * HD * seen}
    if kind == "gdn":
        B, nv, chan = case["B"], case["nv"], (2 * case["nk"] + case["nv"]) * HK
        return {"bytes": 4 * ((1 + B) * (nv * HK * HK + 4 * chan) + B * (chan + nv * HK)),
                "flops": 8.0 * B * nv * HK * HK}
    if kind == "sample":
        return {"bytes": 12 * case["vocab"], "flops": 0}
    n, k, c = case["n_prompt"], case["k"], case["cycles"]
    gdn, att = _layer_weights()
    na = MODEL_LAYERS // 4
    body = (MODEL_LAYERS - na) * gdn + na * att
    head, mtp = E * MODEL_VOCAB, 2 * E * E + att
    per = 136.0 / 256                                         # bytes of a weight (IQ4_XS; the mix is a little more)
    drafts = (k * (mtp + head) + mtp) if k else 0
    state = (MODEL_LAYERS - na) * NV * HK * HK * 4
    kv = lambda p: (na + (1 if k else 0)) * p * NKV * HD * 8  # noqa: E731
    return {"bytes": per * (body + head + (mtp if k else 0)) + kv(n) + 2 * state
            + c * (per * (body + head + drafts) + kv(n) + 2 * state),
            "flops": 2.0 * (n * (body + (mtp if k else 0)) + head) + 2.0 * na * n * n * NH * HD
            + 2.0 * c * ((k + 1) * (body + head) + drafts)}


def tolerance(case):
    # every path keeps 32-bit activations, states and sums; the figures are about four times what the
    # paths differ by from their 64-bit values (gemv 5-7e-7, attn 3.2-3.7e-6, gdn 1.4e-7, generate 2-6e-6)
    return {"gemv": {"rel": 2.6e-6}, "attn": {"rel": 1.5e-5}, "gdn": {"rel": 6e-7}, "sample": {"rel": 1e-7},
            "generate": {"rel": 2.5e-5}}[case["kind"]]


# ---------------------------------------------------------------------------- the same in 64 bits
def _matmul(t, b, x):
    """x [n, ne0] times the transposed matrix, a band of rows at a time"""
    step = max(1, int(2e8) // (b.shape[1] * BLOCK[t][0]))
    return torch.cat([x @ _dequant(t, b[r:r + step]).T for r in range(0, b.shape[0], step)], 1)


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _rotate(x, cos, sin):
    """x [tokens, heads, HD], the first ROPE channels turned by their position's angles"""
    h = ROPE // 2
    a, b, c, s = x[..., :h], x[..., h:ROPE], cos[:, None], sin[:, None]
    return torch.cat([a * c - b * s, a * s + b * c, x[..., ROPE:]], -1)


def _attention(q, k, v, qw, kw, kc, vc, cos, sin, pos):
    """gated attention of B rows at pos; kc, vc [pos, NKV, HD] of earlier rows; also the new caches"""
    B = q.shape[0]
    q = q.view(B, NH, 2, HD)
    at = slice(pos, pos + B)
    kc = torch.cat([kc, _rotate(_rms(k.view(B, NKV, HD), kw), cos[at], sin[at])])
    vc = torch.cat([vc, v.view(B, NKV, HD)])
    qq = _rotate(_rms(q[:, :, 0], qw), cos[at], sin[at]).view(B, NKV, NH // NKV, HD)
    out = []
    late = torch.arange(pos + B, device=q.device)[None] > (pos + torch.arange(B, device=q.device))[:, None]
    for h in range(NKV):
        s = torch.einsum("bgd,td->gbt", qq[:, h], kc[:, h]) / math.sqrt(HD)
        p = torch.softmax(s.masked_fill(late[None], -math.inf), -1)
        out.append(torch.einsum("gbt,td->bgd", p, vc[:, h]))
    out = torch.stack(out, 1).reshape(B, NH, HD) * torch.sigmoid(q[:, :, 1])
    return out.reshape(B, NH * HD), kc, vc


def _recurrence(x, beta, alpha, cw, dtb, a, conv, ssm, keep):
    """conv1d, SiLU, L2 norms and the delta rule over the rows of x; states after every row if keep"""
    B, nv = beta.shape
    nk = (x.shape[1] // HK - nv) // 2
    taps = torch.cat([conv[:, 1:], x.T], 1)                   # [channels, 3 + B]
    y = sum(taps[:, j:j + B] * cw[:, j:j + 1] for j in range(4)).T
    y = y * torch.sigmoid(y)

    def unit(z):
        return z / torch.clamp(z.norm(dim=-1, keepdim=True), min=EPS)
    q = unit(y[:, :nk * HK].reshape(B, nk, HK)).repeat(1, nv // nk, 1) / math.sqrt(HK)
    k = unit(y[:, nk * HK:2 * nk * HK].reshape(B, nk, HK)).repeat(1, nv // nk, 1)
    v = y[:, 2 * nk * HK:].reshape(B, nv, HK)
    bt, dec = torch.sigmoid(beta), torch.exp(a * torch.nn.functional.softplus(alpha + dtb, threshold=30.0))
    out, convs, states = [], [], []
    S = ssm
    for b in range(B):
        S = dec[b][:, None, None] * S
        d = (v[b] - (S * k[b][:, None]).sum(-1)) * bt[b][:, None]
        S = S + d[:, :, None] * k[b][:, None]
        out.append((S * q[b][:, None]).sum(-1).reshape(-1))
        if keep:
            states.append(S)
            convs.append(torch.cat([conv, x.T], 1)[:, b + 1:b + 5])
    return torch.stack(out), (convs if keep else torch.cat([conv, x.T], 1)[:, -4:]), (states if keep else S)


class _Model64:
    """the hybrid model in 64 bits: forwards of any number of rows, states and caches kept"""

    def __init__(self, case, seed, n_ctx):
        self.host, self.spec = _pyqwen().host_lib(), _spec(case, seed)
        self.at = {t.name.decode(): (i, t) for i, t in enumerate(self.host.tensors(self.spec))}
        self.cos, self.sin = (torch.from_numpy(a).cuda().double() for a in _rope_tables(n_ctx))
        self.conv = {i: torch.zeros(CONV, 4, dtype=torch.float64, device="cuda") for i in range(MODEL_LAYERS)}
        self.ssm = {i: torch.zeros(NV, HK, HK, dtype=torch.float64, device="cuda") for i in range(MODEL_LAYERS)}
        self.kv = {i: 2 * (torch.zeros(0, NKV, HD, dtype=torch.float64, device="cuda"),)
                   for i in range(MODEL_LAYERS + 1)}
        self.held = {}

    def raw(self, name):
        if name not in self.held:
            i, t = self.at[name]
            b = torch.from_numpy(self.host.fill(self.spec, i, t.nbytes)).cuda()
            if t.type == 0:
                b = b.view(torch.float32).double()
                self.held[name] = b.view(t.ne[1], t.ne[0]) if t.n_dims == 2 else b
            else:
                be, bs = BLOCK[t.type]
                self.held[name] = (t.type, b.view(t.ne[1], t.ne[0] // be, bs))
        return self.held[name]

    def mul(self, name, x):
        return _matmul(*self.raw(name), x)

    def embed(self, tokens):
        t, b = self.raw("token_embd.weight")
        return _dequant(t, b[torch.from_numpy(np.asarray(tokens, np.int64)).cuda()])

    def ffn(self, p, x):
        z = _rms(x, self.raw(p + "post_attention_norm.weight"))
        g = self.mul(p + "ffn_gate.weight", z)
        return x + self.mul(p + "ffn_down.weight", g * torch.sigmoid(g) * self.mul(p + "ffn_up.weight", z))

    def attn(self, i, x, pos):
        p = "blk.%d." % i
        z = _rms(x, self.raw(p + "attn_norm.weight"))
        kc, vc = (c[:pos] for c in self.kv[i])
        o, kc, vc = _attention(*(self.mul(p + "attn_%s.weight" % n, z) for n in "qkv"),
                               self.raw(p + "attn_q_norm.weight"), self.raw(p + "attn_k_norm.weight"), kc, vc,
                               self.cos, self.sin, pos)
        self.kv[i] = (kc, vc)
        return self.ffn(p, x + self.mul(p + "attn_output.weight", o))

    def gdn(self, i, x):
        p = "blk.%d." % i
        z = _rms(x, self.raw(p + "attn_norm.weight"))
        gate = self.mul(p + "attn_gate.weight", z).view(-1, NV, HK)
        o, self.conv[i], self.ssm[i] = _recurrence(
            self.mul(p + "attn_qkv.weight", z), self.mul(p + "ssm_beta.weight", z), self.mul(p + "ssm_alpha.weight", z),
            self.raw(p + "ssm_conv1d.weight"), self.raw(p + "ssm_dt.bias"), self.raw(p + "ssm_a"), self.conv[i],
            self.ssm[i], False)
        o = _rms(o.view(-1, NV, HK), self.raw(p + "ssm_norm.weight")) * gate * torch.sigmoid(gate)
        return self.ffn(p, x + self.mul(p + "ssm_out.weight", o.reshape(-1, INNER)))

    def forward(self, tokens, pos):
        x = self.embed(tokens)
        for i in range(MODEL_LAYERS):
            x = self.attn(i, x, pos) if i % 4 == 3 else self.gdn(i, x)
        return x

    def head(self, x, norm="output_norm.weight"):
        return self.mul("output.weight", _rms(x, self.raw(norm)))

    def mtp(self, tokens, h, pos):
        p = "blk.%d.nextn." % MODEL_LAYERS
        z = torch.cat([_rms(self.embed(tokens), self.raw(p + "enorm.weight")), _rms(h, self.raw(p + "hnorm.weight"))], 1)
        return self.attn(MODEL_LAYERS, self.mul(p + "eh_proj.weight", z), pos)


def exact(case, seed):
    kind = case["kind"]
    if kind == "gemv":
        t, b, x = _gemv_inputs(case, seed)
        return _matmul(t, b, x.double())
    if kind == "attn":
        s = {k: v.double() for k, v in _attn_inputs(case, seed).items()}
        p, B = case["pos"], case["B"]
        out, kc, vc = _attention(s["q"], s["k"], s["v"], s["qw"], s["kw"], s["kc"][:p].view(-1, NKV, HD),
                                 s["vc"][:p].view(-1, NKV, HD), s["cos"], s["sin"], p)
        s["kc"][:p + B], s["vc"][:p + B] = kc.reshape(p + B, -1), vc.reshape(p + B, -1)
        return {"out": out, "kc": s["kc"], "vc": s["vc"]}
    if kind == "gdn":
        s = {k: v.double() if isinstance(v, torch.Tensor) else v for k, v in _gdn_inputs(case, seed).items()}
        c = case["cur"]
        out, convs, states = _recurrence(s["x"], s["beta"], s["alpha"], s["cw"], s["dtb"], s["a"], s["conv"][c],
                                         s["ssm"][c], True)
        for b in range(case["B"]):
            s["conv"][(c + 1 + b) % NSLOT], s["ssm"][(c + 1 + b) % NSLOT] = convs[b], states[b]
        return {"out": out, "conv": s["conv"], "ssm": s["ssm"]}
    if kind == "sample":
        logits, window = _sample_inputs(case, seed)
        x = logits.double().cpu()
        for t in window.tolist()[:case["window"]]:
            x[t] = x[t] / np.float32(case["penalty"]) if x[t] > 0 else x[t] * np.float32(case["penalty"])
        return {"logits": x, "token": None, "rng": None}
    k, prompt = case["k"], _prompt(case, seed)
    n = len(prompt)
    m = _Model64(case, seed, n + 64)
    h = m.forward(prompt, 0)
    if k:
        state = m.mtp(prompt, h, 0)[-1:]
    first = m.head(h[-1:])[0]
    got = {"logits": first, "tokens": None, "depth": None, "logits_b": None, "h": None, "mtp_h": None}
    if case["cycles"] == 1 and k:
        cand = [int(first.argmax())]
        for d in range(1, k + 1):                               # drafts, each from the last one's state
            state = m.mtp(cand[-1:], state, n - 1 + d)
            cand.append(int(m.head(state, "blk.%d.nextn.shared_head_norm.weight" % MODEL_LAYERS)[0].argmax()))
        h = m.forward(cand, n)
        rows = m.head(h)
        nxt = rows.argmax(1).tolist()
        j = next((i for i in range(k) if nxt[i] != cand[i + 1]), k)
        got.update(logits_b=rows.reshape(-1), h=h.reshape(-1), mtp_h=m.mtp([cand[j]], h[j:j + 1], n + j)[0])
    return got
