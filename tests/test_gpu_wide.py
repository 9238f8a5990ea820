"""The prompt path: products, attention and GDN recurrence over many tokens at once, and whole
prompts through it, against FP64 or the 8-token path."""
import contextlib
import ctypes
import os
import tempfile

import numpy as np
import pytest

import oracle_lib as O
from gpu_util import gpu, rel_err  # noqa: F401
from qwen_pkg import host_lib, pyqwen
from test_gpu_model import ATT_DIMS, _attn_inputs, attn_fp64

pytestmark = pytest.mark.gpu

FORMATS = {"IQ4_XS": 23, "Q4_K": 12, "Q5_K": 13, "Q6_K": 14, "Q8_0": 8}


def norm_err(got, ref):
    return float(np.linalg.norm(got - ref) / np.linalg.norm(ref))


@contextlib.contextmanager
def workspace(gpu, rows, max_k, n_ctx=0, n_kv=0, n_k=0, n_v=0):
    w = ctypes.c_void_p()
    gpu.ok(gpu.L.qgpu_wide_create(rows, max_k, n_ctx, n_kv, n_k, n_v, ctypes.byref(w)))
    try:
        yield w
    finally:
        gpu.ok(gpu.L.qgpu_wide_free(w))


def gemm(gpu, w, Ts, outs, n, flags=0):
    m = len(Ts)
    gpu.ok(gpu.L.qgpu_wide_gemm(w, (ctypes.c_void_p * m)(*[T.h for T in Ts]), m, n,
                                (pyqwen.F32P * m)(*[o.f32() for o in outs]),
                                (ctypes.c_uint64 * m)(*[T.ne1 for T in Ts]), flags))


def copy_act(xb, ld):
    return pyqwen.Act(kind=pyqwen.ACT_COPY, x=xb.f32(), ldx=ld)


# activations keep 2^-22 of each value and the sums take one fp32 rounding per 32 columns (2^-24 of the
# running sum, of random sign): under 2^-22 + 2^-24 sqrt(ne0 / 32) in the 2-norm, 1e-6 with room
WIDE_TOL = 1e-6


@pytest.mark.parametrize("fmt", list(FORMATS))
@pytest.mark.parametrize("ne0,ne1,n", [(256, 16, 1), (256, 48, 17), (512, 300, 33), (1280, 528, 65), (768, 1040, 129),
                                       (6144, 272, 300)])
def test_wide_gemm_vs_fp64(gpu, fmt, ne0, ne1, n):
    """token counts around the 32-, 64- and 128-token tiles, row counts off the 16- and 256-row tiles, runs that
    share tiles between blocks; then accumulation on top of the result"""
    t = FORMATS[fmt]
    W = host_lib().synth_matrix(t, ne0, ne1, 41, 500 + t, 0.02)
    x = host_lib().synth_normal(n * ne0, 42, n).reshape(n, ne0) * np.exp2(np.arange(n) % 40 - 20)[:, None].astype(np.float32)
    ref = x.astype(np.float64) @ O.dequant_rows(t, W, ne0, ne1).reshape(ne1, ne0).astype(np.float64).T
    T, xb, ob = gpu.tensor(W, t, ne0, ne1), gpu.put(x), gpu.put(np.full((n + 1) * ne1, 3.0, np.float32))
    with workspace(gpu, n, ne0) as w:
        a = copy_act(xb, ne0)
        gpu.ok(gpu.L.qgpu_wide_prepare(w, ctypes.byref(a), n, ne0, 1))
        gemm(gpu, w, [T], [ob], n)
        got = ob.download(np.float32).reshape(n + 1, ne1)
        assert (got[n] == 3.0).all()                                  # rows past the call
        for r in range(n):
            assert norm_err(got[r].astype(np.float64), ref[r]) < WIDE_TOL, (fmt, r)
        gemm(gpu, w, [T], [ob], n, flags=1)
        twice = ob.download(np.float32).reshape(n + 1, ne1)[:n]
        assert np.array_equal(twice, got[:n] + got[:n])
    T.close()


def test_wide_gemm_groups_formats(gpu):
    """matrices of several formats and row counts on one prepared input"""
    ne0, n = 512, 70
    host = host_lib()
    x = host.synth_normal(n * ne0, 7, 7).reshape(n, ne0)
    mats = [(23, 300), (13, 512), (23, 48), (8, 16), (23, 257)]
    Ws = [host.synth_matrix(t, ne0, r, 9, i, 0.02) for i, (t, r) in enumerate(mats)]
    Ts = [gpu.tensor(W, t, ne0, r) for W, (t, r) in zip(Ws, mats)]
    xb, outs = gpu.put(x), [gpu.buf(n * r * 4) for _, r in mats]
    with workspace(gpu, 128, ne0) as w:
        a = copy_act(xb, ne0)
        gpu.ok(gpu.L.qgpu_wide_prepare(w, ctypes.byref(a), n, ne0, 1))
        gemm(gpu, w, Ts, outs, n)
        for W, (t, r), o in zip(Ws, mats, outs):
            ref = x.astype(np.float64) @ O.dequant_rows(t, W, ne0, r).reshape(r, ne0).astype(np.float64).T
            assert norm_err(o.download(np.float32).reshape(n, r), ref) < WIDE_TOL
    for T in Ts:
        T.close()


@pytest.mark.parametrize("t", [23, 13, 8])
@pytest.mark.parametrize("ne0,ne1,n", [(256, 16, 3), (512, 400, 40), (2560, 1168, 200)])
def test_wide_gemm_silu(gpu, t, ne0, ne1, n):
    """silu(gate x) * (up x) from the product, rows off the 128-row halves of its blocks"""
    host = host_lib()
    x = host.synth_normal(n * ne0, 8, 8).reshape(n, ne0)
    Ws = [host.synth_matrix(t, ne0, ne1, 12, i, 0.02) for i in range(2)]
    g, u = (x.astype(np.float64) @ O.dequant_rows(t, W, ne0, ne1).reshape(ne1, ne0).astype(np.float64).T for W in Ws)
    Ts = [gpu.tensor(W, t, ne0, ne1) for W in Ws]
    xb, ob = gpu.put(x), gpu.put(np.full((n + 1) * ne1, 3.0, np.float32))
    with workspace(gpu, n, ne0) as w:
        a = copy_act(xb, ne0)
        gpu.ok(gpu.L.qgpu_wide_prepare(w, ctypes.byref(a), n, ne0, 1))
        for _ in range(2):
            gpu.ok(gpu.L.qgpu_wide_gemm_silu(w, Ts[0].h, Ts[1].h, n, ob.f32(), ne1))
        got = ob.download(np.float32).reshape(n + 1, ne1)
        F = gpu.tensor(host.synth_matrix(14, ne0, ne1, 1, 1, 0.02), 14, ne0, ne1)
        assert gpu.L.qgpu_wide_gemm_silu(w, Ts[0].h, F.h, n, ob.f32(), ne1) == -2
        F.close()
    assert (got[n] == 3.0).all()
    assert norm_err(got[:n], g * 0.5 * (1 + np.tanh(g / 2)) * u) < 2e-6        # WIDE_TOL in each factor
    for T in Ts:
        T.close()


@pytest.mark.parametrize("ne0", [256, 6144, 6400, 17408, 24576, 24832])
@pytest.mark.parametrize("kind", ["rmsnorm", "cat", "silu", "gated"])
def test_wide_prepare_kinds(gpu, kind, ne0):
    """each activation transform, at the column counts where the launch shape changes"""
    n, ne1, eps = 19, 64, 1e-6
    host = host_lib()
    x, y = (host.synth_normal(n * ne0, 3, i).reshape(n, ne0) for i in (1, 2))
    wt, w2 = host.synth_normal(ne0, 3, 3), host.synth_normal(ne0, 3, 4)
    X, Y, WT = x.astype(np.float64), y.astype(np.float64), wt.astype(np.float64)
    xb, yb, wb, w2b = gpu.put(x), gpu.put(y), gpu.put(wt), gpu.put(w2)
    a = pyqwen.Act(x=xb.f32(), ldx=ne0, eps=eps)

    def rms(z):
        return z / np.sqrt((z * z).mean(-1, keepdims=True) + eps)
    if kind == "rmsnorm":
        a.kind, a.w = pyqwen.ACT_RMSNORM, wb.f32()
        v = rms(X) * WT
    elif kind == "cat":
        s = ne0 // 2
        a.kind, a.w, a.w2, a.y, a.ldy, a.seg = pyqwen.ACT_RMSNORM, wb.f32(), w2b.f32(), yb.f32(), ne0, s
        v = np.concatenate([rms(X[:, :s]) * WT[:s], rms(Y[:, :s]) * w2[:s].astype(np.float64)], 1)
    elif kind == "silu":
        a.kind, a.y, a.ldy = pyqwen.ACT_SILU_MUL, yb.f32(), ne0
        v = X / (1 + np.exp(-X)) * Y
    else:
        a.kind, a.y, a.ldy, a.w, a.seg = pyqwen.ACT_GATED_NORM, yb.f32(), ne0, wb.f32(), 128
        v = (rms(X.reshape(n, -1, 128)) * WT[:128]).reshape(n, ne0) * (Y / (1 + np.exp(-Y)))
    W = host.synth_matrix(8, ne0, ne1, 5, 6, 0.02)
    T, ob = gpu.tensor(W, 8, ne0, ne1), gpu.buf(n * ne1 * 4)
    with workspace(gpu, n, ne0) as w:
        gpu.ok(gpu.L.qgpu_wide_prepare(w, ctypes.byref(a), n, ne0, 1))
        gemm(gpu, w, [T], [ob], n)
        ref = v @ O.dequant_rows(8, W, ne0, ne1).reshape(ne1, ne0).astype(np.float64).T
        assert norm_err(ob.download(np.float32).reshape(n, ne1), ref) < 2e-6   # WIDE_TOL and the transform's own fp32 steps
    T.close()


def test_wide_rejects(gpu):
    """sizes, alignment and formats outside the path are errors"""
    W = host_lib().synth_matrix(23, 512, 16, 5, 6, 0.02)
    T, F = gpu.tensor(W, 23, 512, 16), gpu.tensor(np.zeros(512 * 16 * 4, np.uint8), 0, 512, 16)
    xb, ob = gpu.buf(200 * 512 * 4), gpu.buf(200 * 16 * 4)
    assert gpu.L.qgpu_wide_supports(T.h) == 1 and gpu.L.qgpu_wide_supports(F.h) == 0
    with workspace(gpu, 128, 512) as w:
        a = copy_act(xb, 512)
        assert gpu.L.qgpu_wide_prepare(w, ctypes.byref(a), 129, 512, 1) == -1
        assert gpu.L.qgpu_wide_prepare(w, ctypes.byref(a), 8, 768, 1) == -1
        a.ldx = 514
        assert gpu.L.qgpu_wide_prepare(w, ctypes.byref(a), 8, 512, 1) == -1
        h, o, ld = (ctypes.c_void_p * 1)(F.h), (pyqwen.F32P * 1)(ob.f32()), (ctypes.c_uint64 * 1)(16)
        assert gpu.L.qgpu_wide_gemm(w, h, 1, 8, o, ld, 0) == -2
        assert gpu.L.qgpu_wide_attn(w, xb.f32(), 512, xb.f32(), xb.f32(), 0, 1, 1, 1, 256, ob.f32(), 256) == -1
    T.close()
    F.close()


# ---------------------------------------------------------------- attention
@pytest.mark.parametrize("pos,n,n_ctx", [(0, 1, 512), (0, 33, 512), (31, 64, 512), (300, 65, 512), (447, 65, 512),
                                         (0, 200, 201)])
def test_wide_attention_vs_fp64(gpu, pos, n, n_ctx):
    nh, nkv, hd, rope_dim, theta, eps, _ = ATT_DIMS
    q, k, v, qw, kw, kc, vc, rc, rs = _attn_inputs(pos, n, n_ctx)
    ref, kref, vref = attn_fp64(q, k, v, qw, kw, kc, vc, pos, n, nh, nkv, hd, rope_dim, theta, eps)
    qb, kb, vb = gpu.put(q), gpu.put(k), gpu.put(v)
    kcb, vcb, ob = gpu.put(kc), gpu.put(vc), gpu.buf(n * nh * hd * 4)
    keep = [gpu.put(a) for a in (qw, kw, rc, rs, np.array([pos], np.int32))]
    with workspace(gpu, n, 256, n_ctx, nkv) as w:
        gpu.ok(gpu.L.qgpu_attn_prep(qb.f32(), 2 * nh * hd, kb.f32(), vb.f32(), nkv * hd, keep[0].f32(), keep[1].f32(),
                                    kcb.f32(), vcb.f32(), keep[2].f32(), keep[3].f32(), rope_dim, keep[4].i32(), n,
                                    nh, nkv, hd, eps))
        gpu.ok(gpu.L.qgpu_wide_attn(w, qb.f32(), 2 * nh * hd, kcb.f32(), vcb.f32(), pos, n, nh, nkv, hd, ob.f32(),
                                    nh * hd))
        got = ob.download(np.float32).reshape(n, nh * hd)
    # bf16 hi + lo parts of the probabilities and values: 2^-16 each, of random sign
    assert norm_err(got, ref) < 2e-5
    assert rel_err(kcb.download(np.float32).reshape(n_ctx, nkv, hd), kref) < 1e-5


@pytest.mark.parametrize("nh,nkv", [(6, 3), (2, 1), (16, 8)])
def test_wide_attention_head_counts(gpu, nh, nkv):
    """kv head counts that divide the 8 XCDs and one that does not, against the decode kernel"""
    n, pos, hd, rng = 40, 100, 256, np.random.default_rng(3)
    q = rng.standard_normal((n, nh * 2 * hd)).astype(np.float32)
    kc, vc = (rng.standard_normal((160, nkv * hd)).astype(np.float32) for _ in range(2))
    qb, kb, vb, ob, o8 = gpu.put(q), gpu.put(kc), gpu.put(vc), gpu.buf(n * nh * hd * 4), gpu.buf(n * nh * hd * 4)
    with workspace(gpu, n, 256, 160, nkv) as w:
        gpu.ok(gpu.L.qgpu_wide_attn(w, qb.f32(), 2 * nh * hd, kb.f32(), vb.f32(), pos, n, nh, nkv, hd, ob.f32(), nh * hd))
        got = ob.download(np.float32).reshape(n, nh * hd)
    for b in range(0, n, 8):
        p = gpu.put(np.array([pos + b], np.int32))
        x = gpu.put(np.ascontiguousarray(q[b:b + 8]))
        gpu.ok(gpu.L.qgpu_attn_decode(x.f32(), 2 * nh * hd, kb.f32(), vb.f32(), p.i32(), 160, 8, nh, nkv, hd, o8.f32(), nh * hd))
        assert norm_err(got[b:b + 8], o8.download(np.float32).reshape(n, -1)[:8]) < 2e-5


# ---------------------------------------------------------------- Gated DeltaNet
@pytest.mark.parametrize("n", [1, 2, 3, 5, 8, 33, 100])
@pytest.mark.parametrize("nk,nv,gate", [(16, 48, 1.0), (2, 4, 1.0), (2, 4, 40.0)])
def test_wide_gdn_vs_batches(gpu, n, nk, nv, gate):
    """against the same tokens in batches of 8 (qgpu_gdn_fused), which carries its own oracle tests; with
    strong gates the decay of a group of 8 tokens leaves fp32 (some single ones too)"""
    hk, eps, slots = 128, 1e-6, 9
    rng = np.random.default_rng(n + nk)
    chan = (2 * nk + nv) * hk
    x = rng.standard_normal((n, chan)).astype(np.float32)
    be, al = (rng.standard_normal((n, nv)).astype(np.float32) for _ in range(2))
    al *= np.float32(gate)
    cw = (0.5 * rng.standard_normal((chan, 4))).astype(np.float32)
    dtb = (0.5 * rng.standard_normal(nv)).astype(np.float32)
    a = (-(0.3 + 0.7 * np.abs(rng.standard_normal(nv)))).astype(np.float32)
    conv = np.zeros((slots, chan, 4), np.float32)
    ssm = np.zeros((slots, nv * hk * hk), np.float32)
    conv[0] = 0.5 * rng.standard_normal((chan, 4))
    ssm[0] = 0.05 * rng.standard_normal(nv * hk * hk)
    cwb, dtbb, ab = gpu.put(cw), gpu.put(dtb), gpu.put(a)
    cb, sb, cur, ref = gpu.put(conv), gpu.put(ssm), 0, []
    for b in range(0, n, 8):
        m = min(8, n - b)
        bufs = [gpu.put(np.ascontiguousarray(z[b:b + m])) for z in (x, be, al)]
        at, o = gpu.put(np.array([cur], np.int32)), gpu.buf(m * nv * hk * 4)
        gpu.ok(gpu.L.qgpu_gdn_fused(bufs[0].f32(), chan, m, chan, cwb.f32(), cb.f32(), chan * 4, bufs[1].f32(),
                                    bufs[2].f32(), nv, dtbb.f32(), ab.f32(), sb.f32(), nv * hk * hk, slots, at.i32(),
                                    nk, nv, hk, eps, o.f32(), nv * hk))
        ref.append(o.download(np.float32).reshape(m, -1))
        cur = (cur + m) % slots
    cref, sref = cb.download(np.float32).reshape(slots, -1)[cur], sb.download(np.float32).reshape(slots, -1)[cur]
    c2, s2 = gpu.put(conv), gpu.put(ssm)
    xb, bb, alb, ob = gpu.put(x), gpu.put(be), gpu.put(al), gpu.buf(n * nv * hk * 4)

    def slot(buf, size):
        return ctypes.cast(ctypes.c_void_p(ctypes.cast(buf.f32(), ctypes.c_void_p).value + size * 4), pyqwen.F32P)
    with workspace(gpu, n, 256, 0, 0, nk, nv) as w:
        gpu.ok(gpu.L.qgpu_wide_gdn(w, xb.f32(), chan, n, cwb.f32(), c2.f32(), slot(c2, chan * 4), bb.f32(), alb.f32(), nv,
                                   dtbb.f32(), ab.f32(), s2.f32(), slot(s2, nv * hk * hk), nk, nv, hk, eps, ob.f32(),
                                   nv * hk))
        got = ob.download(np.float32).reshape(n, -1)
    # fp32 on both sides, sums of 128 in another order: some 2^-24 of each, n steps under decay
    assert norm_err(got, np.concatenate(ref)) < 2e-6
    cn, sn = c2.download(np.float32).reshape(slots, -1), s2.download(np.float32).reshape(slots, -1)
    assert np.array_equal(cn[1], cref) and norm_err(sn[1], sref) < 2e-6
    assert np.array_equal(cn[0], conv[0].ravel()) and np.array_equal(sn[0], ssm[0])


# ---------------------------------------------------------------- whole prompts
@pytest.fixture(scope="module")
def tiny_path():
    td = tempfile.mkdtemp()
    path = os.path.join(td, "m.gguf")
    host_lib().write_tiny_gguf(path, 11, 0)
    yield path
    os.remove(path)


@pytest.mark.parametrize("n,n_ctx", [(16, 64), (17, 64), (24, 64), (25, 64), (63, 64), (137, 256), (2100, 2200)])
@pytest.mark.parametrize("k", [0, 3])
def test_prompt_equals_batches(gpu, tiny_path, n, n_ctx, k):
    """model_spec_begin against the same prompt in batches of 8 through model_forward_batch and
    mtp_forward_batch: last logits, hidden rows of the last batch and the cycles that follow; a second
    prompt on the same model after a reset"""
    rng = np.random.RandomState(n)
    m, r = pyqwen.Model(tiny_path, n_ctx), pyqwen.Model(tiny_path, n_ctx)
    for turn in range(2):
        p = rng.randint(0, 1024, n).astype(np.uint32)
        m.reset()
        r.reset()
        m.spec_begin(p, k)
        for b in range(0, n, 8):
            c = p[b:b + 8]
            lb = r.forward_batch(c, b)
            if k:
                r.mtp_forward_batch(c, b)
        last = m.field("logits", m.V)
        # 2^-22-exact activations on either side (the batches' digits are 2^-23 of a super-block's maximum),
        # through four layers
        assert rel_err(last, lb[-1]) < 1e-4
        room = n_ctx - n
        if room >= 2:
            cyc = min(4, max(1, room // (k + 1) - 1))
            t, js, _ = m.spec_run(k, cyc)
            nxt, got = int(np.argmax(lb[-1])), []
            pos = n
            for tok in t[:4]:                                   # greedy continuation of the batches' model
                if np.diff(np.sort(lb[-1])[-2:])[0] < 1e-3 * np.abs(lb[-1]).max():
                    break                                       # a near tie: either order is right
                assert int(tok) == nxt
                if pos >= n_ctx:
                    break
                lb = r.forward_batch(np.array([nxt], np.uint32), pos)
                nxt, pos = int(np.argmax(lb[-1])), pos + 1
    m.close()
    r.close()
