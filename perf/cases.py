"""Timed cases of the framework: the nets as hosts call them, and their single layers through the kernel-level ABI.

A case is a dict of plain values. The nets go through the bnn_* host API (bnneon.binding), the layers through
include/bnneon_hip.h (bnneon.hip) on device buffers, as a host that keeps its activations on the GPU calls them.
Weights depend on a layer's shape alone (a model's weights are the same for every input), inputs on the seed.
"""
import ctypes
import functools
import math
import os
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "birdnet-neon-engine_amd"))

from bnneon import binding, hip, netbuild, perchnet, s8pack, v24net  # noqa: E402

ACT = {"none": 0, "silu": 1, "relu": 2}


# ------------------------------------------------------------------------------------------------ the list
def listed():
    return [
        # a recorder in the field scores each 5 s window as it is complete: one bnn_infer from host memory, where
        # launches and short serial kernels count
        dict(name="perch_int8_live", op="net", net="perch_int8", windows=1, host=True),
        # an archive of recordings, windows already on the GPU, at the batch the framework's benchmark uses
        dict(name="perch_int8_archive", op="net", net="perch_int8", windows=256, host=False),
        # a station that collects 3 s windows of many microphones: a middle-sized fp16 batch
        dict(name="v24_fp16_station", op="net", net="v24_fp16", windows=48, host=False),
        # an MBConv block's projection on the int8 path: SE gate in, residual added (63 x 16 px, 288 -> 48)
        dict(name="pw_s8_project", op="pw_s8", windows=40, h=63, w=16, k=288, n=48, act="none", gate=True, res=True,
             halo=0),
        # the int8 expansion that runs inside the depthwise conv after it (48 -> 288, 5x5, 63 x 16 px), rows
        # quantised first; outputs and the SE's channel sums
        dict(name="expand_dw_s8", op="expand_dw", windows=36, h=63, w=16, k=48, c=288, ks=5, s=1),
        # the fp32 path's 1x1 conv (also what a default int8 build leaves in fp32): expansion with SiLU into the
        # zero-haloed input of the depthwise conv
        dict(name="pw_f32_expand", op="pw_f32", windows=48, h=32, w=8, k=136, n=816, act="silu", gate=False, res=False,
             halo=2),
        # the fp16 path's gated projection with its residual, K in several blocks (16 x 6 px, 864 -> 108)
        dict(name="pw_f16_project", op="pw_f16", windows=33, h=16, w=6, k=864, n=108, act="none", gate=True, res=True,
             halo=0),
        # the dotprod family's 1x1 conv: gated fp16 rows in, fp16 SiLU out with a halo
        dict(name="qpw_f16", op="qpw", windows=12, h=56, w=117, k=64, n=256, act="silu", gate=True, f16=True, halo=1),
        # the fp16 path's depthwise conv with its channel sums (stride 1, 32 x 12 px x 288)
        dict(name="dw_f16_sums", op="dw", dtype="f16", windows=64, h=32, w=12, c=288, ks=3, s=1),
        # a dense 3x3 conv of the fp16 Winograd path at half the benchmark's image
        dict(name="wino_f16_dense", op="wino", windows=9, h=96, w=128, c=64, k=64, act="silu"),
        # Perch's prototype head on int8: 64 cells x 1536 against 14,795 classes x 4 prototypes
        dict(name="proto_s8_head", op="proto", dtype="s8", windows=20, cells=64, c=1536, classes=14795, ppc=4),
        # the fp32 prototype head with one prototype per class
        dict(name="proto_f32_head", op="proto", dtype="f32", windows=3, cells=64, c=1536, classes=5000, ppc=1),
    ]


def _log(rng, lo, hi):
    """An integer in [lo, hi], even over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _image(rng, limit, per_pixel):
    """(windows, h, w) with at most limit elements in windows * h * w * per_pixel."""
    h, w = _log(rng, 4, 256), _log(rng, 3, 128)
    most = max(1, min(256, limit // (h * w * per_pixel)))
    return _log(rng, 1, most), h, w


def draw(rng):
    op = rng.choice(["net", "pw_s8", "expand_dw", "pw_f32", "pw_f16", "qpw", "dw", "wino", "proto"])
    act = rng.choice(["none", "silu", "relu"])
    if op == "net":
        host = rng.random() < 0.5
        return dict(op=op, net=rng.choice(["perch_int8", "v24_fp16"]), windows=_log(rng, 1, 64 if host else 240),
                    host=host)
    if op in ("pw_s8", "pw_f32", "pw_f16", "qpw"):
        k, n = 4 * _log(rng, 4, 576), _log(rng, 16, 1536)
        if op == "pw_s8" and 48 < k <= 64:  # rows of exactly 64 int8 columns came out wrong once: not compared here
            k = 48
        b, h, w = _image(rng, min(96 << 20, (10 << 30) // (k * n) * (k + n)), k + n)
        c = dict(op=op, windows=b, h=h, w=w, k=k, n=n, act=act, gate=rng.random() < 0.5, res=rng.random() < 0.4,
                 halo=rng.choice([0, 0, 1]))
        if op == "qpw":
            c["f16"] = rng.random() < 0.5
            c["gate"] = c["gate"] and c["f16"]
            del c["res"]
            if c["f16"] and act == "relu":
                c["act"] = "silu"
            c["halo"] = c["halo"] if c["f16"] else 0
        elif c["halo"]:
            c["res"] = False
        return c
    if op == "expand_dw":
        k, e = 8 * _log(rng, 2, 48), rng.choice([4, 6])
        c = (k * e + 15) // 16 * 16
        b, h, w = _image(rng, 64 << 20, k + c)
        ks, s = rng.choice([3, 5]), rng.choice([1, 2])
        while 4 * (ks * (20 * (w + ks + 4) + 80) + 64) + (ks * w + 16) * (28 + k) > 52 << 10:
            w = (w + 1) // 2  # the fused kernel takes images up to the width whose rows fit its block
        return dict(op=op, windows=b, h=h, w=w, k=k, c=c, ks=ks, s=s)
    if op == "dw":
        c = 8 * _log(rng, 3, 240)
        b, h, w = _image(rng, 64 << 20, c)
        return dict(op=op, dtype=rng.choice(["f16", "f32"]), windows=b, h=h, w=w, c=c, ks=rng.choice([3, 5]),
                    s=rng.choice([1, 2]))
    if op == "wino":
        c, k = 8 * rng.randint(2, 8), 8 * rng.randint(2, 8)
        b, h, w = _image(rng, 48 << 20, c + k)
        return dict(op=op, windows=b, h=2 * ((h + 1) // 2), w=2 * ((w + 1) // 2), c=c, k=k, act=act)
    dtype = rng.choice(["s8", "f32", "f32h", "f16"])
    cells, c, ppc = 8 * rng.randint(3, 12), 8 * _log(rng, 24, 192), rng.choice([1, 2, 4])
    classes = _log(rng, 400, 14795 if dtype == "s8" else 6000)
    most = (120 << 30 if dtype == "s8" else 24 << 30) // (cells * c * classes * ppc)
    return dict(op=op, dtype=dtype, windows=_log(rng, 1, max(1, min(128, most))), cells=cells, c=c, classes=classes,
                ppc=ppc)


# ------------------------------------------------------------------------------------------------ helpers
def _r(n, m):
    return (n + m - 1) // m * m


def _p(t):
    return None if t is None else t.data_ptr()


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _acts(g, *shape):
    """What a layer of these nets reads: values after a SiLU or a residual sum."""
    x = _randn(g, *shape) * 1.5
    return x * torch.sigmoid(x) + 0.1 * _randn(g, *shape)


def _same(n, k, s):
    """TF 'same': output size and leading pad."""
    o = (n - 1) // s + 1
    return o, max((o - 1) * s + k - n, 0) // 2


def _weights(n, k, gain=1.0):
    """(w [n][k], b [n]) of a layer: a function of its shape alone."""
    rng = np.random.default_rng(1000003 * n + k)
    return ((rng.standard_normal((n, k)) * gain * np.sqrt(2.0 / k)).astype(np.float32),
            (rng.standard_normal(n) * 0.1).astype(np.float32))


def _panels16(w, kp):
    return netbuild.Net.pack_h16(w, np.zeros(len(w), np.float32), kp)


class _Handle:
    """A weight handle of the library, freed with this object."""

    def __init__(self, h, free):
        if not h:
            hip.check(None, "weights")
        self.h, self.free = h, free

    def __del__(self):
        try:
            self.free(self.h)
        except Exception:
            pass


@functools.lru_cache(maxsize=4)
def _s8w(n, k):
    pk = s8pack.pack_s8(*_weights(n, k))
    return hip.S8Weights(n, k, pk["shape"][2], pk["shape"][3], pk["q"], pk["sw"], pk["cs"], pk["b"])


@functools.lru_cache(maxsize=4)
def _h16w(n, k):
    w, b = _weights(n, k)
    panels, b32, b16, (_, _, kp, np_) = netbuild.Net.pack_h16(w, b, _r(k, 8))
    L = hip.lib()
    return _Handle(L.bnh_h16w_new(n, k, kp, np_, panels.ctypes.data, b32.ctypes.data, b16.ctypes.data),
                   L.bnh_h16w_free)


@functools.lru_cache(maxsize=4)
def _qdw(n, k):
    w, b = _weights(n, k)
    L = hip.lib()
    return _Handle(L.bnh_qdw_new(w.ctypes.data, b.ctypes.data, n, k, n), L.bnh_qdw_free)


@functools.lru_cache(maxsize=4)
def _wino(c, k):
    w, b = _wino_weights(c, k)
    L = hip.lib()
    return _Handle(L.bnh_wino16_new(c, k, w.ctypes.data, b.ctypes.data), L.bnh_wino16_free)


def _wino_weights(c, k):
    w, b = _weights(k, 9 * c)
    return w.reshape(k, 3, 3, c).astype(np.float16).astype(np.float32), b


@functools.lru_cache(maxsize=2)
def _protos(n, k):
    return np.random.default_rng(7 * n + k).standard_normal((n, k), np.float32) * np.float32(np.sqrt(2.0 / k))


@functools.lru_cache(maxsize=2)
def _proto_handle(dtype, n, k):
    """(handle, padded prototypes) of a head."""
    p, L = _protos(n, k), hip.lib()
    if dtype == "s8":
        kp, np_ = _r(k, 16), _r(n, 4)
        q, sw = s8pack.quant_rows_s8(p)
        qp, swp = np.zeros((np_, kp), np.int8), np.zeros(np_, np.float32)
        qp[:n, :k], swp[:n] = q, sw
        panels = s8pack.pack_panels(qp)
        return _Handle(L.bnh_s8p_new(np_, kp, panels.ctypes.data, swp.ctypes.data), L.bnh_s8p_free), np_
    if dtype == "f32":
        panels, _, (_, _, _, np_) = netbuild.Net.fpack(p, np.zeros(n, np.float32), K_pad=8)
        return hip.FProto(0, np_, k, panels), np_
    if dtype == "f16":
        panels, _, _, (_, _, _, np_) = _panels16(p, k)
        return hip.FProto(2, np_, k, panels), np_
    np_ = _r(n, 8)
    w = np.zeros((np_, k), np.float16)
    w[:n] = p
    return hip.FProto(1, np_, k, np.ascontiguousarray(w.reshape(np_ // 8, 8, k).transpose(0, 2, 1))), np_


@functools.lru_cache(maxsize=2)
def _model(net):
    """The net's context: a program keeps it for every window it scores."""
    build = {"perch_int8": lambda: perchnet.PerchNet(seed=0), "v24_fp16": lambda: v24net.V24Net(seed=0)}[net]
    with tempfile.TemporaryDirectory() as d:
        path = build().write(os.path.join(d, net + ".bnpk"))
        return binding.Model(path)


def _windows(net, n, seed):
    """-30 dBFS noise and two chirps a window, on the GPU [n][n_samples]."""
    sr, ns = (perchnet.SR, perchnet.NSAMP) if net == "perch_int8" else (v24net.SR, v24net.NSAMP)
    g = _gen(seed)
    x = _randn(g, n, ns) * 10 ** (-30 / 20)
    t = torch.arange(ns, device="cuda", dtype=torch.float32)[None] / sr
    u = torch.rand((2, 5, n, 1), generator=g, device="cuda")
    for f0, f1, t0, d, a in u:
        f0, f1, t0, d = 1000 + 9000 * f0, 1000 + 9000 * f1, 2 * t0, 0.2 + 0.8 * d
        tt = t - t0
        on = (tt >= 0) & (tt < d)
        x += torch.where(on, 0.2 * a * torch.sin(2 * math.pi * (f0 * tt + (f1 - f0) / (2 * d) * tt * tt)), 0.0)
    return x


# ------------------------------------------------------------------------------------------------ prepare
def prepare(case, seed):
    return _PREPARE[case["op"]](case, seed)


def _prepare_net(c, seed):
    m, n = _model(c["net"]), c["windows"]
    pcm = _windows(c["net"], n, seed)
    if c["host"]:
        return dict(c=c, m=m, pcm=pcm.cpu().numpy())
    return dict(c=c, m=m, pcm=pcm, out=torch.zeros((n, m.info.n_classes), device="cuda"),
                emb=torch.zeros((n, m.info.emb_dim), device="cuda"), status=np.zeros(n, np.int32))


def _epi_rows(c):
    return (c["h"] + 2 * c["halo"]) * (c["w"] + 2 * c["halo"])


def _prepare_pw_s8(c, seed):
    g, b, m, lda, W = _gen(seed), c["windows"], c["h"] * c["w"], _r(c["k"], 8), _s8w(c["n"], c["k"])
    x = _acts(g, b, m, lda)
    gate = torch.sigmoid(_randn(g, b, c["k"])) if c["gate"] else None
    res = _acts(g, b, m, W.Np) if c["res"] else None
    out = torch.zeros((b, _epi_rows(c), W.Np), device="cuda")
    m4 = _r(m, 4)
    return dict(c=c, x=x, gate=gate, res=res, out=out, W=W, q=torch.zeros((b, m4, W.Kp), dtype=torch.int8, device="cuda"),
                sa=torch.zeros((b, m4), device="cuda"), za=torch.zeros((b, m4), dtype=torch.int32, device="cuda"),
                e=hip.Epi32(ACT[c["act"]], _p(out), out[0].numel(), W.Np, c["w"], c["halo"], _p(res),
                            m * W.Np, W.Np if c["res"] else 0, 0, 0))


def _prepare_pw_f32(c, seed):
    g, b, m = _gen(seed), c["windows"], c["h"] * c["w"]
    panels, bias, (_, _, kp, np_) = netbuild.Net.fpack(*_weights(c["n"], c["k"]))
    x = _acts(g, b, m, _r(kp, 8))
    gate = torch.sigmoid(_randn(g, b, kp)) if c["gate"] else None
    res = _acts(g, b, m, np_) if c["res"] else None
    out = torch.zeros((b, _epi_rows(c), np_), device="cuda")
    return dict(c=c, x=x, gate=gate, res=res, out=out, kp=kp, np=np_, w=torch.from_numpy(np.ascontiguousarray(panels)).cuda(),
                bias=torch.from_numpy(bias).cuda(),
                e=hip.Epi32(ACT[c["act"]], _p(out), out[0].numel(), np_, c["w"], c["halo"], _p(res), m * np_,
                            np_ if c["res"] else 0, 0, 0))


def _prepare_pw_f16(c, seed):
    g, b, m, kp, np_ = _gen(seed), c["windows"], c["h"] * c["w"], _r(c["k"], 8), _r(c["n"], 8)
    W = _h16w(c["n"], c["k"])
    x = _acts(g, b, m, kp)
    x[:, :, c["k"]:] = 0
    x = x.half()
    gate = torch.sigmoid(_randn(g, b, kp)).half() if c["gate"] else None
    res = _acts(g, b, m, np_).half() if c["res"] else None
    out = torch.zeros((b, _epi_rows(c), np_), dtype=torch.float16, device="cuda")
    ws = int(hip.lib().bnh_gemm_f16_ws_bytes(m, b, W.h))
    return dict(c=c, x=x, gate=gate, res=res, out=out, kp=kp, np=np_, W=W, ws_bytes=ws,
                ws=torch.zeros(max(ws, 16), dtype=torch.uint8, device="cuda"),
                e=hip.Epi16(ACT[c["act"]], _p(out), out[0].numel(), np_, c["w"], c["halo"], _p(res), m * np_,
                            np_ if c["res"] else 0))


def _prepare_qpw(c, seed):
    g, b, m, k = _gen(seed), c["windows"], c["h"] * c["w"], c["k"]
    n = _r(c["n"], 16)
    x = _acts(g, b, m, _r(k, 8))
    gate = None
    if c["f16"]:
        x = x.half()
        gate = torch.sigmoid(_randn(g, b, k)).half() if c["gate"] else None
    out = torch.zeros((b, _epi_rows(c), n), dtype=torch.float16 if c["f16"] else torch.float32, device="cuda")
    return dict(c=c, x=x, gate=gate, out=out, W=_qdw(n, k), kp=_r(k, 16),
                a=torch.zeros((b, m, _r(k, 16)), dtype=torch.int8, device="cuda"),
                rq=torch.zeros((b, m, 2), device="cuda"),
                e=hip.QdEpi(ACT[c["act"]], int(c["f16"]), _p(out), out[0].numel(), n, c["w"], c["halo"], None, 0))


def _dw_params(c):
    rng = np.random.default_rng(31 * c["c"] + c["ks"])
    kk = c["ks"] ** 2
    return ((rng.standard_normal((kk, c["c"])) * np.sqrt(2.0 / kk)).astype(np.float32),
            (rng.standard_normal(c["c"]) * 0.1).astype(np.float32))


def _dw_geometry(c):
    """(Ho, Wo, pt, pl, fp32 DW3 form) as the nets' builders choose them."""
    (ho, pt), (wo, pl) = _same(c["h"], c["ks"], c["s"]), _same(c["w"], c["ks"], c["s"])
    return ho, wo, pt, pl, c["ks"] == 3 and pt == 1 and pl == 1


def _prepare_expand_dw(c, seed):
    g, b, m, W = _gen(seed), c["windows"], c["h"] * c["w"], _s8w(c["c"], c["k"])
    ho, wo = _dw_geometry(c)[:2]
    w, bias = _dw_params(c)
    m4 = _r(m, 4)
    return dict(c=c, x=_acts(g, b, m, c["k"]), W=W, w=torch.from_numpy(w).cuda(), bias=torch.from_numpy(bias).cuda(),
                q=torch.zeros((b, m4, W.Kp), dtype=torch.int8, device="cuda"), sa=torch.zeros((b, m4), device="cuda"),
                za=torch.zeros((b, m4), dtype=torch.int32, device="cuda"),
                out=torch.zeros((b, ho, wo, c["c"]), device="cuda"), sums=torch.zeros((b, c["c"]), device="cuda"))


def _prepare_dw(c, seed):
    g, b, h = _gen(seed), c["windows"], (c["ks"] - 1) // 2
    ho, wo = _dw_geometry(c)[:2]
    w, bias = _dw_params(c)
    dt = torch.float16 if c["dtype"] == "f16" else torch.float32
    x = torch.zeros((b, c["h"] + 2 * h, c["w"] + 2 * h, c["c"]), dtype=dt, device="cuda")
    x[:, h:h + c["h"], h:h + c["w"]] = _acts(g, b, c["h"], c["w"], c["c"]).to(dt)
    return dict(c=c, x=x, w=torch.from_numpy(w).cuda().to(dt), bias=torch.from_numpy(bias).cuda().to(dt),
                out=torch.zeros((b, ho, wo, c["c"]), dtype=dt, device="cuda"),
                sums=torch.zeros((b, c["c"]), device="cuda"))


def _prepare_wino(c, seed):
    g, b = _gen(seed), c["windows"]
    x = torch.zeros((b, c["h"] + 2, c["w"] + 2, c["c"]), dtype=torch.float16, device="cuda")
    x[:, 1:-1, 1:-1] = _acts(g, b, c["h"], c["w"], c["c"]).half()
    return dict(c=c, x=x, W=_wino(c["c"], c["k"]),
                out=torch.zeros((b, c["h"], c["w"], c["k"]), dtype=torch.float16, device="cuda"))


def _classes(c):
    rng = np.random.default_rng(c["classes"])
    return (rng.uniform(0.5, 1.5, (c["classes"], c["ppc"])).astype(np.float32),
            (rng.standard_normal(c["classes"]) * 0.1).astype(np.float32))


def _prepare_proto(c, seed):
    b, P, k = c["windows"], c["cells"], c["c"]
    W, np_ = _proto_handle(c["dtype"], c["classes"] * c["ppc"], k)
    cw, cb = _classes(c)
    x = _acts(_gen(seed), b, P, k)
    s = dict(c=c, W=W, np=np_, cw=torch.from_numpy(cw).cuda(), cb=torch.from_numpy(cb).cuda(),
             colmax=torch.zeros((b, np_), device="cuda"), logits=torch.zeros((b, c["classes"]), device="cuda"),
             fail=torch.zeros(b, dtype=torch.int32, device="cuda"))
    if c["dtype"] == "s8":
        s.update(x=x, q=torch.zeros((b, P, _r(k, 16)), dtype=torch.int8, device="cuda"),
                 sx=torch.zeros((b, P), device="cuda"))
    else:
        x = x.half() if c["dtype"] == "f16" else x
        s.update(x=x, a=torch.zeros_like(x))
    return s


# ------------------------------------------------------------------------------------------------ run
def run(state):
    return _RUN[state["c"]["op"]](state)


def _run_net(s):
    m, c = s["m"], s["c"]
    if c["host"]:
        if c["windows"] == 1:
            return m.infer(s["pcm"][0])
        return m.infer_batch(s["pcm"])[:2]
    hip.check(m.L.bnn_infer_batch_device(m.ctx, _p(s["pcm"]), c["windows"], _p(s["out"]), _p(s["emb"]),
                                         s["status"].ctypes.data_as(ctypes.POINTER(ctypes.c_int)), None), "infer")
    return s["out"], s["emb"]


def _run_pw_s8(s):
    c, W, x = s["c"], s["W"], s["x"]
    m, m4 = c["h"] * c["w"], s["sa"].shape[1]
    hip.check(hip.lib().bnh_pw_s8(_p(x), x[0].numel(), x.shape[2], m, _p(s["gate"]), c["k"], _p(s["q"]), m4 * W.Kp,
                                  _p(s["sa"]), m4, _p(s["za"]), m4, c["windows"], W.h, s["e"], None), "pw_s8")
    return s["out"]


def _run_pw_f32(s):
    c, x = s["c"], s["x"]
    hip.check(hip.lib().bnh_gemm_f32(_p(x), x[0].numel(), x.shape[2], c["h"] * c["w"], _p(s["gate"]), s["kp"],
                                     _p(s["w"]), _p(s["bias"]), s["kp"], s["np"], s["e"], c["windows"], None),
              "gemm_f32")
    return s["out"]


def _run_pw_f16(s):
    c, L, m = s["c"], hip.lib(), s["c"]["h"] * s["c"]["w"]
    a = (_p(s["x"]), m * s["kp"], s["kp"], m, c["windows"], s["W"].h, s["e"])
    if c["gate"]:
        hip.check(L.bnh_gemm_f16_gated_ws(*a, _p(s["gate"]), s["kp"], _p(s["ws"]), s["ws_bytes"], None), "gemm_f16")
    else:
        hip.check(L.bnh_gemm_f16_ws(*a, _p(s["ws"]), s["ws_bytes"], None), "gemm_f16")
    return s["out"]


def _run_qpw(s):
    c, x, L, m, kp = s["c"], s["x"], hip.lib(), s["c"]["h"] * s["c"]["w"], s["kp"]
    hip.check(L.bnh_qd_quant_rows(_p(x), int(c["f16"]), x[0].numel(), x.shape[2], m, c["k"], _p(s["gate"]), c["k"],
                                  _p(s["a"]), m * kp, _p(s["rq"]), 2 * m, c["windows"], None), "qd_quant_rows")
    hip.check(L.bnh_qd_gemm(_p(s["a"]), m * kp, kp, _p(s["rq"]), 2 * m, 0, m, s["W"].h, s["e"], c["windows"], None),
              "qd_gemm")
    return s["out"]


def _run_expand_dw(s):
    c, W, L = s["c"], s["W"], hip.lib()
    m, m4, (ho, wo, pt, pl, dw3) = c["h"] * c["w"], s["sa"].shape[1], _dw_geometry(c)
    hip.check(L.bnh_s8n_quant_rows(_p(s["x"]), m * c["k"], c["k"], m, c["k"], W.Kp, None, 0, _p(s["q"]), m4 * W.Kp,
                                   _p(s["sa"]), m4, _p(s["za"]), m4, c["windows"], None), "quant_rows")
    hip.check(L.bnh_pwdw_f32(_p(s["q"]), m4 * W.Kp, _p(s["sa"]), m4, _p(s["za"]), m4, c["h"], c["w"], W.h, 1, c["ks"],
                             c["s"], pt, pl, 2 if dw3 else 0, _p(s["w"]), _p(s["bias"]), 1, _p(s["out"]),
                             s["out"][0].numel(), ho, wo, _p(s["sums"]), c["c"], c["windows"], None), "pwdw")
    return s["out"], s["sums"]


def _run_dw(s):
    c, x, L = s["c"], s["x"], hip.lib()
    ho, wo, pt, pl, dw3 = _dw_geometry(c)
    a = (_p(x), x[0].numel(), c["h"], c["w"], c["c"])
    z = (_p(s["out"]), s["out"][0].numel(), ho, wo, _p(s["sums"]), c["c"], c["windows"], None)
    wb = (_p(s["w"]), _p(s["bias"]))
    if c["dtype"] == "f16" and c["ks"] == 3:
        hip.check(L.bnh_dw3_f16(*a, c["s"], pt, pl, *wb, *z), "dw3_f16")
    elif c["dtype"] == "f16":
        hip.check(L.bnh_dwk_f16(*a, c["ks"], c["s"], pt, pl, *wb, 1, *z), "dwk_f16")
    elif dw3:
        hip.check(L.bnh_dw3_f32(*a, c["s"], *wb, *z), "dw3_f32")
    else:
        hip.check(L.bnh_dwk_f32(*a, c["ks"], c["s"], pt, pl, *wb, 1, *z), "dwk_f32")
    return s["out"], s["sums"]


def _run_wino(s):
    c, x = s["c"], s["x"]
    hip.check(hip.lib().bnh_wino_f16(_p(x), x[0].numel(), c["h"], c["w"], c["c"], s["W"].h, ACT[c["act"]],
                                     _p(s["out"]), s["out"][0].numel(), c["k"], 0, None, 0, 0, 0, c["windows"], None),
              "wino_f16")
    return s["out"]


def _run_proto(s):
    c, x, L = s["c"], s["x"], hip.lib()
    b, P, k = c["windows"], c["cells"], c["c"]
    if c["dtype"] == "s8":
        kp = s["q"].shape[2]
        hip.check(L.bnh_quant_cells(_p(x), P * k, P, k, k, 1e-5, _p(s["q"]), P * kp, kp, _p(s["sx"]), P, b, None), "cells")
        hip.check(L.bnh_proto_colmax(_p(s["q"]), P * kp, _p(s["sx"]), P, P, s["W"].h, _p(s["colmax"]), s["np"], b, None),
                  "colmax")
    else:
        hip.check(L.bnh_l2norm_cells(_p(x), P * k, P, k, k, 1e-5, int(c["dtype"] == "f16"), _p(s["a"]), P * k, b, None),
                  "l2norm")
        hip.check(L.bnh_fproto_colmax(_p(s["a"]), P * k, P, s["W"].h, _p(s["colmax"]), s["np"], b, None), "colmax")
    hip.check(L.bnh_proto_logits(_p(s["colmax"]), s["np"], _p(s["cw"]), _p(s["cb"]), c["classes"], c["ppc"],
                                 _p(s["logits"]), c["classes"], b, _p(s["fail"]), 1, None), "logits")
    return s["logits"], s["colmax"]


# ------------------------------------------------------------------------------------------------ work
def _net_work(net):
    """(multiply-adds a window, bytes of weights, samples, outputs) of a net, from its builder's block table."""
    if net == "perch_int8":
        h, w, c0, ns, nc, emb, es = 249, 63, perchnet.STEM_C, perchnet.NSAMP, perchnet.N_CLASSES, perchnet.EMB, 1
        blocks = perchnet.blocks()
    else:
        h, w, c0, ns, nc, emb, es = 128, 47, v24net.STEM_C, v24net.NSAMP, v24net.N_CLASSES, v24net.EMB, 2
        blocks = [(ci, ce, 3, s, co) for ci, ce, s, co in v24net.blocks()]
    macs, weights = 9 * c0 * h * w, 0
    for ci, ce, k, s, co in blocks:
        if ce != ci:
            macs, weights = macs + h * w * ci * ce, weights + ci * ce * es
        h, w = (h - 1) // s + 1, (w - 1) // s + 1
        rd = max(1, ci // 4)
        macs += h * w * ce * (k * k + co) + 2 * rd * ce
        weights += ce * co * es + 4 * ce * (k * k + 2 * rd)
    macs += h * w * blocks[-1][4] * emb + emb * nc
    return macs, weights + (blocks[-1][4] * emb + emb * nc) * es, ns, nc + emb


def work(case):
    c, op = case, case["op"]
    b = c["windows"]
    if op == "net":
        macs, weights, ns, outs = _net_work(c["net"])
        return dict(bytes=weights + 4 * b * (ns + outs), flops=2 * macs * b)
    if op in ("pw_s8", "pw_f32", "pw_f16", "qpw"):
        m = b * c["h"] * c["w"]
        es = 2 if op == "pw_f16" or (op == "qpw" and c["f16"]) else 4
        wb = {"pw_s8": 1, "qpw": 1, "pw_f16": 2, "pw_f32": 4}[op]
        return dict(bytes=m * (c["k"] + c["n"] * (2 if c.get("res") else 1)) * es + wb * c["k"] * c["n"],
                    flops=2 * m * c["k"] * c["n"])
    if op == "expand_dw":
        ho, wo = _dw_geometry(c)[:2]
        return dict(bytes=4 * b * (c["h"] * c["w"] * c["k"] + ho * wo * c["c"]) + c["k"] * c["c"],
                    flops=2 * b * (c["h"] * c["w"] * c["k"] * c["c"] + ho * wo * c["c"] * c["ks"] ** 2))
    if op == "dw":
        ho, wo = _dw_geometry(c)[:2]
        es = 2 if c["dtype"] == "f16" else 4
        return dict(bytes=es * b * c["c"] * (c["h"] * c["w"] + ho * wo), flops=2 * b * ho * wo * c["c"] * c["ks"] ** 2)
    if op == "wino":  # the 16 products of a 2 x 2 tile
        px = b * c["h"] * c["w"]
        return dict(bytes=2 * px * (c["c"] + c["k"]) + 32 * c["c"] * c["k"], flops=2 * 4 * px * c["c"] * c["k"])
    n = c["classes"] * c["ppc"]
    es, ws = {"s8": (4, 1), "f32": (4, 4), "f32h": (4, 2), "f16": (2, 2)}[c["dtype"]]
    return dict(bytes=es * b * c["cells"] * c["c"] + ws * n * c["c"] + 4 * b * (n + c["classes"]),
                flops=2 * b * c["cells"] * n * c["c"])


# ------------------------------------------------------------------------------------------------ tolerance
# Layers: four times the largest error against exact() seen over the listed and drawn cases (the error of a second
# implementation at the same precision is of that size); "max" allows for one value at a tie of its grid, or one
# rounding of a cancelling sum. Nets: the fp16 net with its 1x1 convs summed in another order and precision (its
# matrix-core form) moves the logits by 2e-4 of their range, int8 codes that go the other way about as much a layer.
def tolerance(case):
    op = case["op"]
    if op == "net":
        return dict(rel=4e-3, max=5e-2)
    if op in ("pw_s8", "expand_dw"):   # 32-bit values, but an activation at a tie of its int8 grid may go either way
        return dict(rel=1.2e-4, max=2e-2)
    if op == "pw_f32":                 # 32-bit sums, a one-step reciprocal in the SiLU
        return dict(rel=2e-5, max=1e-3)
    if op == "pw_f16":                 # fp16 sums of up to 128 terms
        return dict(rel=4e-3, max=5e-2)
    if op == "qpw":                    # rows on an int8 grid whose step is rounded to fp16, fp16 out; or all 32-bit
        return dict(rel=7e-3, max=5e-2) if case["f16"] else dict(rel=1.2e-4, max=2e-2)
    if op == "dw":                     # 9 or 25 terms
        return dict(rel=3e-3, max=5e-2) if case["dtype"] == "f16" else dict(rel=2e-5, max=1e-3)
    if op == "wino":                   # fp16 transforms
        return dict(rel=2.5e-3, max=5e-2)
    if case["dtype"] == "f16":
        return dict(rel=4e-3, max=5e-2)
    return dict(rel=6e-5, max=1e-2) if case["dtype"] == "s8" else dict(rel=3e-6, max=1e-4)


# ------------------------------------------------------------------------------------------------ exact
def exact(case, seed):
    """The layers in 64 bits with plain torch; None for a whole net."""
    if case["op"] == "net":
        return None
    return _EXACT[case["op"]](case, prepare(case, seed))


def _act(y, act):
    return y * torch.sigmoid(y) if act == "silu" else torch.relu(y) if act == "relu" else y


def _place(c, y, like):
    """Rows y [b][m][n] in the layout of the output buffer (halo and padding channels zero)."""
    b, _, n = y.shape
    h = c["halo"]
    out = torch.zeros((b, c["h"] + 2 * h, c["w"] + 2 * h, like.shape[2]), dtype=torch.float64, device="cuda")
    out[:, h:h + c["h"], h:h + c["w"], :n] = y.reshape(b, c["h"], c["w"], n)
    return out.reshape(like.shape)


def _product(c, x, w, bias, s, n_out):
    """act(x . w^T + bias) (+ res): [b][m][n_out], weight rows past n zero, window by window."""
    n = w.shape[0]
    wt = torch.zeros((x.shape[2], n_out), dtype=torch.float64, device="cuda")
    wt[:w.shape[1], :n] = torch.from_numpy(w).cuda().double().t()
    bt = torch.zeros(n_out, dtype=torch.float64, device="cuda")
    bt[:n] = torch.from_numpy(bias).cuda().double()
    y = torch.stack([_act(xi @ wt + bt, c["act"]) for xi in x])
    return y if s.get("res") is None else y + s["res"].double()


def _s8_rows(x):
    """Rows on the no-dotprod family's int8 grid, dequantised: lo..hi over 254 steps, lo at -127."""
    lo, hi = x.amin(-1, keepdim=True), x.amax(-1, keepdim=True)
    inv = 254.0 / (hi - lo)
    z = -127 - torch.round(lo * inv)
    return (torch.clamp(torch.round(x * inv) + z, -127, 127) - z) / inv


def _s8_weights(n, k):
    """A layer's int8 weights, dequantised [n][k]."""
    w = _weights(n, k)[0].astype(np.float64)
    sw = np.abs(w).max(1, keepdims=True) / 127.0
    return np.clip(s8pack.half_away(w / sw), -127, 127) * sw


def _exact_pw_s8(c, s):
    x = s["x"][:, :, :c["k"]].double()
    if c["gate"]:
        x = x * s["gate"].double()[:, None]
    y = _product(c, _s8_rows(x), _s8_weights(c["n"], c["k"]), _weights(c["n"], c["k"])[1], s, s["W"].Np)
    return _place(c, y, s["out"])


def _exact_pw_f32(c, s):
    x = s["x"][:, :, :s["kp"]].double()
    if c["gate"]:
        x = x * s["gate"].double()[:, None]
    return _place(c, _product(c, x, *_weights(c["n"], c["k"]), s, s["np"]), s["out"])


def _exact_pw_f16(c, s):
    w, b = _weights(c["n"], c["k"])
    x = s["x"].double()
    if c["gate"]:
        x = x * s["gate"].double()[:, None]
    return _place(c, _product(c, x, w.astype(np.float16).astype(np.float32), b, s, s["np"]), s["out"])


def _exact_qpw(c, s):
    n, k = _r(c["n"], 16), c["k"]
    x = s["x"][:, :, :k].double()
    if c["gate"]:
        x = x * s["gate"].double()[:, None]
    lo, hi = x.amin(-1, keepdim=True).clamp(max=0), x.amax(-1, keepdim=True).clamp(min=0)
    inv = 255.0 / (hi - lo)
    zp = torch.round(lo * inv) + 128
    x = (torch.clamp(torch.round(x * inv) - zp, -128, 127) + zp) / inv
    w, b = _weights(n, k)
    sw = np.abs(w).max(1, keepdims=True).astype(np.float64) / 127.0
    return _place(c, _product(c, x, np.clip(np.rint(w / sw), -127, 127) * sw, b, s, n), s["out"])


def _depthwise(c, xp, w, bias):
    """SiLU of the depthwise conv of the zero-haloed xp [b][h+2p][w+2p][c], and its sums over the pixels."""
    ho, wo, pt, pl, dw3 = _dw_geometry(c)
    k, s, h = c["ks"], c["s"], (c["ks"] - 1) // 2
    xp = torch.nn.functional.pad(xp, (0, 0, 0, s + k, 0, s + k))
    y = bias.double().expand(xp.shape[0], ho, wo, c["c"]).clone()
    for i in range(k):
        for j in range(k):
            t, l_ = i - pt + h, j - pl + h
            y += xp[:, t:t + s * (ho - 1) + 1:s, l_:l_ + s * (wo - 1) + 1:s] * w[i * k + j].double()
    y = _act(y, "silu")
    return y, y.sum((1, 2))


def _exact_expand_dw(c, s):
    e = _product(dict(c, act="silu"), _s8_rows(s["x"].double()), _s8_weights(c["c"], c["k"]),
                 _weights(c["c"], c["k"])[1], {}, c["c"])
    h = (c["ks"] - 1) // 2
    xp = torch.nn.functional.pad(e.reshape(c["windows"], c["h"], c["w"], c["c"]), (0, 0, h, h, h, h))
    return _depthwise(c, xp, s["w"], s["bias"])


def _exact_dw(c, s):
    return _depthwise(c, s["x"].double(), s["w"], s["bias"])


def _exact_wino(c, s):
    w, b = _wino_weights(c["c"], c["k"])
    wt = torch.from_numpy(w).cuda().double()
    y = torch.from_numpy(b).cuda().double().expand(c["windows"], c["h"], c["w"], c["k"]).clone()
    x = s["x"].double()
    for i in range(3):
        for j in range(3):
            y += x[:, i:i + c["h"], j:j + c["w"]] @ wt[:, i, j].t().contiguous()
    return _act(y, c["act"])


def _exact_proto(c, s):
    n, k, b = c["classes"] * c["ppc"], c["c"], c["windows"]
    p = torch.from_numpy(_protos(n, k)).cuda()
    x = s["x"].double()
    den = x.square().sum(-1, keepdim=True).sqrt() + 1e-5
    if c["dtype"] == "s8":
        q, sw = s8pack.quant_rows_s8(p.cpu().numpy())
        p = torch.from_numpy(q).cuda().double() * torch.from_numpy(sw).cuda().double()[:, None]
        mx = x.abs().amax(-1, keepdim=True)
        r = x * (127.0 / mx)
        a = torch.sign(r) * torch.floor(r.abs() + 0.5) * mx / (127.0 * den)
    else:
        a = x / den
        p = (p if c["dtype"] == "f32" else p.half()).double()
    colmax = torch.zeros((b, s["np"]), dtype=torch.float64, device="cuda")
    for i in range(b):
        colmax[i, :n] = (a[i] @ p.t()).amax(0)
    logits = (colmax[:, :n].reshape(b, c["classes"], c["ppc"]) * s["cw"].double()).sum(-1) + s["cb"].double()
    return logits, colmax


_PREPARE = dict(net=_prepare_net, pw_s8=_prepare_pw_s8, pw_f32=_prepare_pw_f32, pw_f16=_prepare_pw_f16,
                qpw=_prepare_qpw, expand_dw=_prepare_expand_dw, dw=_prepare_dw, wino=_prepare_wino, proto=_prepare_proto)
_RUN = dict(net=_run_net, pw_s8=_run_pw_s8, pw_f32=_run_pw_f32, pw_f16=_run_pw_f16, qpw=_run_qpw,
            expand_dw=_run_expand_dw, dw=_run_dw, wino=_run_wino, proto=_run_proto)
_EXACT = dict(pw_s8=_exact_pw_s8, pw_f32=_exact_pw_f32, pw_f16=_exact_pw_f16, qpw=_exact_qpw,
              expand_dw=_exact_expand_dw, dw=_exact_dw, wino=_exact_wino, proto=_exact_proto)
