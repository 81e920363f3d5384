"""Performance cases: the work a user of this library has it do, through its public entry points.

Kinds of case (each takes its sizes from the models the library serves):
  engine    one batch through the wd (EVA02-L) tagger engine, host operands in, host scores out
  wd_attn   wd patch embedding and the attention half of a block: LayerNorm, qkv, attention, out-projection + residual
  wd_mlp    the MLP half of a block on residual rows (LayerNorm, fc1 + SwiGLU, fc2 + residual), then the pooled tag head
  px_attn   PixAI (ViTDet-L) patch embedding and the attention half of a block, windowed or global
  px_mlp    the MLP half of a PixAI block
  px_pool   PixAI attention-pool head and tag head
  gemm      the standalone block-scaled E4M3 GEMM, dense or 2:4-sparse weights
  prep      a decoded image to patch operands: alpha over white, pyramid, the full view and crops
A block is cut in two because every re-quantisation to E4M3 multiplies differences of rounding: behind one of them an
output still tells a wrong kernel from another order of summation. Programs that run a fixed sequence of launchers keep
it as a HIP graph, as the engines do.
"""
import ctypes
import os

import numpy as np
import torch

from xtagger_amd import blob
from xtagger_amd import lib as X
from xtagger_amd.engine import Engine

D, T, TP, NH, HD, HID, HIDP, K0, K0P = 1024, 1025, 1088, 16, 64, 2730, 2816, 588, 592
PX_T, PX_LW, PX_HID = 5184, 576, 4736
QSCALE = float(np.log2(np.e)) / 8.0
NT = 10861                       # tags of the wd tagger; 13461: the PixAI tagger and the extended head

DEV = "cuda:0"
U8, F16, F32, F64, I16 = torch.uint8, torch.float16, torch.float32, torch.float64, torch.int16


def listed():
    return [
        # one image tagged interactively: upload, 24 blocks, scores back on the host
        {"name": "engine_b1", "kind": "engine", "nb": 1, "sparse": False},
        # the reference's own batch of 8: bulk tagging through the default engine
        {"name": "engine_b8", "kind": "engine", "nb": 8, "sparse": False},
        # one image through the layer kernels: short grids, launches count
        {"name": "wd_attn_b1", "kind": "wd_attn", "nb": 1, "sparse": False},
        {"name": "wd_mlp_b1", "kind": "wd_mlp", "nb": 1, "sparse": False, "nt": NT},
        # half of a batch of 32 (the throughput setting): the rows each of the engine's two lanes runs
        {"name": "wd_attn_b16", "kind": "wd_attn", "nb": 16, "sparse": False},
        {"name": "wd_mlp_b16", "kind": "wd_mlp", "nb": 16, "sparse": False, "nt": NT},
        # 2:4-sparse weights, half of a batch of 8, with the extended head
        {"name": "wd_mlp_sparse_b4", "kind": "wd_mlp", "nb": 4, "sparse": True, "nt": 13461},
        # PixAI at its default batch of 4: the two images each lane runs, in a windowed block (28 of the 32)
        {"name": "px_window_b2", "kind": "px_attn", "nb": 2, "window": True},
        {"name": "px_mlp_b2", "kind": "px_mlp", "nb": 2, "rs": False},
        # the PixAI head of the two images of a lane
        {"name": "px_pool_b2", "kind": "px_pool", "nb": 2, "nt": 13461},
        # the qkv projection of one image as a plain GEMM
        {"name": "gemm_m1025", "kind": "gemm", "M": 1025, "N": 3072, "K": 1024, "f32": False, "sparse": False},
        # a camera image with its full view and four crops
        {"name": "prep_3072x2048", "kind": "prep", "w": 3072, "h": 2048, "crops": 4},
    ]


def _log(rng, lo, hi):
    return int(round(float(np.exp(rng.uniform(np.log(lo), np.log(hi))))))


def draw(rng):
    kind = rng.choice(["engine", "wd_attn", "wd_attn", "wd_mlp", "wd_mlp", "px_attn", "px_mlp", "px_pool", "gemm", "gemm",
                       "prep"])
    if kind == "engine":
        return {"kind": kind, "nb": _log(rng, 1, 8), "sparse": rng.random() < 0.5, "extra": rng.randrange(0, 2600)}
    if kind == "wd_attn":
        return {"kind": kind, "nb": _log(rng, 1, 32), "sparse": rng.random() < 0.33}
    if kind == "wd_mlp":
        return {"kind": kind, "nb": _log(rng, 1, 32), "sparse": rng.random() < 0.33, "nt": rng.randrange(9000, 13462)}
    if kind == "px_attn":
        return {"kind": kind, "nb": 2 * rng.randrange(1, 5), "window": rng.random() < 0.6}
    if kind == "px_mlp":         # rs: the per-unit multipliers of a calibrated (v3) weight file
        return {"kind": kind, "nb": rng.randrange(1, 9), "rs": rng.random() < 0.5}
    if kind == "px_pool":
        return {"kind": kind, "nb": rng.randrange(1, 9), "nt": rng.randrange(9000, 13462)}
    if kind == "gemm":
        sparse = rng.random() < 0.25
        n = _log(rng, 64, 13461)
        return {"kind": kind, "M": _log(rng, 1, 8200), "N": (n + 15) // 16 * 16 if sparse else n,
                "K": 128 * _log(rng, 1, 37), "f32": rng.random() < 0.5, "sparse": sparse}
    return {"kind": kind, "w": _log(rng, 300, 4000), "h": _log(rng, 300, 4000), "crops": rng.randrange(0, 7)}


# ---- inputs ---------------------------------------------------------------------------------------------------------
class _Gen:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed))

    def n(self, *shape, std=1.0, mean=0.0, dt=F32):
        return torch.randn(*shape, generator=self.g, device=DEV).mul_(std).add_(mean).to(dt)

    def u(self, *shape):
        return torch.rand(*shape, generator=self.g, device=DEV)

    def patches(self, rows):
        """fp16 patch operands [rows][592]: pixels in [-1, 1], a level per patch and channel with detail on top, the
        four pad columns zero"""
        x = torch.zeros(rows, K0P, dtype=F16, device=DEV)
        v = (self.u(rows, 3, 1) * 2 - 1) + 0.25 * torch.randn(rows, 3, 196, generator=self.g, device=DEV)
        x[:, :K0] = v.clamp_(-1, 1).reshape(rows, K0).to(F16)
        return x


def _z(*shape, dt=U8):
    return torch.zeros(*shape, dtype=dt, device=DEV)


def _st():
    return torch.cuda.current_stream().cuda_stream


def _lns(g, w, *names):
    for k in names:
        w[k + "w"], w[k + "b"] = g.n(D, std=0.1, mean=1.0), g.n(D, std=0.02)


def _embed(g, w, tokens):
    w["pe"] = _z(D, K0P, dt=F16)
    w["pe"][:, :K0] = g.n(D, K0, std=0.02, dt=F16)
    w["pos"] = g.n(tokens, D, std=0.02)


def _qkv(g):
    w = g.n(3 * D, D, std=0.02)
    w[:2 * D] *= 2.5             # logits of a few units: attention that prefers some keys
    w[:D] *= QSCALE              # q rows carry log2(e) / 8
    return w.to(F16)


def _wd_attn_tensors(c, seed):
    """fp16 / fp32 tensors as an exporter writes them, and the patches"""
    g = _Gen(seed)
    w = {"in": g.patches(c["nb"] * 1024), "cs": torch.from_numpy(blob.rope_table()).to(DEV)}
    _embed(g, w, T)
    _lns(g, w, "ln")
    w["wqkv"], w["wo"] = _qkv(g), g.n(D, D, std=0.03, dt=F16)
    return w


def _wd_mlp_tensors(c, seed):
    g, nt = _Gen(seed), c["nt"]
    w = {"x": g.n(c["nb"] * T, D, dt=F16)}
    _lns(g, w, "ln", "fn")
    w12 = _z(2, 2736, D, dt=F16)
    w12[:, :HID] = g.n(2, HID, D, std=0.02, dt=F16)
    w["w12"] = w12.reshape(2, 171, 16, D).transpose(0, 1).reshape(2 * 2736, D).contiguous()
    mw, mb, w2 = _z(2736, dt=F32), _z(2736, dt=F32), _z(D, 2736, dt=F16)
    mw[:HID], mb[:HID], w2[:, :HID] = g.n(HID, std=0.1, mean=1.0), g.n(HID, std=0.02), g.n(D, HID, std=0.02, dt=F16)
    w["mw"], w["mb"], w["w2"] = mw, mb, w2
    w["hw"], w["hb"] = g.n(nt, D, std=0.05, dt=F16), g.n(nt, std=0.1)
    return w


def _px_attn_tensors(c, seed):
    g = _Gen(seed)
    w = {"in": g.patches(c["nb"] * PX_T)}
    _embed(g, w, PX_T)
    _lns(g, w, "lp", "ln")
    a = g.u(PX_LW if c["window"] else PX_T, 32) * 6.2831853
    w["cs"] = torch.stack([torch.cos(a), torch.sin(a)], -1).contiguous()
    w["wqkv"], w["bqkv"] = _qkv(g), g.n(3 * D, std=0.05)
    w["bqkv"][:D] *= QSCALE
    w["wo"], w["bo"] = g.n(D, D, std=0.03, dt=F16), g.n(D, std=0.05)
    return w


def _px_mlp_tensors(c, seed):
    g = _Gen(seed)
    w = {"x": g.n(c["nb"] * PX_T, D, dt=F16)}
    _lns(g, w, "ln")
    w["w1"], w["b1"] = g.n(PX_HID, D, std=0.02, dt=F16), g.n(PX_HID, std=0.05)
    w["w2"], w["b2"] = g.n(D, PX_HID, std=0.02, dt=F16), g.n(D, std=0.05)
    w["rs"] = torch.exp2(g.u(PX_HID) * 2 - 1) if c["rs"] else None
    return w


def _pool_tensors(c, seed):
    g = _Gen(seed)
    return {"x": g.n(c["nb"] * PX_T, D, std=1.5, mean=0.2, dt=F16), "w": g.n(D, std=0.1, mean=1.0),
            "b": g.n(D, std=0.1), "hpos": g.n(PX_T, D, std=0.2, dt=F16), "U": g.n(16, D, std=0.05),
            "wv": g.n(D, D, std=0.03, dt=F16), "hw": g.n(c["nt"], D, std=0.05, dt=F16), "hb": g.n(c["nt"], std=0.1)}


def _gemm_tensors(c, seed):
    g = _Gen(seed)
    return g.n(c["M"], c["K"]), g.n(c["N"], c["K"], std=0.02)


def _prep_inputs(c, seed):
    """an RGBA image (smooth content, grain, a translucent corner) and the rects of its views, the full one first"""
    g, w, h = _Gen(seed), c["w"], c["h"]
    low = torch.nn.functional.interpolate(g.u(1, 3, 9, 13) * 255, size=(h, w), mode="bilinear")[0]
    rgb = (low + 8 * torch.randn(3, h, w, generator=g.g, device=DEV)).clamp_(0, 255)
    img = torch.full((h, w, 4), 255, dtype=U8, device=DEV)
    img[..., :3] = rgb.permute(1, 2, 0).to(U8)
    img[: h // 4, : w // 4, 3] = (g.u(h // 4, w // 4) * 256).to(U8)
    r, rects = np.random.default_rng(int(seed)), [(0, 0, w, h)]
    for _ in range(c["crops"]):
        cw = int(r.integers(min(w, h) // 4, min(w, h) + 1))
        ch = int(np.clip(cw * r.uniform(0.6, 1.6), 64, h))
        rects.append((int(r.integers(0, w - cw + 1)), int(r.integers(0, h - ch + 1)), cw, ch))
    return img, rects


# ---- programs -------------------------------------------------------------------------------------------------------
def _pack(w16, k_in, n_out, k_out, perm=0, col=None):
    """fp16 weight rows to E4M3 with 128x128 scales"""
    n_in, ldw = w16.shape
    q, s = _z(n_out, k_out), _z(n_out // 128, k_out // 128, dt=F32)
    scratch = torch.empty(n_out * k_out, dtype=F32, device=DEV)
    X.check(X.lib.eva_k_prep_w(X.ptr(w16), ldw, n_in, k_in, n_out, k_out, perm, X.ptr(col), X.ptr(scratch), X.ptr(q),
                               X.ptr(s), _st()), "eva_k_prep_w")
    return q, s


def _pack24(q):
    n, k = q.shape
    v, x = _z(n // 16, k // 128, 64, 16), _z(n // 16, k // 128, 64, dt=torch.int32)
    X.check(X.lib.eva_k_prune24(X.ptr(q), n, k, _st()), "eva_k_prune24")
    X.check(X.lib.eva_k_pack24(X.ptr(q), n, k, X.ptr(v), X.ptr(x), None, _st()), "eva_k_pack24")
    return v, x


def _pack_head(hw, nt):
    ldh = (nt + 63) // 64 * 64
    q, s = _z(nt, D), _z(8, ldh, dt=F32)
    X.check(X.lib.eva_k_quant_act(X.ptr(hw), 2, D, nt, D, X.ptr(q), D, X.ptr(s), ldh, _st()), "eva_k_quant_act")
    return q, s, ldh


def _graph(calls):
    """the launches of calls(stream) as a HIP graph, after one direct pass"""
    calls(_st())
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        calls(_st())
    return g


def _weights(name, qs, sparse):
    """the wd launcher `name` and its weight arguments"""
    q, sc = qs
    if sparse:
        v, x = _pack24(q)
        return getattr(X.lib, f"eva_k_{name}_sp"), (X.ptr(v), X.ptr(x), X.ptr(sc)), (v, x, sc)
    return getattr(X.lib, f"eva_k_{name}"), (X.ptr(q), X.ptr(sc)), (q, sc)


def _rows(M):
    """scale-plane stride, residual rows, and packed activations with their scales"""
    lds = (M + 255) // 256 * 256
    return lds, _z(lds, D, dt=F16), _z(lds, D), _z(8, lds, dt=F32)


def _wd_attn_program(c, w):
    L, P, nb = X.lib, X.ptr, c["nb"]
    M = nb * T
    qkv, wqkv, k1 = _weights("qkv", _pack(w["wqkv"], D, 3 * D, D, perm=1), c["sparse"])
    oproj, wo, k2 = _weights("oproj", _pack(w["wo"], D, D, D), c["sparse"])
    lds, x, h8, sh = _rows(M)
    qa, ka, va = _z(nb, NH, TP, HD, dt=I16), _z(nb, NH, TP, HD, dt=I16), _z(nb, NH, HD, TP, dt=I16)

    def calls(st):
        rc = L.eva_k_pe(P(w["in"]), P(w["pe"]), P(w["pos"]), P(x), nb, st)
        rc |= L.eva_k_ln(P(x), P(w["lnw"]), P(w["lnb"]), P(h8), P(sh), M, lds, st)
        rc |= qkv(P(h8), P(sh), lds, *wqkv, P(w["cs"]), P(qa), P(ka), P(va), M, st)
        rc |= L.eva_k_flash(P(qa), P(ka), P(va), P(h8), P(sh), lds, nb, None, st)
        rc |= oproj(P(h8), P(sh), lds, *wo, P(x), M, st)
        X.check(rc, "wd attention half")

    return {"graph": _graph(calls), "out": {"x": x[:M], "k": ka.view(torch.bfloat16)}, "keep": [w, k1, k2, h8, sh, qa, va]}


def _wd_mlp_program(c, w):
    L, P, nb, nt = X.lib, X.ptr, c["nb"], c["nt"]
    M, sp = nb * T, c["sparse"]
    fc1, w1, k1 = _weights("fc1", _pack(w["w12"], D, 2 * HIDP, D), sp)
    q2 = _pack(w["w2"], HID, D, HIDP, col=w["mw"])
    fc2, w2, k2 = _weights("fc2", q2, sp)
    cn, dn = _z(D, dt=F32), _z(D, dt=F32)
    X.check(L.eva_k_fold_cd(P(q2[0]), P(q2[1]), P(w["w2"]), 2736, P(w["mb"]), P(cn), P(dn), _st()), "eva_k_fold_cd")
    hq, hs, ldh = _pack_head(w["hw"], nt)
    lds, x, h8, sh = _rows(M)
    m8, sm, stat = _z(lds, HIDP), _z(22, lds, dt=F32), _z(22, lds, 2, dt=F32)
    pool, pn, pq, ps = _z(nb, D, dt=F32), _z(nb, D, dt=F16), _z(nb, D), _z(8, nb, dt=F32)
    out = _z(nb, nt, dt=F32)

    def calls(st):
        x[:M].copy_(w["x"])      # fc2 updates the rows in place
        rc = L.eva_k_ln(P(x), P(w["lnw"]), P(w["lnb"]), P(h8), P(sh), M, lds, st)
        rc |= fc1(P(h8), P(sh), lds, *w1, P(m8), P(sm), P(stat), M, st)
        rc |= fc2(P(m8), P(sm), lds, *w2, P(stat), P(cn), P(dn), P(x), M, st)
        rc |= L.eva_k_pool(P(x), P(pool), nb, st)
        rc |= L.eva_k_lnh(P(pool), P(w["fnw"]), P(w["fnb"]), P(pn), P(pq), P(ps), nb, nb, st)
        rc |= L.eva_k_head(P(pq), P(ps), nb, P(hq), P(hs), ldh, P(w["hb"]), P(out), nb, nt, st)
        X.check(rc, "wd MLP half")

    return {"graph": _graph(calls), "out": {"x": x[:M], "scores": out},
            "keep": [w, k1, k2, q2, cn, dn, hq, hs, h8, sh, m8, sm, stat, pool, pn, pq, ps]}


def _px_attn_program(c, w):
    L, P, rows = X.lib, X.ptr, c["nb"] * PX_T
    n = PX_LW if c["window"] else PX_T
    S = rows // n
    qw, qo = _pack(w["wqkv"], D, 3 * D, D, perm=1), _pack(w["wo"], D, D, D)
    lds, x, h8, sh = _rows(rows)
    qa, ka, va = _z(S, NH, n, HD, dt=I16), _z(S, NH, n, HD, dt=I16), _z(S, NH, HD, n, dt=I16)

    def calls(st):
        rc = L.px_k_pe(P(w["in"]), P(w["pe"]), P(x), rows, st)
        rc |= L.px_k_pembed(P(x), P(w["pos"]), PX_T, P(w["lpw"]), P(w["lpb"]), rows, st)
        rc |= L.eva_k_ln(P(x), P(w["lnw"]), P(w["lnb"]), P(h8), P(sh), rows, lds, st)
        rc |= L.px_k_qkv(P(h8), P(sh), lds, P(qw[0]), P(qw[1]), P(w["bqkv"]), P(w["cs"]), n, P(qa), P(ka), P(va), rows, st)
        rc |= L.eva_k_flash_seq(P(qa), P(ka), P(va), P(h8), P(sh), lds, S, n, n, None, st)
        rc |= L.px_k_proj(P(h8), P(sh), lds, P(qo[0]), P(qo[1]), P(w["bo"]), P(x), rows, st)
        X.check(rc, "px attention half")

    return {"graph": _graph(calls), "out": {"x": x[:rows], "k": ka.view(torch.bfloat16)}, "keep": [w, qw, qo, h8, sh, qa, va]}


def _px_mlp_program(c, w):
    L, P, rows = X.lib, X.ptr, c["nb"] * PX_T
    q1, q2 = _pack(w["w1"], D, PX_HID, D), _pack(w["w2"], PX_HID, D, PX_HID)
    lds, x, h8, sh = _rows(rows)
    m8, sm = _z(lds, PX_HID), _z(PX_HID // 128, lds, dt=F32)

    def calls(st):
        x[:rows].copy_(w["x"])   # fc2 updates the rows in place
        rc = L.eva_k_ln(P(x), P(w["lnw"]), P(w["lnb"]), P(h8), P(sh), rows, lds, st)
        rc |= L.px_k_fc1(P(h8), P(sh), lds, P(q1[0]), P(q1[1]), P(w["b1"]), P(w["rs"]), P(m8), P(sm), rows, st)
        rc |= L.px_k_fc2(P(m8), P(sm), lds, P(q2[0]), P(q2[1]), P(w["b2"]), P(x), rows, st)
        X.check(rc, "px MLP half")

    return {"graph": _graph(calls), "out": {"x": x[:rows]}, "keep": [w, q1, q2, h8, sh, m8, sm]}


def _pool_program(c, w):
    L, P, nb, nt = X.lib, X.ptr, c["nb"], c["nt"]
    rows, nw = nb * PX_T, PX_T // 288
    hq, hs, ldh = _pack_head(w["hw"], nt)
    y, s, stat = _z(rows, D, dt=F16), _z(rows, 16, dt=F32), _z(nb, PX_T // 576, 16, 2, dt=F32)
    part, o = _z(nb, nw, 16, D, dt=F32), _z(nb, D, dt=F32)
    oq, os_, out = _z(nb, D), _z(8, nb, dt=F32), _z(nb, nt, dt=F32)

    def calls(st):
        rc = L.px_k_hln(P(w["x"]), P(w["w"]), P(w["b"]), P(w["hpos"]), PX_T, P(w["U"]), P(y), P(s), rows, st)
        rc |= L.px_k_hstat(P(s), P(stat), nb, PX_T, st)
        rc |= L.px_k_hpool(P(s), P(stat), P(y), None, P(part), nb, PX_T, st)
        rc |= L.px_k_hproj(P(part), nw, P(w["wv"]), P(o), nb, st)
        rc |= L.eva_k_quant_act(P(o), 1, D, nb, D, P(oq), D, P(os_), nb, st)
        rc |= L.eva_k_head(P(oq), P(os_), nb, P(hq), P(hs), ldh, P(w["hb"]), P(out), nb, nt, st)
        X.check(rc, "px pool head")

    return {"graph": _graph(calls), "out": {"y": y, "pooled": o, "scores": out},
            "keep": [w, hq, hs, s, stat, part, oq, os_]}


_file = {}                       # the wd model's weight file, in memory, made once per process


def _weight_file():
    if "path" not in _file:
        _file["path"] = f"/proc/{os.getpid()}/fd/{os.memfd_create('eva02')}"
        # a well-conditioned model: residual branches scaled as a trained network's layer scale keeps them
        blob.write_v2(_file["path"], blob.synth_model(seed=0, nt=NT, layer_scale=0.01, head_std=0.002))
    return _file["path"]


_PROGRAMS = {"wd_attn": (_wd_attn_tensors, _wd_attn_program), "wd_mlp": (_wd_mlp_tensors, _wd_mlp_program),
             "px_attn": (_px_attn_tensors, _px_attn_program), "px_mlp": (_px_mlp_tensors, _px_mlp_program),
             "px_pool": (_pool_tensors, _pool_program)}


def prepare(case, seed):
    c, kind = case, case["kind"]
    if kind == "engine":
        e = Engine(_weight_file(), nb=c["nb"], extra=c.get("extra", 0), sparse=c["sparse"])
        e.ready()
        return {"kind": kind, "engine": e, "in": blob.synth_smooth_inputs(c["nb"], seed=int(seed))}
    if kind in _PROGRAMS:
        tensors, program = _PROGRAMS[kind]
        s = program(c, tensors(c, seed))
    elif kind == "gemm":
        M, N, K = c["M"], c["N"], c["K"]
        a, w = _gemm_tensors(c, seed)
        Np = (N + 127) // 128 * 128
        s = {"c": c, "qa": _z(M, K), "sa": _z(K // 128, M, dt=F32), "qw": _z(Np, K), "sw": _z(Np // 128, K // 128, dt=F32),
             "y": _z(M, N, dt=F32 if c["f32"] else torch.bfloat16)}
        X.check(X.lib.eva_k_quant_act(X.ptr(a), 1, K, M, K, X.ptr(s["qa"]), K, X.ptr(s["sa"]), M, _st()), "quant_act")
        X.check(X.lib.eva_k_quant_w(X.ptr(w), N, K, X.ptr(s["qw"]), X.ptr(s["sw"]), _st()), "quant_w")
        if c["sparse"]:
            s["v"], s["x"] = _pack24(s["qw"])
        torch.cuda.synchronize()
    else:
        img, rects = _prep_inputs(c, seed)
        nbl, nbs = X.lib.eva_img_pyramid_bytes(c["w"], c["h"], 448), X.lib.eva_img_prep_bytes(448, 4 * 448 - 1)
        s = {"img": img, "rects": rects, "lv": _z(max(nbl, 256)), "nbl": nbl, "scratch": _z(nbs), "nbs": nbs,
             "out": _z(len(rects), 1024, K0P, dt=F16)}
    s["kind"] = kind
    return s


def run(s):
    kind = s["kind"]
    if kind == "engine":
        n = s["engine"].submit(0, s["in"])
        return s["engine"].wait(0, n)
    if "graph" in s:
        s["graph"].replay()
        return s["out"]
    L, P, st = X.lib, X.ptr, _st()
    if kind == "gemm":
        c = s["c"]
        M, N, K, f32 = c["M"], c["N"], c["K"], int(c["f32"])
        if c["sparse"]:
            rc = L.eva_k_gemm_sp(P(s["qa"]), K, P(s["sa"]), M, P(s["v"]), P(s["x"]), P(s["sw"]), M, N, K, P(s["y"]), N,
                                 f32, st)
        else:
            rc = L.eva_k_gemm(P(s["qa"]), K, P(s["sa"]), M, P(s["qw"]), P(s["sw"]), M, N, K, P(s["y"]), N, f32, st)
        X.check(rc, "gemm")
        return s["y"]
    img = s["img"]
    h, w = img.shape[:2]
    p = X.EvaPyr()
    p.lv[0], p.ls[0], p.lw[0], p.lh[0] = img.data_ptr(), w * 4, w, h
    X.check(L.eva_img_over_white(P(img), w * 4, w, h, st), "eva_img_over_white")
    X.check(L.eva_img_pyramid(ctypes.byref(p), P(s["lv"]), s["nbl"], 448, st), "eva_img_pyramid")
    for k, r in enumerate(s["rects"]):
        X.check(L.eva_img_prep(ctypes.byref(p), *r, 448, P(s["scratch"]), s["nbs"],
                               ctypes.c_void_p(s["out"].data_ptr() + k * 1024 * K0P * 2), st), "eva_img_prep")
    return s["out"]


# ---- work and tolerances --------------------------------------------------------------------------------------------
def work(case):
    c, kind = case, case["kind"]
    nb, sp = c.get("nb", 0), 0.625 if c.get("sparse") else 1.0    # 2:4 weights: half the bytes and an eighth in indices
    attn = lambda rows, n: 2.0 * rows * D * 4 * D + 4.0 * rows * n * D
    if kind == "engine":
        nt, M = NT + c.get("extra", 0), nb * T
        return {"bytes": 24 * D * (4 * D + 3 * HID) * sp + nt * D + nb * (1024 * K0P * 2 + nt * 4) + D * K0P * 2 + T * D * 4,
                "flops": 24 * (attn(M, T) + 6.0 * M * D * HID) + 2.0 * nb * (1024 * D * K0 + nt * D)}
    if kind == "wd_attn":
        M = nb * T
        return {"bytes": 4 * D * D * sp + D * K0P * 2 + T * D * 4 + nb * 1024 * K0P * 2 + M * D * 4,
                "flops": attn(M, T) + 2.0 * nb * 1024 * D * K0}
    if kind == "wd_mlp":
        M, nt = nb * T, c["nt"]
        return {"bytes": 3 * D * HID * sp + nt * D + M * D * 4 + nb * nt * 4, "flops": 6.0 * M * D * HID + 2.0 * nb * nt * D}
    if kind == "px_attn":
        rows, n = nb * PX_T, PX_LW if c["window"] else PX_T
        return {"bytes": 4 * D * D + D * K0P * 2 + PX_T * D * 4 + rows * (K0P * 2 + D * 4),
                "flops": attn(rows, n) + 2.0 * rows * D * K0}
    if kind == "px_mlp":
        return {"bytes": 2 * D * PX_HID + nb * PX_T * D * 4, "flops": 4.0 * nb * PX_T * D * PX_HID}
    if kind == "px_pool":
        nb, nt = c["nb"], c["nt"]
        return {"bytes": nb * (PX_T * D * 4 + D * 4 + nt * 4) + PX_T * D * 2 + 16 * D * 4 + D * D * 2 + nt * D,
                "flops": 2.0 * nb * (2 * PX_T * D * 16 + D * D + nt * D)}
    if kind == "gemm":
        M, N, K = c["M"], c["N"], c["K"]
        return {"bytes": M * K + N * K * (0.625 if c["sparse"] else 1.0) + M * N * (4 if c["f32"] else 2),
                "flops": 2.0 * M * N * K}
    px = c["w"] * c["h"]
    return {"bytes": 8.0 * px + (1 + c["crops"]) * 1024 * K0P * 2, "flops": 0.0}


def tolerance(case):
    kind = case["kind"]
    if kind == "prep":
        return "exact"           # the operand is specified bit for bit
    if kind == "gemm":
        return {"rel": 5e-5} if case["f32"] else {"rel": 5e-3}
    if kind == "engine":
        return {"rel": 4e-3}     # 24 re-quantised blocks: one changed rounding travels to the scores
    if kind == "px_pool":
        return {"rel": 1e-3}
    return {"rel": 1e-2}         # E4M3 activations re-quantised inside, bf16 attention operands


# ---- 64-bit values ----------------------------------------------------------------------------------------------------
def _q_rows(x):
    """E4M3 rounding of activations in 1x128 blocks, scale amax / 448 in fp32"""
    b = x.reshape(x.shape[0], -1, 128)
    m = b.abs().amax(-1, keepdim=True)
    s = torch.where(m > 0, (m / 448).to(F32).to(F64), torch.ones_like(m))
    return ((b / s).clamp(-448, 448).to(F32).to(torch.float8_e4m3fn).to(F64) * s).reshape(x.shape)


def _q_weight(w):
    """E4M3 rounding of weights in 128x128 blocks (rows and columns padded with zeros): the codes and the scales"""
    n, k = w.shape
    p = torch.zeros((n + 127) // 128 * 128, (k + 127) // 128 * 128, dtype=F64, device=w.device)
    p[:n, :k] = w
    b = p.reshape(p.shape[0] // 128, 128, -1, 128)
    m = b.abs().amax((1, 3), keepdim=True)
    s = torch.where(m > 0, (m / 448).to(F32).to(F64), torch.ones_like(m))
    return (b / s).clamp(-448, 448).to(F32).to(torch.float8_e4m3fn).to(F64), s


def _deq(qs, n, k):
    q, s = qs
    return (q * s).reshape(q.shape[0] * 128, -1)[:n, :k]


def _prune(qs):
    """2:4: the two smallest magnitudes of every four consecutive k set to zero, ties dropping the lower k first"""
    q, s = qs
    g = q.reshape(*q.shape[:-1], 32, 4)
    drop = torch.argsort(g.abs(), dim=-1, stable=True)[..., :2]
    return g.scatter(-1, drop, 0.0).reshape(q.shape), s


def _w64(w, sparse=False):
    qs = _q_weight(w.to(F64))
    return _deq(_prune(qs) if sparse else qs, *w.shape)


def _ln64(x, w, b, eps):
    m = x.mean(-1, keepdim=True)
    v = ((x - m) ** 2).mean(-1, keepdim=True)
    return (x - m) / torch.sqrt(v + eps) * w.to(F64) + b.to(F64)


def _rope64(y, cs):
    """y [S][t][16][64], cs [t][32][2]: pairs (2i, 2i + 1) rotated"""
    c, s = cs[:, None, :, 0].to(F64), cs[:, None, :, 1].to(F64)
    a, b = y[..., 0::2], y[..., 1::2]
    return torch.stack([a * c - b * s, b * c + a * s], -1).reshape(y.shape)


def _attn64(q, k, v):
    """[S][t][16][64], logits in units of log 2 -> [S t][1024]"""
    bf = lambda t: t.to(F32).to(torch.bfloat16).to(F64)
    q, k, v = bf(q), bf(k), bf(v)
    out = torch.empty_like(q)
    for s in range(q.shape[0]):
        for h in range(NH):
            p = q[s, :, h] @ k[s, :, h].T
            p = torch.exp2(p - p.amax(-1, keepdim=True))
            out[s, :, h] = (p @ v[s, :, h]) / p.sum(-1, keepdim=True)
    return out.reshape(-1, D)


def _half(x):
    return x.to(F32).to(F16).to(F64)


def _pad_rows(k, tp):
    """[S][t][16][64] -> [S][16][tp][64]"""
    out = torch.zeros(k.shape[0], NH, tp, HD, dtype=F64, device=k.device)
    out[:, :, :k.shape[1]] = k.transpose(1, 2)
    return out


def _exact_wd_attn(c, seed):
    w, nb, sp = _wd_attn_tensors(c, seed), c["nb"], c["sparse"]
    x = torch.empty(nb, T, D, dtype=F64, device=DEV)
    x[:, 1:] = (w["in"].to(F64) @ w["pe"].to(F64).T).reshape(nb, 1024, D) + w["pos"][1:].to(F64)
    x[:, 0] = w["pos"][0].to(F64)
    x = _half(x).reshape(-1, D)
    y = (_q_rows(_ln64(x, w["lnw"], w["lnb"], 1e-6)) @ _w64(w["wqkv"], sp).T).reshape(nb, T, 3, NH, HD)
    q, k, v = y[:, :, 0].clone(), y[:, :, 1].clone(), y[:, :, 2]
    q[:, 1:], k[:, 1:] = _rope64(q[:, 1:], w["cs"]), _rope64(k[:, 1:], w["cs"])
    x = x + _q_rows(_attn64(q, k, v)) @ _w64(w["wo"], sp).T
    return {"x": x, "k": _pad_rows(k, TP)}


def _exact_wd_mlp(c, seed):
    w, nb, sp = _wd_mlp_tensors(c, seed), c["nb"], c["sparse"]
    x = w["x"].to(F64)
    y = _q_rows(_ln64(x, w["lnw"], w["lnb"], 1e-6)) @ _w64(w["w12"], sp).T
    y = y.reshape(-1, 171, 2, 16)
    h = (torch.nn.functional.silu(y[:, :, 0]) * y[:, :, 1]).reshape(-1, 2736)[:, :HID]
    mean = h.mean(-1, keepdim=True)
    rstd = 1 / torch.sqrt((h * h).mean(-1, keepdim=True) - mean * mean + 1e-6)
    hp = torch.zeros(h.shape[0], HIDP, dtype=F64, device=DEV)
    hp[:, :HID] = h
    w2 = torch.zeros(D, HIDP, dtype=F64, device=DEV)
    w2[:, :HID] = (w["w2"][:, :HID].to(F32) * w["mw"][:HID]).to(F64)
    w2 = _w64(w2, sp)
    x = x + rstd * (_q_rows(hp) @ w2.T - mean * w2.sum(1)) + w["w2"].to(F64) @ w["mb"].to(F64)
    p = _half(_ln64(_half(x).reshape(nb, T, D)[:, 1:].mean(1), w["fnw"], w["fnb"], 1e-6))
    z = _q_rows(p) @ _q_rows(w["hw"].to(F64)).T + w["hb"].to(F64)
    return {"x": x, "scores": torch.sigmoid(z)}


def _exact_px_attn(c, seed):
    w, nb = _px_attn_tensors(c, seed), c["nb"]
    n = PX_LW if c["window"] else PX_T
    x = _half(w["in"].to(F64) @ w["pe"].to(F64).T).reshape(nb, PX_T, D) + w["pos"].to(F64)
    x = _half(_ln64(x, w["lpw"], w["lpb"], 1e-5)).reshape(-1, D)
    y = _q_rows(_ln64(x, w["lnw"], w["lnb"], 1e-6)) @ _w64(w["wqkv"]).T + w["bqkv"].to(F64)
    y = y.reshape(-1, n, 3, NH, HD)
    k = _rope64(y[:, :, 1], w["cs"])
    o = _attn64(_rope64(y[:, :, 0], w["cs"]), k, y[:, :, 2])
    return {"x": x + _q_rows(o) @ _w64(w["wo"]).T + w["bo"].to(F64), "k": _pad_rows(k, n)}


def _exact_px_mlp(c, seed):
    w = _px_mlp_tensors(c, seed)
    x = w["x"].to(F64)
    h = _q_rows(_ln64(x, w["lnw"], w["lnb"], 1e-6)) @ _w64(w["w1"]).T + w["b1"].to(F64)
    h = h * 0.5 * torch.erfc(-h / 2.0 ** 0.5)
    if c["rs"]:
        h = h * w["rs"].to(F64)
    return {"x": x + _q_rows(h) @ _w64(w["w2"]).T + w["b2"].to(F64)}


def _exact_pool(c, seed):
    w, nb = _pool_tensors(c, seed), c["nb"]
    y = _ln64(w["x"].to(F64), w["w"], w["b"], 1e-5).reshape(nb, PX_T, D) + w["hpos"].to(F64)
    y = _half(y)
    s = y @ w["U"].to(F64).T
    p = torch.exp2(s - s.amax(1, keepdim=True))
    p = p / p.sum(1, keepdim=True)
    pooled = torch.stack([p[b].T @ y[b] for b in range(nb)])                       # [nb][16][1024]
    wv = w["wv"].to(F64).reshape(NH, HD, D)
    o = _half(torch.stack([(wv * pooled[b][:, None, :]).sum(-1).reshape(-1) for b in range(nb)]))
    z = _q_rows(o) @ _q_rows(w["hw"].to(F64)).T + w["hb"].to(F64)
    return {"y": y.reshape(-1, D), "pooled": o, "scores": torch.sigmoid(z)}


def _axis64(S, side, off, length):
    """bicubic (Keys, a = -1/2) resampling of `length` samples centred on a white line of `side`: weights [S][length]
    and the share of white per output"""
    scale = side / S
    fs = max(scale, 1.0)
    pos = np.arange(side)
    c = (np.arange(S)[:, None] + 0.5) * scale
    x = np.abs((pos[None, :] - c + 0.5) / fs)
    w = np.where(x < 1, (1.5 * x - 2.5) * x * x + 1, np.where(x < 2, ((-0.5 * x + 2.5) * x - 4) * x + 2, 0.0))
    w /= w.sum(1, keepdims=True)
    inside = w[:, off:off + length]
    return torch.from_numpy(inside.copy()).to(DEV), torch.from_numpy(1 - inside.sum(1)).to(DEV)


def _exact_prep(c, seed):
    img, rects = _prep_inputs(c, seed)
    S, v = 448, img.to(torch.int32)
    t = v[..., :3] * v[..., 3:] + 255 * (255 - v[..., 3:])
    lv = [(t + 128 + ((t + 128) >> 8)) >> 8]
    while max(lv[-1].shape[:2]) >> 1 >= 2 * S and min(lv[-1].shape[:2]) >= 2 and len(lv) < 12:
        a = lv[-1][: lv[-1].shape[0] // 2 * 2, : lv[-1].shape[1] // 2 * 2]
        a = (a[0::2] + a[1::2] + 1) >> 1
        lv.append((a[:, 0::2] + a[:, 1::2]) >> 1)
    out = torch.zeros(len(rects), 1024, K0P, dtype=F64, device=DEV)
    for k, (x0, y0, cw, ch) in enumerate(rects):
        n = 0
        while n + 1 < len(lv) and max(cw, ch) >> (n + 1) >= 2 * S:
            n += 1
        h, w = lv[n].shape[:2]
        x1, y1 = min((x0 + cw) >> n, w), min((y0 + ch) >> n, h)
        xa, ya = min(x0 >> n, w - 1), min(y0 >> n, h - 1)
        r = lv[n][ya:max(y1, ya + 1), xa:max(x1, xa + 1)].to(F64)
        h, w = r.shape[:2]
        side = max(h, w)
        wy, ky = _axis64(S, side, (side - h) >> 1, h)
        wx, kx = _axis64(S, side, (side - w) >> 1, w)
        u = torch.stack([(wy @ r[..., 2 - j] + 255 * ky[:, None]) @ wx.T + 255 * kx for j in range(3)])
        u = (u / 127.5 - 1).clamp(-1, 1)
        out[k, :, :K0] = u.reshape(3, 32, 14, 32, 14).permute(1, 3, 0, 2, 4).reshape(1024, K0)
    return out


_EXACT = {"wd_attn": _exact_wd_attn, "wd_mlp": _exact_wd_mlp, "px_attn": _exact_px_attn, "px_mlp": _exact_px_mlp,
          "px_pool": _exact_pool, "prep": _exact_prep}


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "engine":
        return None              # 24 re-quantised blocks: 64-bit sums take other roundings from block to block
    if kind in _EXACT:
        return _EXACT[kind](c, seed)
    if kind == "gemm":
        a, w = _gemm_tensors(c, seed)
        qs = _q_weight(w.to(F64))
        return _q_rows(a.to(F64)) @ _deq(_prune(qs) if c["sparse"] else qs, *w.shape).T
    raise ValueError(kind)
