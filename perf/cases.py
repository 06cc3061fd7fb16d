"""The work whose time counts: the calls that a user of this framework makes, on seeded synthetic data.

Sizes are those of the repository's own geometries: the 5120-wide model (17408 intermediate, GDN 16/48 heads of
128, 62080 vocabulary) with either attention geometry (32 query / 8 kv heads of 128; the reference checkpoint's
24 / 4 heads of 256 with 64 rotary dims), and the tiny one (1024 wide). Kernel-tier cases chain the entry points
as a program on them does, on the null stream; engine cases run a 4-layer slice (one attention period: three GDN
layers and an attention layer, the MTP layer and the full vocabulary head) whose context a program keeps between
requests.
"""
import ctypes
import importlib.util
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_LIB = os.path.join(_ROOT, "qwen3.8-27b-mi50-cpp-engine_amd", "q27x.py")


def _load():
    if "q27x" not in sys.modules:
        spec = importlib.util.spec_from_file_location("q27x", _LIB)
        mod = importlib.util.module_from_spec(spec)
        sys.modules["q27x"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["q27x"]


HIDDEN, INTER, VOCAB = 5120, 17408, 62080
# (query heads, kv heads, head dim, rotary dims)
GEOMS = {"base": (32, 8, 128, 32), "trunk": (24, 4, 256, 64), "tiny": (4, 1, 128, 32)}
EPS = 1e-6


def listed():
    return [
        # the smallest call: the tiny geometry's out_proj on one row (quantize + project + residual), launch latency
        {"name": "proj_tiny", "kind": "proj", "rows": 1024, "K": 768, "nr": 1, "bf16": True, "res": "bf16"},
        # an ordinary verify projection: down of K=2 speculation (3 rows)
        {"name": "proj_down", "kind": "proj", "rows": HIDDEN, "K": INTER, "nr": 3, "bf16": False, "res": "bf16"},
        # a whole MLP block on the most rows a verify has (K=7): norm, gate, up, SwiGLU, down + residual
        {"name": "mlp_8", "kind": "mlp", "hidden": HIDDEN, "inter": INTER, "nr": 8},
        # one GDN layer's recurrence: commit 2 accepted rows, verify 3 new ones
        {"name": "gdn_3", "kind": "gdn", "kh": 16, "vh": 48, "nr": 3, "npend": 2},
        # one attention layer (prep + attention) at a short context, the 128-wide heads
        {"name": "attn_base_1k", "kind": "attn", "geom": "base", "pos0": 1101, "nr": 3, "kv_group": 32},
        # the reference checkpoint's heads at a long context, 8 rows
        {"name": "attn_trunk_16k", "kind": "attn", "geom": "trunk", "pos0": 16003, "nr": 8, "kv_group": 32},
        # the vocabulary head of a K=2 verify: logits and their argmax
        {"name": "head_3", "kind": "head", "rows": VOCAB, "K": HIDDEN, "nr": 3},
        # ingest GEMM at its largest (the reference's default arm: one group over K)
        {"name": "gemm_4096", "kind": "gemm", "M": 4096, "N": INTER, "K": HIDDEN, "gs": 0, "res": False},
        # ingest GEMM of a short, ragged prompt, 1024-column groups, residual
        {"name": "gemm_77", "kind": "gemm", "M": 77, "N": HIDDEN, "K": INTER, "gs": 1024, "res": True},
        # loading one matrix: per-64 mirror of the fp32 weights, then the ingest GEMM's representation
        {"name": "load_qkvz", "kind": "load", "rows": 16384, "K": HIDDEN, "gs": 0},
        # a whole prompt ingest on the reference checkpoint's attention geometry
        {"name": "prefill_trunk", "kind": "prefill", "geom": "trunk", "n": 3000, "gs": 0},
        # a whole short request: prompt ingest, then speculative decode with K=2
        {"name": "request_base", "kind": "request", "geom": "base", "n": 203, "gen": 24, "K": 2},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng):
    """An input width that the projections take: up to 2048 or 3136 to 6144, a multiple of 64."""
    return 64 * (_log(rng, 8, 32) if rng.random() < 0.5 else _log(rng, 49, 96))


def draw(rng):
    kind = rng.choice(["proj", "mlp", "gdn", "attn", "head", "gemm", "gemm", "load", "attn", "prefill", "request"])
    if kind == "proj":
        if rng.random() < 0.5:
            rows, K = rng.choice([(5120, 17408), (16384, 5120), (10240, 5120), (14336, 5120), (5120, 6144),
                                  (5120, 4096), (34816, 5120), (4096, 1024), (1024, 2048)])
        else:
            rows, K = _log(rng, 256, 34816), _width(rng)
        return {"kind": kind, "rows": rows, "K": K, "nr": rng.randint(1, 8), "bf16": rng.random() < 0.5,
                "res": rng.choice(["none", "bf16", "f32"])}
    if kind == "mlp":
        return {"kind": kind, "hidden": 1024 * rng.choice([1, 2, 4, 5]), "inter": rng.choice([INTER, 2048, _width(rng)]),
                "nr": rng.randint(1, 8)}
    if kind == "gdn":
        kh = rng.choice([1, 2, 4, 8, 16])
        nr = rng.randint(1, 8)
        return {"kind": kind, "kh": kh, "vh": kh * rng.choice([1, 2, 3]), "nr": nr, "npend": rng.randint(0, nr)}
    if kind == "attn":
        return {"kind": kind, "geom": rng.choice(["base", "base", "trunk", "trunk", "tiny"]),
                "pos0": _log(rng, 1, 16003), "nr": rng.randint(1, 8), "kv_group": rng.choice([16, 32, 32, 64])}
    if kind == "head":
        return {"kind": kind, "rows": _log(rng, 4096, VOCAB), "K": rng.choice([1024, 2048, 4096, 5120, 8 * _log(rng, 64, 640)]),
                "nr": rng.randint(1, 8)}
    if kind == "gemm":
        N, K = rng.choice([(5120, 17408), (34816, 5120), (16384, 5120), (10240, 5120), (14336, 5120), (5120, 6144),
                           (5120, 4096), (2048, 1024), (128 * _log(rng, 4, 136), 64 * _log(rng, 16, 96))])
        gs = 1024 if K % 1024 == 0 and rng.random() < 0.4 else 0
        M = _log(rng, 1, 2000 if N > 20000 else 4096)
        return {"kind": kind, "M": M, "N": N, "K": K, "gs": gs, "res": rng.random() < 0.5}
    if kind == "load":
        K = 64 * _log(rng, 16, 272)
        return {"kind": kind, "rows": max(16, min(16384, _log(rng, 16, 16384) * 4096 // K)), "K": K,
                "gs": 1024 if K % 1024 == 0 and rng.random() < 0.5 else 0}
    if kind == "prefill":
        return {"kind": kind, "geom": rng.choice(["base", "trunk"]), "n": _log(rng, 8, 2990), "gs": rng.choice([0, 0, 1024])}
    return {"kind": kind, "geom": rng.choice(["base", "trunk"]), "n": _log(rng, 8, 700), "gen": rng.randint(4, 24),
            "K": rng.randint(1, 7)}


# ---------------------------------------------------------------- inputs
class _Gen:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.g, device="cuda") * std

    def bf16(self, *shape, std=1.0):
        return self.normal(*shape, std=std).bfloat16()

    def uniform(self, lo, hi, *shape):
        return torch.rand(*shape, generator=self.g, device="cuda") * (hi - lo) + lo


def _groups(v, group):
    """Symmetric int8 codes with one fp32 scale per `group` columns."""
    x = v.view(v.shape[0], -1, group)
    s = x.abs().amax(-1) * (1.0 / 127.0)
    c = torch.round(x / s.clamp_min(1e-30)[..., None]).clamp_(-127, 127).to(torch.int8)
    return c.view(v.shape), s.contiguous()


def _weights(g, rows, K, group=64):
    return _groups(g.normal(rows, K, std=0.02), group)


def _p(t):
    return None if t is None else t.data_ptr()


_engines = {}


def _engine(X, case):
    """The model context a program keeps between requests (a few geometries at most)."""
    K, gs = case.get("K", 2), case.get("gs", 0)
    key = (case["geom"], K, gs)
    if key not in _engines:
        while len(_engines) >= 4:
            _engines.pop(next(iter(_engines))).close()
        nq, nkv, hd, rot = GEOMS[case["geom"]]
        cfg = X.default_config(n_layers=4, n_q=nq, n_kv=nkv, head_dim=hd, rot_dims=rot, spec_k=K, ctx=4096, pf_gs=gs)
        _engines[key] = X.Engine(cfg, 0x51E70003)
    return key


def _proj(X, w, s, xq, xs, y, res, nr):
    """Arguments of q27x_proj_rows: y[n] = W x[n] (+ res[n])."""
    h = X.I8G(w.data_ptr(), s.data_ptr(), 1.0, w.shape[0], w.shape[1])
    return (h, (ctypes.byref(h), _p(xq), w.shape[1], _p(xs), _p(y), w.shape[0], int(y.dtype == torch.bfloat16), _p(res),
                int(res is not None and res.dtype == torch.bfloat16), w.shape[0] if res is not None else 0,
                1.0 if res is not None else 0.0, nr, None))


def prepare(case, seed):
    X = _load()
    X.lib()
    kind = case["kind"]
    if kind in ("prefill", "request"):
        ids = torch.randint(0, VOCAB, (case["n"],), generator=torch.Generator().manual_seed(seed), dtype=torch.int32)
        return {"case": case, "key": _engine(X, case), "ids": ids.numpy()}
    t = _inputs(case, seed)
    L, calls = X.lib(), []
    dev = dict(device="cuda")
    if kind == "proj":
        nr, K, rows = case["nr"], case["K"], case["rows"]
        t["xq"], t["xs"] = torch.empty(nr, K, dtype=torch.int8, **dev), torch.empty(nr, K // 16, **dev)
        t["y"] = torch.empty(nr, rows, dtype=torch.bfloat16 if case["bf16"] else torch.float32, **dev)
        t["h"], args = _proj(X, t["w"], t["s"], t["xq"], t["xs"], t["y"], t.get("res"), nr)
        calls = [(L.q27x_quant_rows, (_p(t["x"]), K, _p(t["xq"]), K, _p(t["xs"]), K // 16, K, 1.0, nr, None)),
                 (L.q27x_proj_rows, args)]
        out = {"y": t["y"], "xq": t["xq"]}
    elif kind == "mlp":
        nr, H, I = case["nr"], case["hidden"], case["inter"]
        t["h16"] = torch.empty(nr, H, dtype=torch.bfloat16, **dev)
        t["xq"], t["xs"] = torch.empty(nr, H, dtype=torch.int8, **dev), torch.empty(nr, H // 16, **dev)
        t["g"], t["u"] = torch.empty(nr, I, **dev), torch.empty(nr, I, **dev)
        t["aq"], t["as"] = torch.empty(nr, I, dtype=torch.int8, **dev), torch.empty(nr, I // 16, **dev)
        t["y"] = torch.empty(nr, H, **dev)
        t["hg"], ag = _proj(X, t["wg"], t["sg"], t["xq"], t["xs"], t["g"], None, nr)
        t["hu"], au = _proj(X, t["wu"], t["su"], t["xq"], t["xs"], t["u"], None, nr)
        t["hd"], ad = _proj(X, t["wd"], t["sd"], t["aq"], t["as"], t["y"], t["h16"], nr)
        calls = [(L.q27x_rmsnorm_quant_rows, (_p(t["x"]), 0, H, _p(t["nw"]), 1.0, EPS, H, _p(t["h16"]), None, H,
                                              _p(t["xq"]), _p(t["xs"]), 0, 1.0, nr, None)),
                 (L.q27x_proj_rows, ag), (L.q27x_proj_rows, au),
                 (L.q27x_swiglu_quant_rows, (_p(t["g"]), _p(t["u"]), I, _p(t["aq"]), _p(t["as"]), I, 1.0, nr, None)),
                 (L.q27x_proj_rows, ad)]
        out = {"y": t["y"], "g": t["g"], "u": t["u"], "aq": t["aq"]}
    elif kind == "gdn":
        kh, vh, nr, npend = case["kh"], case["vh"], case["nr"], case["npend"]
        nqkv, nz = (2 * kh + vh) * 128, vh * 128
        t["pend"] = torch.zeros(L.q27x_gdn_pend_bytes(kh, vh, 128, 8), dtype=torch.uint8, **dev)
        t["out"] = torch.empty(nr, nz, dtype=torch.bfloat16, **dev)
        t["xq"], t["xs"] = torch.empty(nr, nz, dtype=torch.int8, **dev), torch.empty(nr, nz // 16, **dev)

        def verify(row0, rows, pending):
            return (_p(t["qkv"][row0:]), nqkv, _p(t["z"][row0:]), nz, _p(t["a"][row0:]), _p(t["b"][row0:]), vh, _p(t["A_log"]),
                    _p(t["dt"]), _p(t["nw"]), _p(t["conv"]), _p(t["S"]), _p(t["hist"]), _p(t["pend"]), pending, kh, vh, 128,
                    _p(t["out"]), nz, _p(t["xq"]), _p(t["xs"]), rows, None)

        # the round before: its rows are what this call commits npend of
        X.check(L.q27x_gdn_verify(*verify(0, nr, 0)))
        calls = [(L.q27x_gdn_verify, verify(nr, nr, npend))]
        out = {"out": t["out"], "xq": t["xq"], "xs": t["xs"], "S": t["S"]}
    elif kind == "attn":
        nq, nkv, hd, rot = GEOMS[case["geom"]]
        nr, pos0, G = case["nr"], case["pos0"], case["kv_group"]
        qkv_rows = 2 * nq * hd + 2 * nkv * hd
        t["qh"] = torch.empty(nr, nq * hd, dtype=torch.bfloat16, **dev)
        t["work"] = torch.empty(L.q27x_attn_work_bytes(nq, hd, pos0 + nr, nr), dtype=torch.uint8, **dev)
        t["out"] = torch.empty(nr, nq * hd, dtype=torch.bfloat16, **dev)
        t["xq"], t["xs"] = torch.empty(nr, nq * hd, dtype=torch.int8, **dev), torch.empty(nr, nq * hd // 16, **dev)
        calls = [(L.q27x_attn_prep_rows, (_p(t["qkv"]), qkv_rows, _p(t["qn"]), _p(t["kn"]), _p(t["cos"]), _p(t["sin"]), rot,
                                          _p(t["kc"]), _p(t["ks"]), _p(t["vc"]), _p(t["vs"]), G, _p(t["qh"]), nq, nkv, hd, 1,
                                          EPS, pos0, nr, None)),
                 (L.q27x_attn_rows, (_p(t["qh"]), _p(t["qkv"]), qkv_rows, _p(t["kc"]), _p(t["ks"]), _p(t["vc"]), _p(t["vs"]),
                                     G, nq, nkv, hd, 1, pos0, nr, _p(t["work"]), _p(t["out"]), _p(t["xq"]), _p(t["xs"]),
                                     None))]
        out = {"out": t["out"], "xq": t["xq"], "xs": t["xs"], "qh": t["qh"], "k": t["kc"][pos0:], "v": t["vc"][pos0:]}
    elif kind == "head":
        nr, K, rows = case["nr"], case["K"], case["rows"]
        t["y"], t["idx"], t["val"] = (torch.empty(nr, rows, **dev), torch.empty(nr, dtype=torch.int32, **dev),
                                      torch.empty(nr, **dev))
        calls = [(L.q27x_bf16_gemv_rows, (_p(t["w"]), rows, K, _p(t["x"]), K, _p(t["y"]), rows, 0, nr, None)),
                 (L.q27x_argmax_rows, (_p(t["y"]), rows, rows, nr, _p(t["idx"]), _p(t["val"]), None))]
        out = {"logits": t["y"], "idx": t["idx"], "val": t["val"]}
    elif kind == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        gs = case["gs"] or K
        t["xq"], t["xs"] = torch.empty(M, K, dtype=torch.int8, **dev), torch.empty(M, K // gs, **dev)
        t["y"] = torch.empty(M, N, **dev)
        calls = [(L.q27x_quant_tok_groups, (_p(t["x"]), K, M, K, gs, _p(t["xq"]), _p(t["xs"]), None)),
                 (L.q27x_gemm_i8g, (_p(t["w"]), _p(t["s"]), N, K, gs, 1.0, _p(t["xq"]), _p(t["xs"]), M, _p(t["y"]), N,
                                    _p(t.get("res")), N if case["res"] else 0, 1.0 if case["res"] else 0.0, None))]
        out = {"y": t["y"], "xq": t["xq"]}
    else:                                                     # load
        rows, K = case["rows"], case["K"]
        gs = case["gs"] or K
        t["q"], t["s"] = torch.empty(rows, K, dtype=torch.int8, **dev), torch.empty(rows, K // 64, **dev)
        t["gq"], t["gscale"] = torch.empty(rows, K, dtype=torch.int8, **dev), torch.empty(rows, K // gs, **dev)
        calls = [(L.q27x_quant_weights_i8g64, (_p(t["w"]), rows, K, _p(t["q"]), _p(t["s"]), None)),
                 (L.q27x_i8g64_to_grp, (_p(t["q"]), _p(t["s"]), rows, K, gs, _p(t["gq"]), _p(t["gscale"]), None))]
        out = {"q": t["q"], "s": t["s"], "gq": t["gq"], "gscale": t["gscale"]}
    return {"case": case, "tensors": t, "calls": calls, "out": out, "check": X.check}


def _inputs(case, seed):
    """The seeded device tensors a kernel-tier case reads (and the state it updates)."""
    g, kind, t = _Gen(seed), case["kind"], {}
    if kind == "proj":
        t["x"] = g.bf16(case["nr"], case["K"])
        t["w"], t["s"] = _weights(g, case["rows"], case["K"])
        if case["res"] != "none":
            t["res"] = g.normal(case["nr"], case["rows"]).to(torch.bfloat16 if case["res"] == "bf16" else torch.float32)
    elif kind == "mlp":
        H, I = case["hidden"], case["inter"]
        t["x"], t["nw"] = g.normal(case["nr"], H, std=3.0), g.bf16(H, std=0.02)
        for n, r, k in (("g", I, H), ("u", I, H), ("d", H, I)):
            t["w" + n], t["s" + n] = _weights(g, r, k)
    elif kind == "gdn":
        kh, vh, nr = case["kh"], case["vh"], case["nr"]
        nqkv, nz = (2 * kh + vh) * 128, vh * 128
        t["qkv"], t["z"] = g.bf16(2 * nr, nqkv), g.bf16(2 * nr, nz)          # the round before, then this one
        t["a"], t["b"] = g.uniform(-4, 0, 2 * nr, vh), g.uniform(-4, 0, 2 * nr, vh)
        t["A_log"], t["dt"] = g.uniform(0, 2.7, vh).bfloat16(), g.bf16(vh, std=0.1)
        t["nw"], t["conv"] = (1 + g.normal(128, std=0.02)).bfloat16(), g.bf16(nqkv, 4, std=0.3)
        t["S"], t["hist"] = g.normal(vh, 128, 128, std=0.1), g.bf16(nqkv, 3)
    elif kind == "attn":
        nq, nkv, hd, rot = GEOMS[case["geom"]]
        nr, pos0, ctx, kv = case["nr"], case["pos0"], case["pos0"] + case["nr"], nkv * hd
        t["qkv"] = g.bf16(nr, 2 * nq * hd + 2 * kv)
        t["qn"], t["kn"] = g.bf16(hd, std=0.02), g.bf16(hd, std=0.02)
        ang = torch.arange(ctx, dtype=torch.float64, device="cuda")[:, None] * \
            1e7 ** (-torch.arange(rot // 2, dtype=torch.float64, device="cuda") * 2 / rot)
        t["cos"], t["sin"] = ang.cos().float().contiguous(), ang.sin().float().contiguous()
        for n in ("k", "v"):
            t[n + "c"], t[n + "s"] = _groups(g.normal(ctx, kv), case["kv_group"])
    elif kind == "head":
        t["w"], t["x"] = g.bf16(case["rows"], case["K"], std=0.02), g.bf16(case["nr"], case["K"])
    elif kind == "gemm":
        t["x"] = g.normal(case["M"], case["K"])
        t["w"], t["s"] = _weights(g, case["N"], case["K"], case["gs"] or case["K"])
        if case["res"]:
            t["res"] = g.normal(case["M"], case["N"])
    else:
        t["w"] = g.normal(case["rows"], case["K"], std=0.02)
    return t


def run(state):
    if "calls" in state:
        for fn, args in state["calls"]:
            rc = fn(*args)
            if rc:
                state["check"](rc)
        return state["out"]
    case, eng = state["case"], _engines[state["key"]]
    tokens = [eng.prefill_gemm(state["ids"])]
    if case["kind"] == "request":
        tokens, _ = eng.generate(case["gen"], spec=True)
    # the last committed position's final hidden row (the engine keeps no logits: they are its product with the head)
    h = torch.from_numpy(eng.read("hprev", -1, "uint16", HIDDEN).view("int16")).view(torch.bfloat16)
    return {"tokens": torch.tensor(tokens), "hidden": h}


# ---------------------------------------------------------------- what a pass cannot do without
def _weight_bytes(rows, K):
    return rows * (K + K // 16)                                # int8 codes + fp32 scales per 64


def work(case):
    kind = case["kind"]
    if kind == "proj":
        nr, rows, K = case["nr"], case["rows"], case["K"]
        res = {"none": 0, "bf16": 2, "f32": 4}[case["res"]]
        return {"bytes": _weight_bytes(rows, K) + nr * (3 * K + K // 4 + rows * ((2 if case["bf16"] else 4) + res)),
                "flops": 2.0 * nr * rows * K}
    if kind == "mlp":
        nr, H, I = case["nr"], case["hidden"], case["inter"]
        return {"bytes": 2 * _weight_bytes(I, H) + _weight_bytes(H, I) + nr * (8 * H + 9 * I), "flops": 6.0 * nr * H * I}
    if kind == "gdn":
        kh, vh, nr = case["kh"], case["vh"], case["nr"]
        nqkv = (2 * kh + vh) * 128
        rows = nr * (2 * nqkv + vh * 128 * 5 + 8 * vh)         # inputs, gate, output with codes and scales
        return {"bytes": 2 * vh * 65536 + 20 * nqkv + rows, "flops": (nr * 6.0 + case["npend"] * 2) * vh * 16384}
    if kind == "attn":
        nq, nkv, hd, _ = GEOMS[case["geom"]]
        nr, ctx = case["nr"], case["pos0"] + case["nr"]
        return {"bytes": 2 * ctx * nkv * hd * (1 + 4 / case["kv_group"]) + nr * hd * (nq * 9 + nkv * 4),
                "flops": 4.0 * nr * nq * hd * ctx}
    if kind == "head":
        nr, rows, K = case["nr"], case["rows"], case["K"]
        return {"bytes": 2 * rows * K + nr * (2 * K + 4 * rows), "flops": 2.0 * nr * rows * K}
    if kind == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": N * K + 5 * M * K + M * N * (8 if case["res"] else 4), "flops": 2.0 * M * N * K}
    if kind == "load":
        return {"bytes": case["rows"] * case["K"] * (4 + 1 + 1 + 1 / 16), "flops": 0.0}
    nq, nkv, hd, _ = GEOMS[case["geom"]]
    attn = HIDDEN * (2 * nq * hd + 2 * nkv * hd) + HIDDEN * nq * hd
    gdn = HIDDEN * 16384 + HIDDEN * 6144
    params = 4 * 3 * HIDDEN * INTER + 3 * gdn + attn                 # the 4-layer slice
    n = case["n"]
    w = {"bytes": params * 1.0 + 2 * VOCAB * HIDDEN, "flops": 2.0 * n * (params + 3 * HIDDEN * HIDDEN) + 2.0 * nq * hd * n * n}
    if kind == "request":
        # at least gen / (K + 1) rounds of K drafts and a verify, each reading the weights and the head once
        draft = attn + 3 * HIDDEN * INTER + 2 * HIDDEN * HIDDEN + 2 * VOCAB * HIDDEN
        rounds = math.ceil((case["gen"] - 1) / (case["K"] + 1))
        w["bytes"] += rounds * (case["K"] * draft + params * 17 / 16 + 2 * VOCAB * HIDDEN)
    return w


def tolerance(case):
    # about four times the distance to the 64-bit results: bf16 outputs are 1.6e-3 to 1.8e-3 off them; the int8
    # codes of bf16 values meet exact half ties (3e-4 of a projection's fp32 result), those of fp32 values hardly
    # any (3e-5 of a GEMM's); fp32 sums alone are 1e-7 off
    return {
        "proj": {"rel": 7e-3 if case.get("bf16") else 1.4e-3, "differ": 1e-3},
        "mlp": {"rel": 1e-4, "differ": 1e-3},
        "gdn": {"rel": 7e-3, "differ": 5e-3},
        "attn": {"rel": 7e-3, "differ": 5e-3},
        "head": {"rel": 4e-7, "differ": 0.0},
        "gemm": {"rel": 1.4e-4, "differ": 1e-5},
        "load": {"rel": 2e-7, "differ": 1e-5},
        # bf16 rounding and int8 code flips travel through four layers; tokens have to stay the same
        "prefill": {"rel": 1e-2, "max": 0.5, "differ": 0.0},
        "request": {"rel": 1e-2, "max": 0.5, "differ": 0.0},
    }[case["kind"]]


# ---------------------------------------------------------------- the same in 64 bits
def _q(v, group):
    x = v.view(v.shape[0], -1, group)
    s = x.abs().amax(-1, keepdim=True) / 127
    return (torch.round(x / s.clamp_min(1e-300)).clamp(-127, 127) * s).view(v.shape)


def _deq(c, s, group):
    return (c.double().view(c.shape[0], -1, group) * s.double()[..., None]).view(c.shape)


def _rms(x, w=None):
    y = x / (x.square().mean(-1, keepdim=True) + EPS).sqrt()
    return y if w is None else y * (1 + w.double())


def _mm(w, s, x, group=64):
    """x W^T by row blocks, so the 64-bit copy of the weights stays small."""
    return torch.cat([x @ _deq(w[r:r + 8192], s[r:r + 8192], group).t() for r in range(0, w.shape[0], 8192)], 1)


def _silu(x):
    return x * torch.sigmoid(x)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("prefill", "request"):
        return None
    t = _inputs(case, seed)
    if kind == "proj":
        y = _mm(t["w"], t["s"], _q(t["x"].double(), 16))
        return {"y": y + t["res"].double() if "res" in t else y, "xq": None}
    if kind == "mlp":
        x = t["x"].double()
        xn = _q(_rms(x, t["nw"]), 16)
        g, u = _mm(t["wg"], t["sg"], xn), _mm(t["wu"], t["su"], xn)
        return {"y": _mm(t["wd"], t["sd"], _q(_silu(g) * u, 16)) + t["x"].bfloat16().double(), "g": g, "u": u, "aq": None}
    if kind == "gdn":
        return _exact_gdn(case, t)
    if kind == "attn":
        return _exact_attn(case, t)
    if kind == "head":
        y = torch.cat([t["x"].double() @ t["w"][r:r + 8192].double().t() for r in range(0, case["rows"], 8192)], 1)
        return {"logits": y, "idx": None, "val": y.amax(1)}
    if kind == "gemm":
        gs = case["gs"] or case["K"]
        y = _mm(t["w"], t["s"], _q(t["x"].double(), gs), gs)
        return {"y": y + t["res"].double() if case["res"] else y, "xq": None}
    s = t["w"].double().view(case["rows"], -1, 64).abs().amax(-1) / 127
    gs = case["gs"] or case["K"]
    return {"q": None, "s": s, "gq": None, "gscale": s.view(case["rows"], -1, gs // 64).amax(-1)}


def _exact_gdn(case, t):
    kh, vh, nr, npend = case["kh"], case["vh"], case["nr"], case["npend"]
    d, hist = 128, t["hist"].double()
    S = t["S"].double()

    def rows(S, hist, r0, n, keep):
        """n rows from row r0; the state after `keep` of them and every row's output."""
        kept, outs = S, []
        for i in range(n):
            x = t["qkv"][r0 + i].double()
            w = torch.cat([hist, x[:, None]], 1)
            hist = w[:, 1:]
            c = _silu((w * t["conv"].double()).sum(1)).bfloat16().double()
            q, k, v = c[:kh * d].view(kh, d), c[kh * d:2 * kh * d].view(kh, d), c[2 * kh * d:].view(vh, d)
            q = q / (q.square().sum(-1, keepdim=True) + 1e-6).sqrt() / math.sqrt(d)
            k = k / (k.square().sum(-1, keepdim=True) + 1e-6).sqrt()
            q, k = (m.repeat_interleave(vh // kh, 0) for m in (q, k))
            beta = torch.sigmoid(t["b"][r0 + i].double())[:, None]
            dec = torch.exp(-t["A_log"].double().exp() *
                            torch.nn.functional.softplus(t["a"][r0 + i].double() + t["dt"].double()))[:, None]
            delta = (v - dec * (S * k[:, :, None]).sum(1)) * beta
            S = dec[:, :, None] * S + k[:, :, None] * delta[:, None, :]
            o = (S * q[:, :, None]).sum(1)
            o = _rms(o) * t["nw"].double() * _silu(t["z"][r0 + i].double().view(vh, d))
            outs.append(o.reshape(-1))
            if i + 1 == keep:
                kept, hist_kept = S, hist
        return kept, (hist_kept if keep else None), torch.stack(outs)

    kept, h, _ = rows(S, hist, 0, nr, npend)
    _, _, out = rows(kept, hist if h is None else h, nr, nr, 0)
    return {"out": out, "xq": None, "xs": None, "S": kept}


def _exact_attn(case, t):
    nq, nkv, hd, rot = GEOMS[case["geom"]]
    nr, pos0, G = case["nr"], case["pos0"], case["kv_group"]
    kv = nkv * hd
    qkv = t["qkv"].double()
    qg = qkv[:, :2 * nq * hd].view(nr, nq, 2 * hd)
    q, gate, k, v = qg[..., :hd], qg[..., hd:], qkv[:, 2 * nq * hd:2 * nq * hd + kv], qkv[:, 2 * nq * hd + kv:]
    cos, sin = (t[n][pos0:].double()[:, None, :].repeat(1, 1, 2) for n in ("cos", "sin"))

    def rope(x):
        r, h = x[..., :rot], rot // 2
        turned = torch.cat([-r[..., h:], r[..., :h]], -1)
        return torch.cat([r * cos + turned * sin, x[..., rot:]], -1)

    q = rope(_rms(q, t["qn"])).bfloat16().double()
    k = _q(rope(_rms(k.reshape(nr, nkv, hd), t["kn"])).reshape(nr, kv), G)
    K = torch.cat([_deq(t["kc"][:pos0], t["ks"][:pos0], G), k]).view(-1, nkv, hd)
    V = torch.cat([_deq(t["vc"][:pos0], t["vs"][:pos0], G), _q(v.reshape(nr, kv), G)]).view(-1, nkv, hd)
    out = torch.empty(nr, nq, hd, dtype=torch.float64, device="cuda")
    seen = torch.arange(pos0 + nr, device="cuda")[None, :] <= pos0 + torch.arange(nr, device="cuda")[:, None]
    for h in range(nq):
        j = h // (nq // nkv)
        s = (q[:, h] @ K[:, j].t()) / math.sqrt(hd)
        out[:, h] = torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ V[:, j]
    return {"out": (out * torch.sigmoid(gate)).view(nr, -1), "xq": None, "xs": None, "qh": q.reshape(nr, -1), "k": None, "v": None}
