"""Performance cases: the work that a program using this framework has it do.

A case names a kind of work and its sizes; prepare() builds what a program holds
before the call (modules with loaded and packed weights, inputs on the GPU), run()
makes one pass through the public entry points, exact() gives the same outputs in
64 bits with plain torch. Kinds:

  layer    TuckerMoE.forward: prefill and decode, bf16 / fp32 / fp8 weights, both
           routers, narrow and wide routers, with or without the routing outputs
  ffn      TuckerFFN.forward: the transformer block's FFN sub-block (three layers)
  outproj  TuckerOutProj.forward: the Mamba block's output sub-block (one layer)
  latent   FusedLatentMoE forward and backward, the training layer's expert
           contraction

"router" is "topk" (softmax over the top-k logits) or "capped" (the router that the
trained checkpoints use). Sizes are those of the workloads C1..C5, F1 / F2 and the
reference model's layers (d 768, x_up 1536 -> 6144, r = (32, 512, 256), E 8, k 2).
"""
import importlib.util
import math
import os
import sys

import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
_PKG = "mamba_tuckermoe_amd"
_EPS = 1e-5
_DT = {"bf16": torch.bfloat16, "fp32": torch.float32}


def _package():
    """The package, whose folder's name is no Python identifier."""
    if _PKG not in sys.modules:
        d = os.path.join(_ROOT, "mamba-tuckermoe_amd")
        spec = importlib.util.spec_from_file_location(
            _PKG, os.path.join(d, "__init__.py"), submodule_search_locations=[d])
        sys.modules[_PKG] = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(sys.modules[_PKG])
    return sys.modules[_PKG]


# (d_in, d_out, E, k, r1, r2, r3) of the layers
_C = dict(d_in=1536, d_out=2304, E=16, k=2, r1=4, r2=1024, r3=256)
_XUP = dict(d_in=1536, d_out=6144, E=8, k=2, r1=32, r2=512, r3=256)
_C1 = dict(d_in=512, d_out=1024, E=8, k=2, r1=4, r2=256, r3=128)
_REF = dict(E=8, k=2, r1=32, r2=512, r3=256)          # the reference model's ranks


def _layer(T, shape, dtype="bf16", router="topk", fp8=False, routing=False, **over):
    return dict(dict(kind="layer", T=T, dtype=dtype, router=router, fp8=fp8, routing=routing),
                **dict(shape, **over))


def _ffn(T, dtype="bf16", router="topk", r1=32):
    return dict(dict(kind="ffn", T=T, dtype=dtype, router=router, d=768, expand=6),
                **dict(_REF, r1=r1))


def _outproj(T, dtype="bf16", router="topk"):
    return dict(dict(kind="outproj", T=T, dtype=dtype, router=router, d=768), **_REF)


def _latent(B, dtype="bf16", p32=True, E=8, k=2):
    return dict(kind="latent", B=B, dtype=dtype, p32=p32, E=E, k=k, r3=256, r2=1024)


def listed():
    return [
        # one sequence's decode step through one layer: launch and host latency
        dict(_layer(1, _C), name="decode_T1"),
        # a decode batch of 32 sequences (C2)
        dict(_layer(32, _C), name="decode_T32"),
        # a small fp32 layer that also reports its routing, as load statistics need (C1)
        dict(_layer(64, _C1, dtype="fp32", routing=True), name="fp32_T64_routing"),
        # the transformer block's FFN in one token's generation step, with the router
        # of the trained checkpoints
        dict(_ffn(1, router="capped"), name="ffn_decode_T1"),
        # the Mamba block's output sub-block on an odd batch of rows between the decode
        # and prefill sizes
        dict(_outproj(193, router="capped"), name="outproj_T193"),
        # the reference model's widest projection in its checkpoints' own type
        dict(_layer(1021, _XUP, dtype="fp32"), name="xup_fp32_T1021"),
        # prefill of one 2048-token sequence
        dict(_layer(2048, _C), name="prefill_T2048"),
        # fp8 weights on a ragged batch of prompts
        dict(_layer(5003, _C, fp8=True), name="prefill_fp8_T5003"),
        # a wide router: 256 experts, top-8 (C4)
        dict(_layer(4096, _C, E=256, k=8), name="prefill_E256_T4096"),
        # the transformer block's FFN on a prompt, the reference model's sizes (F1)
        dict(_ffn(4096), name="ffn_prefill_T4096"),
        # prefill of eight 2048-token sequences (C3)
        dict(_layer(16384, _C), name="prefill_T16384"),
        # one training step of the expert contraction: forward and backward
        dict(_latent(16384), name="latent_train_B16384"),
    ]


def _log_int(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choices(["layer", "wide", "ffn", "outproj", "latent"], [45, 15, 15, 10, 15])[0]
    router = rng.choice(["topk", "topk", "capped"])
    if kind == "layer":
        shape = rng.choice([_C, _C, _XUP, _C1])
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp32"])
        top = 1024 if dtype == "fp32" else (6144 if shape is _XUP else 16384)
        over = {}
        if shape is _C:
            over["E"] = rng.choice([4, 8, 16, 24, 32])
            over["k"] = rng.choice([1, 2, 2, 3, 4])
        return _layer(_log_int(rng, 1, top), shape, dtype=dtype, router=router,
                      fp8=dtype == "bf16" and rng.random() < 0.25, routing=rng.random() < 0.2,
                      **over)
    if kind == "wide":
        return _layer(_log_int(rng, 1, 6144), _C, router=router, routing=rng.random() < 0.2,
                      E=rng.choice([48, 64, 96, 128, 160, 256]), k=rng.choice([2, 4, 6, 8]))
    if kind == "ffn":
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp32"])
        return _ffn(_log_int(rng, 1, 256 if dtype == "fp32" else 4096), dtype=dtype,
                    router=router, r1=rng.choice([4, 32]))
    if kind == "outproj":
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp32"])
        return _outproj(_log_int(rng, 1, 2048 if dtype == "fp32" else 16384), dtype=dtype,
                        router=router)
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp32"])
    E = rng.choice([4, 8, 8, 16])
    # the contraction's present form is dense over the experts: bounded so that no drawn
    # case costs more than the listed one in that form either
    top = (131072 if dtype == "bf16" else 8192) // E
    return _latent(_log_int(rng, 256, top), dtype=dtype, p32=rng.random() < 0.7, E=E,
                   k=rng.choice([1, 2, 2, 4]))


# ---- inputs --------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 13)
    return g


def _normal(g, shape, std=1.0, mean=0.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std + mean


def _layer_params(g, d_in, d_out, c):
    """float32 parameters of one layer, N(0, 1/fan_in) as the reference's tests draw them."""
    E, r1, r2, r3 = c["E"], c["r1"], c["r2"], c["r3"]
    # the capped router's checkpoints have sharper logits, some of them bent by the cap
    rstd = (0.02 if E > 128 else d_in ** -0.5) * (4.0 if c["router"] == "capped" else 1.0)
    return {
        "router.weight": _normal(g, (E, d_in), rstd),
        "U_in": _normal(g, (d_in, r3), d_in ** -0.5),
        "inner_norm.weight": _normal(g, (r3,), 0.1, 1.0),
        "U_expert": _normal(g, (E, r1)),
        "core": _normal(g, (r1, r3, r2), (r1 * r3) ** -0.5),
        "U_out": _normal(g, (r2, d_out), r2 ** -0.5),
        "bias": _normal(g, (d_out,), 0.1),
    }


_LAYERS = {"layer": ("",), "ffn": ("ffn_gate.", "ffn_up.", "ffn_down."), "outproj": ("out_proj.",)}


def _dims(case, name):
    if case["kind"] == "layer":
        return case["d_in"], case["d_out"]
    d, dff = case["d"], case["d"] * case.get("expand", 1)
    return (dff, d) if name == "ffn_down." else (d, dff)


def _quantised(w, dims):
    """(e4m3 codes, fp32 scales, the fp32 weight they stand for): absmax over the rows."""
    s = w.abs().amax(dim=dims, keepdim=True) / 448.0
    q = (w / s).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    return q, s.squeeze(dims).contiguous(), q.float() * s


def _inputs(case, seed):
    """(weights a module loads, fp8 codes and scales or None, the weights that the
    computed layer has, x)."""
    g, dt = _gen(seed), _DT[case["dtype"]]
    sd, fp8 = {}, None
    for name in _LAYERS[case["kind"]]:
        d_in, d_out = _dims(case, name)
        for k, v in _layer_params(g, d_in, d_out, case).items():
            sd[name + k] = v
    if case["kind"] != "layer":
        norm, ls = ("norm_ffn", "ls_ffn") if case["kind"] == "ffn" else ("norm_out_proj",
                                                                        "ls_out_proj")
        sd[norm + ".weight"] = _normal(g, (case["d"],), 0.1, 1.0)
        sd[ls + ".gamma"] = _normal(g, (case["d"],), 0.1, 1.0)
    x = _normal(g, (case["T"], case.get("d_in", case.get("d")))).to(dt)
    ref = {k: v.to(dt) for k, v in sd.items()}
    if case.get("fp8"):
        fp8 = []
        for k, dims in (("U_in", (0,)), ("core", (1,)), ("U_out", (0,))):
            q, s, w = _quantised(sd[k], dims)
            fp8 += [q, s]
            ref[k] = w
    return {k: v.to(dt) for k, v in sd.items()}, fp8, ref, x


def _latent_inputs(case, seed):
    g, dt = _gen(seed), _DT[case["dtype"]]
    B, E, k, r3, r2 = case["B"], case["E"], case["k"], case["r3"], case["r2"]
    x = _normal(g, (B, r3)).to(dt)
    G = _normal(g, (E, r3, r2), r3 ** -0.5).to(dt)
    # a router's choice: every expert drawn, some more often than others
    logits = _normal(g, (B, E)) + _normal(g, (E,), 0.5)
    top, idx = torch.topk(logits, k, dim=-1)
    p = torch.softmax(top, dim=-1)
    if not case["p32"]:
        p = p.to(dt)
    dout = _normal(g, (B, r2)).to(dt)
    return x, G, idx, p, dout


# ---- a pass --------------------------------------------------------------------

class _Cfg:
    def __init__(self, c):
        self.rms_norm_eps = _EPS
        self.kmoe_num_experts, self.kmoe_top_k = c["E"], c["k"]
        self.kmoe_r1, self.kmoe_r2, self.kmoe_r3 = c["r1"], c["r2"], c["r3"]
        self.ffn_expand = c.get("expand", 1)


def prepare(case, seed):
    pkg = _package()
    if case["kind"] == "latent":
        x, G, idx, p, dout = _latent_inputs(case, seed)
        return {"kind": "latent", "fn": pkg.FusedLatentMoE, "x": x.requires_grad_(),
                "G": G.requires_grad_(), "idx": idx, "p": p.requires_grad_(), "dout": dout}
    sd, fp8, _, x = _inputs(case, seed)
    cfg = _Cfg(case)
    with torch.device("cuda"):
        if case["kind"] == "layer":
            m = pkg.TuckerMoE(case["d_in"], case["d_out"], cfg)
        elif case["kind"] == "ffn":
            m = pkg.TuckerFFN(case["d"], cfg)
        else:
            m = pkg.TuckerOutProj(case["d"], cfg)
    m = m.to(_DT[case["dtype"]]).eval()
    m.load_state_dict(sd)
    layers = [mod for mod in m.modules() if isinstance(mod, pkg.TuckerMoE)]
    for layer in layers:
        if case["router"] == "capped":
            layer.set_router_mode("capped")
        if fp8 is not None:
            layer.load_fp8(*fp8)
        layer.packed()           # the kernels' copy of the weights, kept by the module
    return {"kind": case["kind"], "m": m, "x": x, "routing": case.get("routing", False)}


def run(state):
    if state["kind"] == "latent":
        x, G, p = state["x"], state["G"], state["p"]
        out = state["fn"].apply(x, G, state["idx"], p)
        dx, dG, dp = torch.autograd.grad(out, (x, G, p), state["dout"])
        return {"out": out.detach(), "dx": dx, "dG": dG, "dp": dp}
    with torch.no_grad():
        if state["routing"]:
            out, idx, w, logits = state["m"].forward_with_routing(state["x"], logits=True)
            return {"out": out, "idx": idx, "w": w, "logits": logits}
        return state["m"](state["x"])


# ---- what a pass cannot do without ---------------------------------------------

def _layer_work(T, d_in, d_out, c, es, fp8=False):
    """(weight bytes, flops) of one layer: each token's k experts' contraction (no more
    ranks than min(r1, k)), in the cheaper of its two orders."""
    E, r1, r2, r3 = c["E"], c["r1"], c["r2"], c["r3"]
    proj = d_in * r3 + r1 * r3 * r2 + r2 * d_out
    small = E * d_in + r3 + E * r1 + d_out
    nbytes = small * es + (proj + 4 * (r3 + r1 * r2 + d_out) if fp8 else proj * es)
    rk = min(r1, c["k"])
    rest = min(rk * r3 * r2 + r2 * d_out, rk * r3 * d_out)
    return nbytes, 2 * T * (E * d_in + d_in * r3 + rest)


def work(case):
    es = 4 if case["dtype"] == "fp32" else 2
    if case["kind"] == "latent":
        B, E, k, r3, r2 = case["B"], case["E"], case["k"], case["r3"], case["r2"]
        ps = 4 if case["p32"] else es
        acts = es * (2 * B * r3 + 2 * B * r2) + B * k * (8 + 2 * ps)
        return {"bytes": acts + 2 * es * E * r3 * r2, "flops": 6 * B * k * r3 * r2}
    T = case["T"]
    if case["kind"] == "layer":
        wb, fl = _layer_work(T, case["d_in"], case["d_out"], case, es, case["fp8"])
        nbytes = wb + T * (case["d_in"] + case["d_out"]) * es
        if case["routing"]:
            nbytes += T * (case["k"] * 12 + case["E"] * 4)
        return {"bytes": nbytes, "flops": fl}
    nbytes, flops = 2 * T * case["d"] * es + 2 * case["d"] * es, 0
    for name in _LAYERS[case["kind"]]:
        wb, fl = _layer_work(T, *_dims(case, name), case, es)
        nbytes, flops = nbytes + wb, flops + fl
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Relative 2-norm differences, about four times what was measured against exact()
    (but for the FFN). One layer in bf16 is 3.3e-3 to 4.1e-3 from it (16-bit
    intermediates and output), in fp32 2.5e-7 to 9.3e-7 (sums of up to 1536 and 2048
    terms); the contraction's forward and gradients 2.3e-3 and 6e-7. In the FFN a row whose
    gate, up or down router sees two nearly equal logits may route differently (1.5% of
    the rows in bf16, since the routers' inputs are rounded): 5.9e-2 on a prompt."""
    fp32 = case["dtype"] == "fp32"
    if case["kind"] == "latent":
        return {"rel": 3e-6 if fp32 else 1e-2}
    if case["kind"] == "ffn":
        return {"rel": 1e-5 if fp32 else 1e-1}
    rel = {"rel": 4e-6 if fp32 else 1.4e-2}
    return dict(rel, differ=1e-3) if case.get("routing") else rel


# ---- the same outputs in 64 bits -----------------------------------------------

def _rms(v, w):
    return v / (v.pow(2).mean(-1, keepdim=True) + _EPS).sqrt() * w


def _layer_f64(x, sd, name, c):
    """One layer: (out, idx, weights, logits)."""
    w = {k: sd[name + k].double() for k in ("router.weight", "U_in", "inner_norm.weight",
                                            "U_expert", "core", "U_out", "bias")}
    logits = x @ w["router.weight"].t()
    if c["router"] == "capped":
        scores = 10.0 * torch.tanh(logits / 10.0) / 0.5
        _, idx = torch.topk(scores, c["k"], dim=-1)
        top = torch.softmax(scores, dim=-1).gather(-1, idx)
        p = top / (top.sum(-1, keepdim=True) + 1e-6)
    else:
        top, idx = torch.topk(logits, c["k"], dim=-1)
        p = torch.softmax(top, dim=-1)
    z = _rms(x @ w["U_in"], w["inner_norm.weight"])
    coef = (p.unsqueeze(-1) * w["U_expert"][idx]).sum(1)
    mid = torch.zeros(x.shape[0], c["r2"], dtype=torch.float64, device=x.device)
    for r in range(c["r1"]):
        mid += (coef[:, r:r + 1] * z) @ w["core"][r]
    return mid @ w["U_out"] + w["bias"], idx, p, logits


def exact(case, seed):
    if case["kind"] == "latent":
        x, G, idx, p, dout = _latent_inputs(case, seed)
        x, G, p, dout = x.double(), G.double(), p.double(), dout.double()
        out, dx = torch.zeros_like(dout), torch.zeros_like(x)
        dG, dp = torch.zeros_like(G), torch.zeros_like(p)
        for e in range(case["E"]):
            for j in range(case["k"]):
                rows = (idx[:, j] == e).nonzero().squeeze(-1)
                if rows.numel() == 0:
                    continue
                xe, de, pe = x[rows], dout[rows], p[rows, j:j + 1]
                y, back = xe @ G[e], de @ G[e].t().contiguous()
                out[rows] += pe * y
                dx[rows] += pe * back
                dp[rows, j] = (de * y).sum(-1)
                dG[e] += (pe * xe).t().contiguous() @ de
        return {"out": out, "dx": dx, "dG": dG, "dp": dp}
    _, _, sd, x = _inputs(case, seed)
    x = x.double()
    if case["kind"] == "layer":
        out, idx, p, logits = _layer_f64(x, sd, "", case)
        if not case["routing"]:
            return out
        return {"out": out, "idx": idx, "w": p, "logits": logits}
    if case["kind"] == "outproj":
        y = _layer_f64(_rms(x, sd["norm_out_proj.weight"].double()), sd, "out_proj.", case)[0]
        return x + sd["ls_out_proj.gamma"].double() * y
    xf = _rms(x, sd["norm_ffn.weight"].double())
    gate = _layer_f64(xf, sd, "ffn_gate.", case)[0]
    h = gate * torch.sigmoid(gate) * _layer_f64(xf, sd, "ffn_up.", case)[0]
    return x + sd["ls_ffn.gamma"].double() * _layer_f64(h, sd, "ffn_down.", case)[0]
