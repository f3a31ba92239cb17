"""Folded bf16 batches between the decode launch and the large-tile kernels: 64 < T <= 256,
where they pay (test_batch_rules.py has the rules), for unfolded plans while the 64 x 128 out-projection tiles number at most 256. Against
the float64 oracle at the bf16 bar, at the edges of the token and column tiles, of the rule
and of the K slices (1, several, 8), with each front (small, K-sliced, plain), the fused
epilogues of the sub-blocks, fp8 weights and under graph capture."""
import numpy as np
import pytest
import torch

from oracle import tucker_moe_np as onp

pytestmark = pytest.mark.gpu


def _layer(pkg, dev, shape, T, fp8=False):
    E, k, r1, r3, r2, d_in, d_out = shape
    w = pkg.Workload("custom", T, d_in, d_out, E, k, r1, r3, r2, torch.bfloat16, 93, fp8=fp8)
    if fp8:
        params, codes, ref = pkg.synth.make_fp8_params(w, affine="random")
    else:
        params = ref = pkg.synth.make_params(w, affine="random")
    m = pkg.TuckerMoE(w.d_in, w.d_out, w.cfg()).to(dev, w.dtype)
    m.load_state_dict({k_: v.to(dev) for k_, v in params.items()})
    if fp8:
        m.load_fp8(*(codes[n].to(dev) for n in ("U_in_q", "U_in_scale", "core_q", "core_scale",
                                                "U_out_q", "U_out_scale")))
    return w, ref, m, pkg.synth.make_x(w)


def _run(m, x):
    with torch.no_grad():
        got = m.forward_with_routing(x, logits=True)
    torch.cuda.synchronize()
    return got


def _check(m, x, dev, ref, k):
    out, idx, wts, lg = _run(m, x.to(dev))
    m.check_signals()
    want = onp.forward_f64(x, ref, k)
    err = onp.rel_l2(out.float().cpu().numpy(), want["out"])
    print(f"T={x.shape[0]}: {err:.2e}", end=" ", flush=True)
    assert np.array_equal(idx.cpu().numpy(), want["idx"])
    assert onp.rel_l2(lg.cpu().numpy(), want["logits"]) < 1e-5
    assert err <= 1e-2
    return out


# (E, k, r1, r3, r2, d_in, d_out), the T's that run as a folded batch, and T's on the other side
# of a rule's edge: folded with a sliced and with the small front, a wide router, a ragged last
# column tile; folded in one round of the skinny out-projection (no batch); the reference's
# ranks at the smallest T, one row past a tile, the last T of the range and the first past it;
# 256 tiles and past them (the two GEMMs); rank 4 unfolded; K = 64 (one slice) in one round
# (no batch) and in two; K 768 on both sides of its line
@pytest.mark.parametrize("shape,Ts,others", [
    ((16, 2, 4, 256, 1024, 1536, 2304), (65, 129, 200, 256), (64, 257)),
    ((64, 4, 4, 256, 1024, 512, 2320), (80, 255), (65, 79)),
    ((64, 4, 4, 256, 1024, 512, 304), (), (65, 255)),
    ((8, 2, 32, 256, 512, 768, 768), (65, 193, 256), (257,)),
    ((8, 2, 32, 256, 512, 1536, 6144), (128, 255), ()),
    ((8, 2, 4, 256, 512, 768, 4608), (129, 250), ()),
    ((8, 2, 8, 256, 256, 256, 8192), (192, 193, 256), ()),
    ((8, 2, 8, 64, 64, 256, 10880), (192,), (193,)),
    ((4, 1, 1, 64, 256, 256, 64), (), (70, 256)), ((4, 1, 1, 64, 256, 256, 4112), (65, 70, 256), ()),
    ((4, 2, 3, 256, 1024, 256, 2304), (96, 250), (65, 95)),
], ids=lambda v: str(v))
def test_batch_fold(pkg, dev, shape, Ts, others):
    for T in Ts + others:
        w, ref, m, x = _layer(pkg, dev, shape, T)
        assert bool(m.plan().forward_form(T) & pkg._lib.TMOE_FORM_BATCH) == (T in Ts), T
        _check(m, x, dev, ref, w.k)


def test_batch_fold_fp8(pkg, dev):
    for shape in ((16, 2, 4, 256, 1024, 1536, 2304), (8, 2, 4, 256, 512, 768, 4608)):
        w, ref, m, x = _layer(pkg, dev, shape, 100, fp8=True)
        assert m.plan().forward_form(100) & pkg._lib.TMOE_FORM_BATCH
        _check(m, x, dev, ref, w.k)


def test_batch_fold_capture_and_flags(pkg, dev):
    """Captured (the K-sliced front's two launches) and without in-launch signals: the same
    bits; set_fold(False) keeps the two GEMMs."""
    w, ref, m, x = _layer(pkg, dev, (8, 2, 32, 256, 512, 1536, 768), 150)
    assert m.plan().forward_form(150) == (pkg._lib.TMOE_FORM_FOLDED | pkg._lib.TMOE_FORM_BATCH |
                                          pkg._lib.TMOE_FORM_FRONT_SLICED)
    out = _check(m, x, dev, ref, w.k)
    xs = x.to(dev)
    g = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(g):
        cap = m(xs)
    for _ in range(3):
        cap.zero_()
        g.replay()
        assert torch.equal(cap, out)
        assert torch.equal(_run(m, xs)[0], out)
    m.set_fuse(False)
    assert torch.equal(_run(m, xs)[0], out)
    m.set_fuse(True).set_fold(False)
    _check(m, x, dev, ref, w.k)


@pytest.mark.parametrize("T", [65, 200, 300])
def test_batch_fold_epilogues(pkg, dev, T):
    """The sub-blocks' fused epilogues (and an in-place residual) against the layers' own
    outputs combined in float64 from the same inputs."""
    cfg = pkg.TuckerMoEConfig(kmoe_r1=32)
    g = torch.Generator().manual_seed(T)
    ffn = pkg.TuckerFFN(256, cfg).to(dev, torch.bfloat16)
    sd = {k: torch.randn(v.shape, generator=g) * (v.shape[-2] ** -0.5 if v.dim() > 1 else 0.1)
          + (0.0 if v.dim() > 1 or "bias" in k else 1.0) for k, v in ffn.state_dict().items()}
    ffn.load_state_dict({k: v.to(dev, torch.bfloat16) for k, v in sd.items()})
    x = torch.randn(T, 256, generator=g).to(dev, torch.bfloat16)
    with torch.no_grad():
        st = ffn.stages(x)
        up = ffn.ffn_up(st["x_f"]).double()
        gate = st["gate"].double()
        h = torch.nn.functional.silu(gate) * up
        dn = ffn.ffn_down(st["h"]).double()
        want = x.double() + ffn.ls_ffn.gamma.double() * dn
        out = ffn(x)
        xi = x.clone()
        ffn(xi, inplace=True)
    assert (st["h"].double() - h).norm() <= 6e-3 * h.norm()      # two roundings to bf16
    assert (st["out"].double() - want).norm() <= 6e-3 * want.norm()
    assert torch.equal(out, st["out"]) and torch.equal(xi, out)
