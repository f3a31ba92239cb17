"""Unfolded plans at decode sizes (T <= 64): one folded launch against the W^T packed
beside the two-GEMM weights. Against the float64 oracle at the bf16 bar, at the edges of its
token blocks and of the rule (K = rk r3 of 2048 in one and two weight groups a wave, W^T of
32 MB; test_batch_rules.py has it whole), and no less exact than the two-GEMM form (both round c z, and the one W^T where the
other rounds its intermediate: errors within a tenth of each other)."""
import numpy as np
import pytest
import torch

from oracle import tucker_moe_np as onp

pytestmark = pytest.mark.gpu

# (E, k, r1, r3, r2, d_in, d_out): the expert form of the reference's ranks, more consumers
# than compute units, rank 4 unfolded, r3 = 64 with 32 ranks, K not a multiple of 128 wide
# tiles, the smallest d_out, W^T of exactly 32 MB (folded from 33 tokens on), three rounds of
# consumers
SHAPES = [
    (8, 2, 32, 256, 512, 768, 768), (8, 2, 32, 256, 512, 768, 4608),
    (8, 2, 4, 256, 512, 768, 4608), (16, 3, 32, 64, 64, 256, 1040),
    (16, 16, 3, 64, 64, 512, 272), (4, 1, 64, 128, 64, 1536, 128),
    (8, 2, 8, 256, 256, 256, 8192), (16, 2, 4, 128, 256, 512, 12288),
]


def _layer(pkg, dev, shape, T, dtype=torch.bfloat16):
    E, k, r1, r3, r2, d_in, d_out = shape
    w = pkg.Workload("custom", T, d_in, d_out, E, k, r1, r3, r2, dtype, 91)
    params = pkg.synth.make_params(w, affine="random")
    m = pkg.TuckerMoE(w.d_in, w.d_out, w.cfg()).to(dev, w.dtype)
    m.load_state_dict({k_: v.to(dev) for k_, v in params.items()})
    return w, params, m, pkg.synth.make_x(w)


def _run(m, x):
    with torch.no_grad():
        got = m.forward_with_routing(x)
    torch.cuda.synchronize()
    return got


@pytest.mark.parametrize("T", [1, 16, 17, 33, 64])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_decode_fold(pkg, dev, shape, T):
    w, params, m, x = _layer(pkg, dev, shape, T)
    assert not m.plan().folded()
    decode = T > 32 or shape != SHAPES[6]
    assert (m.plan().forward_path(T) == pkg._lib.TMOE_PATH_DECODE) == decode
    assert m.plan().forward_path(65) != pkg._lib.TMOE_PATH_DECODE
    out, idx, wts, _ = _run(m, x.to(dev))
    m.check_signals()
    ref = onp.forward_f64(x, params, w.k)
    err = onp.rel_l2(out.float().cpu().numpy(), ref["out"])
    assert np.array_equal(idx.cpu().numpy(), ref["idx"])
    assert np.abs(wts.cpu().numpy() - ref["w"]).max() < 1e-5
    m.set_fold(False)
    assert m.plan().forward_path(T) == pkg._lib.TMOE_PATH_SMALL
    out2, idx2, _, _ = _run(m, x.to(dev))
    err2 = onp.rel_l2(out2.float().cpu().numpy(), ref["out"])
    print(f"{shape} T={T}: folded {err:.2e} two GEMMs {err2:.2e}", flush=True)
    assert torch.equal(idx, idx2) and err <= 1e-2 and err2 <= 1e-2
    if not decode:
        assert torch.equal(out, out2)
    # the errors of n outputs are known to 1 / sqrt(2 n) of themselves: four deviations of the
    # two forms' ratio, beside the tenth
    assert err <= (1.1 + 4 / out.numel() ** 0.5) * err2


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("T", [1, 16, 20, 64])
def test_decode_fold_capture(pkg, dev, dtype, T):
    """A captured forward (the kernel's two halves, a launch each) has the eager one's bits,
    routing outputs included, on every replay."""
    for shape in ((8, 2, 4, 256, 512, 768, 768), (8, 2, 4, 128, 256, 512, 1040),
                  (16, 3, 8, 64, 192, 256, 272)) + tuple(
            SHAPES[1:2] if dtype == torch.bfloat16 else ()):
        _, _, m, x = _layer(pkg, dev, shape, T, dtype)
        if m.plan().folded():
            shape = shape[:4] + (64,) + shape[5:]     # r2 of 64: not folded at other T
            _, _, m, x = _layer(pkg, dev, shape, T, dtype)
        assert not m.plan().folded()
        assert m.plan().forward_path(T) == pkg._lib.TMOE_PATH_DECODE
        xs = x.to(dev)
        ref = _run(m, xs)
        g = torch.cuda.CUDAGraph()
        with torch.no_grad(), torch.cuda.graph(g):
            got = m.forward_with_routing(xs)
        for _ in range(3):
            for t in got[:3]:
                t.zero_()
            g.replay()
            torch.cuda.synchronize()
            for a, b, c in zip(got[:3], ref[:3], _run(m, xs)[:3]):
                assert torch.equal(a, b) and torch.equal(c, b), (shape, T)


def test_decode_fold_fp8(pkg, dev):
    E, k, r1, r3, r2, d_in, d_out = (8, 2, 4, 256, 512, 768, 4608)
    w = pkg.Workload("custom", 48, d_in, d_out, E, k, r1, r3, r2, torch.bfloat16, 92, fp8=True)
    params, codes, ref = pkg.synth.make_fp8_params(w, affine="random")
    m = pkg.TuckerMoE(d_in, d_out, w.cfg()).to(dev, w.dtype)
    m.load_state_dict({k_: v.to(dev) for k_, v in params.items()})
    m.load_fp8(*(codes[n].to(dev) for n in ("U_in_q", "U_in_scale", "core_q", "core_scale",
                                            "U_out_q", "U_out_scale")))
    assert not m.plan().folded()
    assert m.plan().forward_path(48) == pkg._lib.TMOE_PATH_DECODE
    x = pkg.synth.make_x(w)
    out, idx, _, _ = _run(m, x.to(dev))
    want = onp.forward_f64(x, ref, k)
    assert np.array_equal(idx.cpu().numpy(), want["idx"])
    assert onp.rel_l2(out.float().cpu().numpy(), want["out"]) <= 1e-2


# fp32: one and two weight groups a wave (K 512 and 1024), the expert form, r3 = 64 with a K
# of 576 (groups that do not split evenly over the waves), ragged d_out
@pytest.mark.parametrize("T", [1, 15, 32, 33, 64])
@pytest.mark.parametrize("shape", [
    (8, 2, 4, 128, 256, 512, 1024), (16, 2, 4, 256, 1024, 1536, 2304),
    (8, 2, 32, 256, 512, 768, 768), (9, 3, 9, 64, 192, 320, 1040),
], ids=str)
def test_decode_fold_fp32(pkg, dev, shape, T):
    E, k, r1, r3, r2, d_in, d_out = shape
    w = pkg.Workload("custom", T, d_in, d_out, E, k, r1, r3, r2, torch.float32, 94)
    params = pkg.synth.make_params(w, affine="random")
    m = pkg.TuckerMoE(d_in, d_out, w.cfg()).to(dev, w.dtype)
    m.load_state_dict({k_: v.to(dev) for k_, v in params.items()})
    assert not m.plan().folded()
    assert m.plan().forward_path(T) == pkg._lib.TMOE_PATH_DECODE
    x = pkg.synth.make_x(w)
    out, idx, wts, _ = _run(m, x.to(dev))
    m.check_signals()
    ref = onp.forward_f64(x, params, w.k)
    err = onp.rel_l2(out.cpu().numpy(), ref["out"])
    m.set_fold(False)
    out2, idx2, wts2, _ = _run(m, x.to(dev))
    err2 = onp.rel_l2(out2.cpu().numpy(), ref["out"])
    print(f"{shape} T={T}: folded {err:.2e} two GEMMs {err2:.2e}", flush=True)
    assert np.array_equal(idx.cpu().numpy(), ref["idx"]) and torch.equal(idx, idx2)
    assert np.abs(wts.cpu().numpy() - ref["w"]).max() < 1e-5
    # W^T is summed in fp64: no further from exact than the two GEMMs, but for the few
    # elements of a single row (2304 values at most 10% apart by chance)
    assert err <= 1e-5 and err2 <= 1e-5 and err <= 1.1 * err2
