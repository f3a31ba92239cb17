"""fp32 layers at 256 < T <= 4096: the K-sliced front over 32-token tiles, the core in K
slices of 64 x 64 tiles and the out-projection's three tile sizes, against the float64
oracle (rel-L2 1e-5: sums of at most 2048 fp32 products, measured 1e-6) and against the
separate launches (bit-identical: the same slices in the same order)."""
import numpy as np
import pytest
import torch

from oracle import tucker_moe_np as onp

pytestmark = pytest.mark.gpu


def _layer(pkg, dev, shape, T, seed=90):
    E, k, r1, r3, r2, d_in, d_out = shape
    w = pkg.Workload("custom", T, d_in, d_out, E, k, r1, r3, r2, torch.float32, seed)
    params = pkg.synth.make_params(w, affine="random")
    m = pkg.TuckerMoE(w.d_in, w.d_out, w.cfg()).to(dev, w.dtype)
    m.load_state_dict({k_: v.to(dev) for k_, v in params.items()})
    return w, params, m, pkg.synth.make_x(w)


def _forward(m, x):
    with torch.no_grad():
        got = m.forward_with_routing(x, logits=True)
    torch.cuda.synchronize()
    return got


# (E, k, r1, r3, r2, d_in, d_out): d_in of 16 K tiles (the first sliced one) and of 15 (not
# sliced); the expert form (E < r1) with 8 core slices and r2 of one tile; a router of 100
# columns; ragged column tiles of both GEMMs; the last T of the core's 64 x 64 tiles and the
# first of its 128 x 128 ones
@pytest.mark.parametrize("shape,T", [
    ((8, 2, 32, 256, 512, 1536, 1008), 257), ((8, 2, 32, 256, 512, 1536, 1008), 1021),
    ((16, 2, 4, 256, 192, 512, 208), 300), ((16, 2, 4, 256, 192, 576, 208), 288),
    ((8, 2, 4, 64, 64, 448, 64), 1000), ((100, 4, 8, 128, 320, 512, 656), 2049),
    ((8, 2, 4, 64, 64, 512, 16), 4096), ((4, 1, 2, 128, 1024, 640, 2304), 4097),
    ((4, 1, 2, 128, 1024, 640, 272), 3072), ((4, 1, 2, 128, 1024, 640, 272), 3073),
], ids=lambda v: str(v))
def test_fp32_mid(pkg, dev, shape, T):
    w, params, m, x = _layer(pkg, dev, shape, T)
    out, idx, wts, lg = _forward(m, x.to(dev))
    m.check_signals()
    ref = onp.forward_f64(x, params, w.k)
    err = onp.rel_l2(out.cpu().numpy(), ref["out"])
    lerr = onp.rel_l2(lg.cpu().numpy(), ref["logits"])
    print(f"{shape} T={T}: out {err:.2e} logits {lerr:.2e}", flush=True)
    assert np.array_equal(idx.cpu().numpy(), ref["idx"])
    assert err <= 1e-5 and lerr <= 1e-6
    m.set_fuse(False)
    for a, b in zip((out, idx, wts, lg), _forward(m, x.to(dev))):
        assert torch.equal(a, b)


def test_fp32_mid_capture(pkg, dev):
    _, _, m, x = _layer(pkg, dev, (8, 2, 32, 256, 512, 768, 768), 700)
    xs = x.to(dev)
    ref = _forward(m, xs)[0]
    g = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(g):
        out = m(xs)
    for _ in range(3):
        out.zero_()
        g.replay()
        assert torch.equal(out, ref)
        assert torch.equal(_forward(m, xs)[0], ref)


def test_fp32_static_without_slices(pkg, dev):
    """A T whose planes do not fit the static scratch runs there without them."""
    T = 4096
    w, params, m, x = _layer(pkg, dev, (8, 2, 4, 256, 2304, 512, 64), T)
    L, plan, packed = pkg._lib.lib(), m.plan(), m.packed()
    assert plan.workspace_bytes(T) > L.tmoe_static_scratch_bytes()
    xs, out = x.to(dev), torch.empty(T, 64, device=dev)
    pkg._lib.check(L.tmoe_forward_static(plan.ptr, xs.data_ptr(), T, packed.data_ptr(),
                                         out.data_ptr(), None, None, None,
                                         torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert onp.rel_l2(out.cpu().numpy(), onp.forward_f64(x, params, w.k)["out"]) <= 1e-5
