"""FusedLatentMoE grouped by expert (bf16, r3 and r2 multiples of 128, few of the experts
selected per token) against the float64 formulation, at the edges of its row tiles (128
tokens of one pair), chunks and dispatch rule, with experts nobody selects, one that
everybody does, repeated experts and indices outside [0, E). bf16 bar as in
test_gpu_latent.py: rel-L2 1e-2 (16-bit operands and outputs give about 2.3e-3)."""
import numpy as np
import pytest
import torch

from oracle import latent_np as ln
from oracle import tucker_moe_np as onp

pytestmark = pytest.mark.gpu


def _check(pkg, dev, x, G, idx, p, dout, forms=None):
    if forms is not None:   # the kernels of (forward, backward) this case is for
        f = pkg._lib
        sizes = (x.shape[0], G.shape[0], idx.shape[1], G.shape[1], G.shape[2], f.TMOE_BF16)
        assert (f.lib().tmoe_latent_form(*sizes, 0), f.lib().tmoe_latent_form(*sizes, 1)) == forms
    xs, Gs, ps = (t.to(dev).requires_grad_(True) for t in (x, G, p))
    out = pkg.FusedLatentMoE.apply(xs, Gs, idx.to(dev), ps)
    out.backward(dout.to(dev))
    torch.cuda.synchronize()
    valid = (idx >= 0) & (idx < G.shape[0])
    i0, p0 = torch.where(valid, idx, 0), torch.where(valid, p, torch.zeros_like(p))
    dx, dG, dp = ln.backward(x, G, i0, p0, dout)
    dp = np.where(valid.numpy(), dp, 0.0)
    ref = {"out": ln.forward(x, G, i0, p0), "dx": dx, "dG": dG, "dp": dp}
    got = {"out": out.detach(), "dx": xs.grad, "dG": Gs.grad, "dp": ps.grad}
    for n, v in got.items():
        v = v.float().cpu().numpy()
        assert np.isfinite(v).all(), n
        if not np.any(ref[n]):
            assert not np.any(v), n
            continue
        err = onp.rel_l2(v, ref[n])
        print(f"{n}={err:.2e}", end=" ", flush=True)
        assert err <= 1e-2, (n, err)
    return got


def _inputs(B, E, k, r3, r2, seed, p32):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(B, r3, generator=g).bfloat16()
    G = (torch.randn(E, r3, r2, generator=g) * r3 ** -0.5).bfloat16()
    v, idx = torch.topk(torch.randn(B, E, generator=g), k, dim=-1)
    p = torch.softmax(v, -1).to(torch.float32 if p32 else torch.bfloat16)
    return x, G, idx, p, torch.randn(B, r2, generator=g).bfloat16()


# (forward, backward) bits of tmoe_latent_form: dense but for dG; all grouped; none
DG, ALL, DENSE = (0, 2), (1, 3), (0, 0)


# (E, k, r3, r2, B): k = 2 pairs from B = 1110 on at E = 8 (the rule's first size and one
# below it), k = 1 from 91 at E = 16, 4 of 16 experts (dG alone grouped), one token,
# entries that do not fill a K tile, one tile of r2; the widest router (2080 pairs, most of
# them of a token or two) on both sides of its line and well past it; few experts, whose
# forward is dense where the backward is grouped
@pytest.mark.parametrize("E,k,r3,r2,B,forms", [
    (8, 2, 256, 1024, 1109, DG), (8, 2, 256, 1024, 1110, ALL), (8, 2, 128, 128, 2049, ALL),
    (16, 1, 256, 512, 90, DG), (16, 1, 256, 512, 91, ALL), (16, 1, 128, 384, 129, ALL),
    (16, 4, 256, 256, 1, DG), (16, 4, 256, 256, 65, DG), (64, 2, 128, 128, 4300, DG),
    (8, 6, 128, 128, 333, DG), (64, 2, 128, 128, 5637, DG), (64, 2, 128, 128, 5638, ALL),
    (64, 2, 128, 256, 8001, ALL), (64, 1, 128, 128, 4099, ALL),
    (8, 6, 128, 128, 8192, DG), (8, 6, 128, 128, 8193, DENSE), (16, 9, 128, 128, 700, DENSE),
])
@pytest.mark.parametrize("p32", [False, True], ids=["pbf16", "pf32"])
def test_grouped(pkg, dev, E, k, r3, r2, B, forms, p32):
    _check(pkg, dev, *_inputs(B, E, k, r3, r2, B + E, p32), forms=forms)


@pytest.mark.parametrize("kind", ["one", "repeat", "outside", "none"])
@pytest.mark.parametrize("B,E,k,forms", [
    (1500, 16, 1, ALL), (1500, 16, 2, DG), (1500, 16, 4, DG), (2000, 16, 2, ALL),
    (1400, 8, 2, ALL), (5700, 64, 2, ALL),
])
def test_grouped_odd_routing(pkg, dev, kind, B, E, k, forms):
    x, G, idx, p, dout = _inputs(B, E, k, 128, 256, 5, True)
    if kind == "one":              # every token the same expert first: one group of all
        idx = torch.where(idx == 3, idx[:, :1], idx)
        idx[:, 0] = 3
    elif kind == "repeat":         # a token that selects one expert k times
        idx[::3] = idx[::3, :1]
    elif kind == "outside":
        idx[::4, 0] = -1
        idx[1::4, k - 1] = E
        idx[2::8] = 1 << 40
    else:
        idx[:] = -5
    _check(pkg, dev, x, G, idx, p, dout, forms=forms)


def test_grouped_is_deterministic(pkg, dev):
    args = _inputs(3000, 8, 2, 256, 512, 9, True)
    a, b = _check(pkg, dev, *args), _check(pkg, dev, *args)
    for n in a:
        assert torch.equal(a[n], b[n]), n


@pytest.mark.parametrize("E,k,B", [(8, 6, 1), (8, 2, 63), (4, 2, 700), (16, 1, 300)])
def test_infinite_dout_stays_infinite(pkg, dev, E, k, B):
    """A column of dout that is infinite: positive x and p make dG infinite there for the experts
    that were selected, and nothing NaN (the rows that fill a chunk's last K tile add zeros)."""
    x, G, idx, p, dout = _inputs(B, E, k, 128, 256, 3, True)
    x = x.abs() + 0.125
    dout[:, 5] = float("inf")
    f = pkg._lib
    assert f.lib().tmoe_latent_form(B, E, k, 128, 256, f.TMOE_BF16, 1) & f.TMOE_LATENT_DG
    Gs = G.to(dev).requires_grad_(True)
    pkg.FusedLatentMoE.apply(x.to(dev), Gs, idx.to(dev), p.to(dev)).backward(dout.to(dev))
    dG = Gs.grad.float().cpu()
    used = torch.bincount(idx.flatten(), minlength=E) > 0
    assert not torch.isnan(dG).any()
    assert torch.isposinf(dG[used][:, :, 5]).all() and bool((dG[~used] == 0).all())
    rest = torch.cat((dG[:, :, :5], dG[:, :, 6:]), 2)
    assert torch.isfinite(rest).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_no_tokens(pkg, dev, dtype):
    x, idx, p = torch.zeros(0, 128), torch.zeros(0, 2, dtype=torch.int64), torch.zeros(0, 2)
    torch.full((1 << 20,), 7.0, device=dev)            # memory that the gradient may be given
    xs, Gs, ps = (t.to(dev, dtype).requires_grad_(True) for t in (x, torch.randn(8, 128, 256), p))
    out = pkg.FusedLatentMoE.apply(xs, Gs, idx.to(dev), ps)
    out.backward(torch.zeros_like(out))
    assert out.shape == (0, 256) and xs.grad.shape == (0, 128) and ps.grad.shape == (0, 2)
    assert bool((Gs.grad == 0).all())


@pytest.mark.parametrize("E,k,r3,r2,counts", [
    (5, 4, 128, 128, (257, 257, 257, 257, 260)),        # every expert a full chunk and a rest
    (8, 2, 128, 128, (1, 1, 1, 1, 1, 1, 1, 1)),         # rests only
    (8, 2, 256, 256, (4096, 1, 1, 1, 1, 1, 1, 2098)),   # few long ones
], ids=str)
def test_backward_stays_in_its_workspace(pkg, dev, E, k, r3, r2, counts):
    """Expert loads with the most dG chunks that the workspace's planes are counted for: the
    bytes past it stay as they were, dG is right."""
    f, n = pkg._lib, sum(counts)
    B = n // k
    assert B * k == n
    flat = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    idx = flat[torch.randperm(n, generator=torch.Generator().manual_seed(1))].reshape(B, k)
    x, G, _, _, dout = _inputs(B, E, k, r3, r2, 11, True)
    p = torch.rand(B, k, generator=torch.Generator().manual_seed(2))
    dt = f.TMOE_BF16 | f.TMOE_LATENT_P_F32
    L = f.lib()
    assert L.tmoe_latent_form(B, E, k, r3, r2, dt, 1) & f.TMOE_LATENT_DG
    nbytes = L.tmoe_latent_workspace_bytes(B, E, r3, r2, dt, 1)
    ws = torch.full((nbytes + 65536,), 0xA5, dtype=torch.uint8, device=dev)
    xs, Gs, i, ps, d = (t.to(dev) for t in (x, G, idx, p, dout))
    dx, dG, dp = torch.empty_like(xs), torch.empty_like(Gs), torch.empty_like(ps)
    f.check(L.tmoe_latent_backward(
        xs.data_ptr(), Gs.data_ptr(), i.data_ptr(), ps.data_ptr(), d.data_ptr(), B, E, k, r3, r2,
        dt, dx.data_ptr(), dG.data_ptr(), dp.data_ptr(), ws.data_ptr(), nbytes,
        torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert bool((ws[nbytes:] == 0xA5).all())
    for got, ref in zip((dx, dG, dp), ln.backward(x, G, idx, p, dout)):
        assert onp.rel_l2(got.float().cpu().numpy(), ref) <= 1e-2
