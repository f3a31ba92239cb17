"""The GLU epilogue on the 288-column out-projection tiles (bf16, d_out a multiple of 288)
against the plain out-projection and silu and product in torch, at the rows where the tiles
and the rule change: one round of 128-token tiles (its first and last T, ragged), 256-token
tiles in several rounds with a ragged last tile, the rounds at which the 192-column tiles
stay, K of one tile, the gate read from another tensor than `out` and in place."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# (E, k, r1, r3, r2, d_in, d_out): the reference's up projection, folded, K = 64. The folded
# one has 64 experts: with 32 or fewer the plain forward's large T goes in one launch, whose
# own front sums z in another order, so that y would not be the same out-projection's.
@pytest.mark.parametrize("shape,Ts", [
    ((8, 2, 32, 256, 512, 768, 4608), (1361, 1365, 1366, 1999, 2048, 2049, 4095, 4097, 6000, 8191)),
    ((64, 4, 4, 256, 1024, 768, 2304), (2731, 4000, 4097, 5400, 8100)),
    ((4, 1, 1, 64, 256, 256, 288), (21846, 32767, 43700, 65000)),
], ids=["reference", "folded", "k64"])
def test_glu_wide(pkg, dev, shape, Ts):
    E, k, r1, r3, r2, d_in, d_out = shape
    for T in Ts:
        w = pkg.Workload("custom", T, d_in, d_out, E, k, r1, r3, r2, torch.bfloat16, 77)
        m = pkg.TuckerMoE(w.d_in, w.d_out, w.cfg()).to(dev, w.dtype)
        m.load_state_dict({n: v.to(dev) for n, v in pkg.synth.make_params(w, affine="random").items()})
        x = pkg.synth.make_x(w).to(dev)
        g = torch.randn(T, d_out, device=dev).mul_(3).to(torch.bfloat16)
        g[0, :6] = torch.tensor([float("inf"), float("-inf"), 0.0, -0.0, 88.0, -300.0])
        with torch.no_grad():
            y = m(x)
            h = m.forward_raw(x, epi=pkg._lib.TMOE_EPI_GLU, epi_a=g)[0]
            inplace = g.clone()
            m.forward_raw(x, epi=pkg._lib.TMOE_EPI_GLU, epi_a=inplace, out=inplace)
        torch.cuda.synchronize()
        # y may come from tiles of another size: its K sum is the same up to fp32 order, so
        # R(y) one unit (2^-8) apart; silu one unit apart (its last fp32 places), each product
        # rounded: 2^-8 (1 + 1 + 1/2 + 1/2)
        s = g.float() / (1 + torch.exp(-g.float()))   # NaN at -inf, as torch's silu
        want = s.to(torch.bfloat16).float() * y.float()
        ok = ((h.float() - want).abs() <= 3 * 2.0 ** -8 * want.abs() + 1e-30) | (h.float() == want) \
            | (h.isnan() & want.isnan())
        print(f"T={T}: {(h != want.to(torch.bfloat16)).float().mean():.1e}", end=" ", flush=True)
        assert bool(ok.all()), (T, (~ok).nonzero()[:4].tolist())
        assert torch.equal(h.view(torch.int16), inplace.view(torch.int16)), T
