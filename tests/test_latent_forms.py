"""Which kernels FusedLatentMoE's sizes take (host-side rules, as on a 256-compute-unit
MI355X): the edges at which test_gpu_latent_grouped.py runs them."""
import pytest
import torch


def _form(pkg, B, E, k, r3, r2, backward, dtype=torch.bfloat16):
    return pkg._lib.lib().tmoe_latent_form(B, E, k, r3, r2, pkg._lib.dtype_code(dtype),
                                           int(backward))


# (E, k, r3, r2, B, forward by pairs, dx and dp by pairs, dG by expert)
@pytest.mark.parametrize("E,k,r3,r2,B,fwd,pairs,dg", [
    (8, 2, 256, 1024, 1109, 0, 0, 1), (8, 2, 256, 1024, 1110, 1, 1, 1),
    (16, 1, 256, 512, 90, 0, 0, 1), (16, 1, 256, 512, 91, 1, 1, 1),
    (64, 2, 128, 128, 5637, 0, 0, 1), (64, 2, 128, 128, 5638, 1, 1, 1),
    (16, 2, 128, 256, 1688, 0, 0, 1), (16, 2, 128, 256, 1689, 1, 1, 1),
    (16, 4, 256, 256, 16384, 0, 0, 1), (8, 6, 128, 128, 333, 0, 0, 1),
    (8, 7, 128, 128, 333, 0, 0, 0), (2, 2, 256, 1024, 4096, 0, 0, 0),
    (8, 2, 64, 1024, 4096, 0, 0, 0), (8, 2, 256, 192, 4096, 0, 0, 0),
    # many slots: by the columns, the tokens and the share of the experts
    (8, 4, 256, 128, 65536, 0, 0, 1), (8, 5, 256, 128, 8192, 0, 0, 1), (8, 5, 256, 128, 8193, 0, 0, 0),
    (8, 5, 256, 384, 8193, 0, 0, 0), (8, 5, 256, 512, 65536, 0, 0, 1), (16, 8, 128, 512, 65536, 0, 0, 1),
    (16, 9, 256, 1024, 2048, 0, 0, 0), (18, 9, 256, 1024, 2048, 0, 0, 1), (64, 16, 256, 128, 8193, 0, 0, 0),
    (64, 16, 256, 512, 8193, 0, 0, 1),
    # few experts and a full chip: dense forward, grouped backward
    (2, 1, 256, 1024, 16384, 0, 1, 1), (2, 1, 128, 512, 16384, 0, 1, 1),
    (3, 2, 256, 1024, 16384, 0, 1, 1), (3, 2, 128, 512, 32768, 0, 1, 1),
    (4, 2, 128, 512, 32768, 0, 1, 1), (2, 1, 256, 2048, 65536, 0, 1, 1),
    (2, 1, 128, 2048, 4572, 0, 1, 1), (2, 1, 256, 512, 21516, 0, 1, 1),
    (3, 1, 128, 1024, 16384, 0, 1, 1), (3, 1, 128, 2048, 65536, 0, 1, 1),
    (3, 1, 128, 2048, 50000, 1, 1, 1),
    (4, 2, 256, 1024, 8192, 1, 1, 1), (4, 1, 256, 1024, 32768, 1, 1, 1),
    (8, 2, 256, 1024, 16384, 1, 1, 1), (8, 2, 128, 512, 32768, 1, 1, 1),
])
def test_latent_forms(pkg, E, k, r3, r2, B, fwd, pairs, dg):
    f = pkg._lib
    assert _form(pkg, B, E, k, r3, r2, False) == (f.TMOE_LATENT_PAIRS if fwd else 0)
    assert _form(pkg, B, E, k, r3, r2, True) == ((f.TMOE_LATENT_PAIRS if pairs else 0) |
                                                 (f.TMOE_LATENT_DG if dg else 0))
    for backward in (False, True):
        assert _form(pkg, B, E, k, r3, r2, backward, torch.float32) == 0
        assert _form(pkg, 0, E, k, r3, r2, backward) == 0


def test_latent_form_rejects(pkg):
    assert _form(pkg, 64, 8, 9, 256, 1024, False) == pkg._lib.TMOE_EINVAL
    assert _form(pkg, 64, 65, 2, 256, 1024, True) == pkg._lib.TMOE_EUNSUPPORTED


def test_backward_workspace_follows_B(pkg):
    """The grouped dG's planes (one (r3, r2) fp32 plane per 256 entries and one per expert) are
    sized by the tokens, not by the chip: 1 MB each here."""
    f = pkg._lib.lib().tmoe_latent_workspace_bytes
    by_B = [f(B, 8, 256, 1024, pkg._lib.TMOE_BF16, 1) for B in (1, 64, 256, 1024, 4096, 16384)]
    assert by_B == sorted(by_B)
    assert by_B[0] < 9 << 20 and by_B[2] < 18 << 20   # 33 MB with the chip's 32 planes
    assert f(64, 2, 256, 1024, pkg._lib.TMOE_BF16, 1) < 5 << 20
