"""Which forms batches of 65 to 256 tokens take (host-side rules, as on a 256-compute-unit
MI355X)."""
import pytest
import torch


def _form(pkg, T, d_in=1536, d_out=2304, E=8, k=2, r1=4, r2=1024, r3=256, dtype=torch.bfloat16,
          flags=0):
    plan = pkg._lib.Plan(d_in, d_out, E, k, r1, r2, r3, dtype, 1e-5, flags=flags)
    return plan.forward_form(T)


# the front's K slices from 24 K tiles of 64 on, from 40 with more than 64 experts; larger T
# from 16 on
@pytest.mark.parametrize("E,d_in,sliced", [
    (8, 1024, False), (8, 1472, False), (8, 1536, True), (32, 1472, False), (32, 1536, True),
    (64, 1472, False), (64, 1536, True), (65, 1536, False), (128, 2496, False),
    (128, 2560, True), (256, 3072, False),
])
def test_batch_front_slices(pkg, E, d_in, sliced):
    S = pkg._lib.TMOE_FORM_FRONT_SLICED
    for T in (65, 128, 200, 256):
        assert bool(_form(pkg, T, d_in=d_in, d_out=4096, E=E) & S) == sliced, T
    assert bool(_form(pkg, 257, d_in=d_in, d_out=4096, E=E) & S) == (E <= 128)
    assert not _form(pkg, 64, d_in=d_in, d_out=4096, E=E) & S
