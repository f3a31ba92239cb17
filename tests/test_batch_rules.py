"""Which forms batches of up to 256 tokens take (host-side rules, as on a 256-compute-unit
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


# a folded plan takes the batch form (d_out, K = r1 r3, T): in one round of the skinny
# out-projection's work-groups not, unless K is past 1024; in two rounds with one K slice, or
# from 16 tokens in the last block of 64 on (32 where K is short and the second round few), or
# where the blocks before it fill the chip
@pytest.mark.parametrize("d_out,r1,r3,T,batch", [
    (768, 4, 256, 65, False), (768, 4, 256, 256, False), (1024, 4, 256, 256, False),
    (1040, 4, 256, 256, True), (1040, 4, 256, 192, False), (1040, 4, 256, 207, False),
    (1040, 4, 256, 208, True), (2048, 4, 256, 128, False), (2064, 4, 256, 79, False),
    (2064, 4, 256, 80, True), (4080, 4, 256, 65, False), (4096, 4, 256, 65, True),
    (768, 2, 256, 128, False), (768, 4, 128, 128, False), (768, 1, 256, 65, False),
    (768, 4, 64, 256, False), (1040, 4, 64, 256, True), (2048, 1, 256, 65, False),
    (2064, 1, 256, 65, True), (2064, 6, 64, 65, True), (2064, 2, 256, 95, False),
    (2064, 2, 256, 96, True), (2304, 3, 256, 95, False), (2544, 3, 256, 95, False),
    (2560, 3, 256, 80, True), (2560, 3, 256, 79, False), (4096, 2, 256, 65, True),
])
def test_folded_plan_batches(pkg, d_out, r1, r3, T, batch):
    f = pkg._lib
    got = _form(pkg, T, d_in=768, d_out=d_out, r1=r1, r3=r3)
    assert got & f.TMOE_FORM_FOLDED and bool(got & f.TMOE_FORM_BATCH) == batch
    # behind a sliced front, and past K of 1024
    assert _form(pkg, T, d_in=1536, d_out=d_out, r1=r1, r3=r3) & f.TMOE_FORM_BATCH
    assert not _form(pkg, 64, d_in=768, d_out=d_out, r1=r1, r3=r3) & f.TMOE_FORM_BATCH
    assert not _form(pkg, 257, d_in=768, d_out=d_out, r1=r1, r3=r3) & f.TMOE_FORM_BATCH


def test_other_batches(pkg):
    """K past 1024 of a folded plan; unfolded plans up to 256 tiles of 64 x 128; fp32 and
    NO_FOLD never."""
    f = pkg._lib
    both = f.TMOE_FORM_FOLDED | f.TMOE_FORM_BATCH
    assert _form(pkg, 65, d_in=768, d_out=64, r1=32, r2=512) == both     # folded, K 2048
    for T in (65, 193, 256):
        assert _form(pkg, T, d_in=768, d_out=768, r1=32, r2=512) == both
        assert _form(pkg, T, d_in=768, d_out=768, r1=32, r2=512, dtype=torch.float32) == 0
        assert _form(pkg, T, d_in=768, d_out=768, r1=32, r2=512, flags=f.TMOE_FLAG_NO_FOLD) == 0
    shape = dict(d_in=256, d_out=10880, r1=8, r2=64, r3=64)
    assert _form(pkg, 192, **shape) == both and _form(pkg, 193, **shape) == 0
    assert _form(pkg, 32, **shape) == f.TMOE_FORM_FOLDED and _form(pkg, 0, **shape) == 0
    assert _form(pkg, 64, **shape) == 0


# plans that are not folded otherwise, by rounds of 4096 columns: (d_in, r1, r3, r2, d_out, dtype)
# and the T of 16, 17, 32, 33, 64 that run folded
BF, F32 = torch.bfloat16, torch.float32
ALL, UP32, FROM33, MID, FROM17 = (16, 17, 32, 33, 64), (16, 17, 32), (33, 64), (17, 32), (17, 32, 33, 64)


@pytest.mark.parametrize("d_in,r1,r3,r2,d_out,dtype,folded", [
    (768, 8, 256, 64, 4096, BF, ALL), (128, 2, 256, 256, 4096, F32, ALL),        # one round
    (768, 8, 256, 512, 6144, BF, ALL), (768, 8, 256, 256, 8192, BF, FROM33),     # two: W^T's extra bytes
    (768, 8, 256, 512, 8192, BF, FROM33), (768, 8, 256, 1024, 8192, BF, ALL),
    (768, 4, 256, 512, 8192, BF, ALL), (768, 16, 128, 512, 8192, BF, ALL),
    (768, 2, 256, 256, 8192, BF, UP32), (768, 2, 256, 256, 6144, BF, ALL),       # two: a short core
    (1024, 2, 256, 256, 8192, BF, ALL), (448, 2, 256, 256, 6144, BF, UP32),
    (448, 4, 256, 256, 4112, BF, UP32), (448, 4, 256, 512, 8192, BF, ALL), (128, 2, 128, 256, 8192, BF, ALL),
    (768, 2, 256, 256, 8192, F32, ALL), (448, 2, 256, 256, 8192, F32, UP32),
    (448, 2, 256, 256, 6144, F32, ALL), (768, 1, 256, 64, 8192, F32, UP32),
    (768, 4, 256, 512, 9216, BF, UP32), (768, 4, 256, 512, 12288, BF, UP32),     # three
    (768, 4, 256, 256, 9216, BF, ()), (768, 4, 256, 512, 8208, F32, ()),
    (768, 4, 128, 256, 12288, BF, ALL), (448, 4, 128, 256, 12288, BF, UP32),
    (768, 4, 128, 64, 9216, BF, MID), (768, 8, 64, 64, 9216, BF, MID), (1024, 8, 64, 64, 9216, BF, FROM17),
    (768, 16, 64, 256, 12288, BF, FROM17),
    (768, 4, 256, 512, 12304, BF, ()), (768, 2, 256, 256, 16384, BF, ()),        # four
])
def test_decode_forms(pkg, d_in, r1, r3, r2, d_out, dtype, folded):
    f = pkg._lib
    for T in ALL:
        got = _form(pkg, T, d_in=d_in, d_out=d_out, E=16, r1=r1, r3=r3, r2=r2, dtype=dtype)
        assert got == (f.TMOE_FORM_FOLDED if T in folded else 0), T


@pytest.mark.parametrize("d_out,dtype,packed", [
    (12288, F32, False), (4096, F32, True), (16384, BF, True), (16400, BF, False),
])
def test_wt_only_where_some_batch_reads_it(pkg, d_out, dtype, packed):
    """W^T beside the two-GEMM weights: in bf16 also for batches past 64 tokens alone."""
    args = (768, d_out, 16, 2, 2, 256, 256, dtype, 1e-5)
    extra = (pkg._lib.Plan(*args).packed_bytes() -
             pkg._lib.Plan(*args, flags=pkg._lib.TMOE_FLAG_NO_FOLD).packed_bytes())
    assert extra == (512 * d_out * (2 if dtype == BF else 4) if packed else 0)
    assert not pkg._lib.Plan(*args).folded()
