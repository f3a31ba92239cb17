"""A workspace sized for one T serves a smaller T whose fastest form would want more
(host-side checks; the GPU tests run such forwards in test_gpu_workspace_fit.py)."""
import pytest
import torch

# (plan: d_in, d_out, E, k, r1, r2, r3; dtype; T the workspace is sized for; T's that it serves)
CASES = [
    ((1536, 6144, 8, 2, 32, 512, 256), torch.float32, 4097, (257, 1021, 2048, 3000, 4096)),
    ((512, 1024, 8, 2, 4, 256, 128), torch.bfloat16, 2048, (65, 128, 256)),
    ((768, 768, 8, 2, 32, 512, 256), torch.bfloat16, 700, (65, 193, 256)),
]


def _rc(L, plan, T, nbytes):
    """tmoe_forward's return code with stand-in addresses: without a GPU a workspace that
    passes the size check ends in the first launch's error (-3)."""
    a = 4096
    return L.tmoe_forward(plan.ptr, a, T, a, a, None, None, None, a, nbytes, None)


@pytest.mark.skipif(torch.cuda.is_available(), reason="stand-in addresses: host checks only")
@pytest.mark.parametrize("shape,dtype,sized,Ts", CASES, ids=lambda v: str(v))
def test_smaller_T_is_served(pkg, shape, dtype, sized, Ts):
    L = pkg._lib.lib()
    plan = pkg._lib.Plan(*shape, dtype, 1e-5)
    nbytes = plan.workspace_bytes(sized)
    assert any(plan.workspace_bytes(T) > nbytes for T in Ts)
    for T in Ts:
        assert _rc(L, plan, T, nbytes) == pkg._lib.TMOE_EHIP, (T, L.tmoe_last_error())
        assert L.tmoe_forward_glu(plan.ptr, 4096, T, 4096, 4096, 4096, 4096, 8192, nbytes,
                                  None) == pkg._lib.TMOE_EHIP
        # z alone: too small for any form
        z_bytes = T * shape[6] * (4 if dtype is torch.float32 else 2)
        assert _rc(L, plan, T, z_bytes) == pkg._lib.TMOE_EINVAL
