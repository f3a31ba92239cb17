"""Host-side limits of the fp32 plans' workspace: its K slices' planes take no T from
tmoe_forward_static that fits the static scratch without them."""
import torch


def test_static_accepts_what_fits_without_planes(pkg):
    L = pkg._lib.lib()
    plan = pkg._lib.Plan(512, 64, 8, 2, 4, 2304, 256, torch.float32, 1e-5)
    cap = L.tmoe_static_scratch_bytes()
    T = 4096
    assert plan.workspace_bytes(T) > cap
    if torch.cuda.is_available():
        return
    # past the size checks: without a GPU the scratch lookup fails (-3), not the size (-2)
    assert L.tmoe_forward_static(plan.ptr, 16, T, 16, 16, None, None, None, None) == -3
    assert L.tmoe_forward_static(plan.ptr, 16, 2 * T, 16, 16, None, None, None, None) == -2
