"""Forwards in a workspace sized for a larger T, which holds only the smaller form of their
own (tmoe_workspace_bytes): against the float64 oracle, fp32 at rel-L2 1e-5 (sums of at most
2048 fp32 products) and bf16 at 1e-2, with the bytes past the workspace untouched."""
import numpy as np
import pytest
import torch

from oracle import tucker_moe_np as onp
from test_workspace_fit import CASES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,dtype,sized,Ts", CASES, ids=lambda v: str(v))
def test_runs_in_a_larger_T_workspace(pkg, dev, shape, dtype, sized, Ts):
    d_in, d_out, E, k, r1, r2, r3 = shape
    L = pkg._lib.lib()
    for T in Ts:
        w = pkg.Workload("custom", T, d_in, d_out, E, k, r1, r3, r2, dtype, 95)
        params = pkg.synth.make_params(w, affine="random")
        m = pkg.TuckerMoE(d_in, d_out, w.cfg()).to(dev, dtype)
        m.load_state_dict({n: v.to(dev) for n, v in params.items()})
        plan, packed = m.plan(), m.packed()
        nbytes, guard = plan.workspace_bytes(sized), 4096
        x = pkg.synth.make_x(w)
        xs, out = x.to(dev), torch.empty(T, d_out, dtype=dtype, device=dev)
        idx = torch.empty(T, k, dtype=torch.int32, device=dev)
        ws = torch.full((nbytes + guard,), 0xA5, dtype=torch.uint8, device=dev)
        pkg._lib.check(L.tmoe_forward(plan.ptr, xs.data_ptr(), T, packed.data_ptr(),
                                      out.data_ptr(), idx.data_ptr(), None, None, ws.data_ptr(),
                                      nbytes, torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        ref = onp.forward_f64(x, params, k)
        err = onp.rel_l2(out.float().cpu().numpy(), ref["out"])
        print(f"T={T}: {err:.2e}", end=" ", flush=True)
        assert bool((ws[nbytes:] == 0xA5).all())
        assert np.array_equal(idx.cpu().numpy(), ref["idx"])
        assert err <= (1e-5 if dtype is torch.float32 else 1e-2)
