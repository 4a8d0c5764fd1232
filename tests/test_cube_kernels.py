"""Whole-cube kernels of edges 8 and 16 (convfpga_amd/csrc/kernels/small_cube.h):
against the FP64 oracle at the FP32 bound, and bitwise against the axis passes,
which run the same line transforms in the same order (the drop-in call, which
reports its halves separately, still runs them)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("own,in_place", [(False, False), (True, False), (True, True)])
@pytest.mark.parametrize("count", [1, 7])
@pytest.mark.parametrize("n", [8, 16])
def test_cube_conv(gpu, oracle, n, count, own, in_place):
    import torch
    api = gpu.api
    P = n ** 3
    print("case cube conv N=%d count=%d own=%s in_place=%s" % (n, count, own, in_place), flush=True)
    sig = oracle.uniform(count * P, 41000 + n + count)
    filt = oracle.uniform((count if own else 1) * P, 42000 + n)
    spec = gpu.Spectrum(n, torch.from_numpy(filt).cuda(), count if own else 1)
    ds = torch.from_numpy(sig).cuda()
    out = ds if in_place else torch.full_like(ds, float("nan"))
    gpu.conv3d_device(spec, ds, out, count, scale=api.CF_SCALE_NONE)
    got = out.cpu().numpy()
    for k in range(count):
        s = np.ascontiguousarray(sig[k * P:(k + 1) * P])
        f = np.ascontiguousarray(filt[k * P:(k + 1) * P] if own else filt)
        assert oracle.rel_l2(np.ascontiguousarray(got[k * P:(k + 1) * P]), oracle.conv3d_f64(n, s, f)) <= 1e-5
        axis = np.zeros_like(s)
        assert gpu.fpgaf_conv3D(n, s, f, axis).valid
        assert np.array_equal(got[k * P:(k + 1) * P].view(np.uint32), axis.view(np.uint32))
