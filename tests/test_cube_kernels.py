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


@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("dist", ["uniform", "loguniform"])
def test_one_64_cube_equals_plane_passes(gpu, oracle, dist, in_place):
    """One 64^3 cube runs the plane plan with y split over the passes
    (plane_split.h): the same bits as the plane passes, which the drop-in call
    and a batch of two run, and the FP64 oracle within the FP32 bound."""
    import torch
    api = gpu.api
    n, P = 64, 64 ** 3
    print("case one 64^3 cube %s in_place=%s" % (dist, in_place), flush=True)
    gen = oracle.uniform if dist == "uniform" else oracle.loguniform
    sig, filt = gen(P, 43001), gen(P, 43002)
    api.set_plan(n, api.CF_PLAN_PLANE3)
    try:
        spec = gpu.Spectrum(n, torch.from_numpy(filt).cuda())
        plane = np.zeros_like(sig)
        assert gpu.fpgaf_conv3D(n, sig, filt, plane).valid
    finally:
        api.set_plan(n, api.CF_PLAN_AUTO)
    ds = torch.from_numpy(sig).cuda()
    two_in = torch.cat([ds, ds])
    two = torch.empty_like(two_in)
    gpu.conv3d_device(spec, two_in, two, 2, scale=api.CF_SCALE_NONE)
    out = ds if in_place else torch.full_like(ds, float("nan"))
    gpu.conv3d_device(spec, ds, out, scale=api.CF_SCALE_NONE)
    got = out.cpu().numpy()
    assert oracle.rel_l2(got, oracle.conv3d_f64(n, sig, filt)) <= 1e-5
    assert np.array_equal(got.view(np.uint32), plane.view(np.uint32))
    assert np.array_equal(got.view(np.uint32), two[:P].cpu().numpy().view(np.uint32))
