"""Spectra made in memory that an earlier, destroyed spectrum of the same size
used: the convolutions still queued with the old one, on the same or on another
stream, keep its values, and the kept memory is bounded."""
import pytest

pytestmark = pytest.mark.gpu


def _bits(x):
    import torch
    return torch.view_as_real(x).view(torch.int32)


@pytest.mark.parametrize("n", [32, 128, 256])
@pytest.mark.parametrize("other_stream", [False, True])
def test_new_spectrum_waits_for_the_old_one(gpu, n, other_stream):
    import torch
    api = gpu.api
    print("case spectrum reuse N=%d other_stream=%s" % (n, other_stream), flush=True)
    P, rounds = n ** 3, 6
    filt = torch.empty((rounds, P), dtype=torch.complex64, device="cuda")
    sig = torch.empty(P, dtype=torch.complex64, device="cuda")
    api.fill_uniform(filt, 2 * filt.numel(), 64001 + n)
    api.fill_uniform(sig, 2 * P, 64002 + n)
    keep = [gpu.Spectrum(n, filt[k]) for k in range(rounds)]
    want = torch.empty_like(filt)
    for k in range(rounds):
        gpu.conv3d_device(keep[k], sig, want[k])
    torch.cuda.synchronize()
    for s in keep:
        s.close()
    out = torch.empty_like(filt)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    for k in range(rounds):  # each closed with its convolution still queued
        st = streams[k % 2 if other_stream else 0]
        spec = gpu.Spectrum(n, filt[k], stream=st)
        gpu.conv3d_device(spec, sig, out[k], stream=st)
        spec.close()
    torch.cuda.synchronize()
    assert torch.equal(_bits(out), _bits(want))


def test_kept_memory_is_bounded(gpu):
    import torch
    n, count = 256, 2
    print("case spectrum memory bound", flush=True)
    filt = torch.zeros((count, n ** 3), dtype=torch.complex64, device="cuda")
    torch.cuda.synchronize()
    gpu.Spectrum(n, filt, count).close()  # (workspace and tables are there)
    free0 = torch.cuda.mem_get_info()[0]
    specs = [gpu.Spectrum(n, filt, count) for _ in range(8)]  # 2 GiB
    for s in specs:
        s.close()
    assert free0 - torch.cuda.mem_get_info()[0] <= 1 << 30


@pytest.mark.parametrize("n,count", [(64, 37), (128, 5), (256, 3)])
@pytest.mark.parametrize("other_stream", [False, True])
def test_old_spectrum_is_read_while_the_next_is_made(gpu, n, count, other_stream):
    """The only kept block of a size is that of a spectrum whose convolutions are
    still queued when the next spectrum of the size is made, on the same or on
    another stream: the last of them, which runs after that, has the old values.
    (Five passes without a workspace, which would order the streams.)"""
    import torch
    api = gpu.api
    print("case spectrum read N=%d count=%d other_stream=%s" % (n, count, other_stream), flush=True)
    gpu.fpga_final()  # nothing is kept: closing a fifth spectrum would free the oldest one, and wait
    assert gpu.fpga_initialize("gfx950", gpu.CODE_OBJECT, True) == 0
    api.set_plan(n, api.CF_PLAN_AXIS5)
    try:
        filt = torch.empty((2, count, n ** 3), dtype=torch.complex64, device="cuda")
        sig = torch.empty((count, n ** 3), dtype=torch.complex64, device="cuda")
        api.fill_uniform(filt, 2 * filt.numel(), 67001 + n)
        api.fill_uniform(sig, 2 * sig.numel(), 67002 + n)
        want, out = torch.empty_like(filt), torch.empty_like(filt)
        for k in range(2):
            spec = gpu.Spectrum(n, filt[k], count)
            gpu.conv3d_device(spec, sig, want[k], count)
            spec.data_ptr()  # the address is taken: freed, not kept
            spec.close()
        a = torch.cuda.Stream()
        b = torch.cuda.Stream() if other_stream else a
        torch.cuda.synchronize()
        old = gpu.Spectrum(n, filt[0], count, stream=a)
        for _ in range(200):
            gpu.conv3d_device(old, sig, out[0], count, stream=a)
        queued = torch.cuda.Event()
        queued.record(a)
        old.close()
        new = gpu.Spectrum(n, filt[1], count, stream=b)
        assert not other_stream or not queued.query()
        gpu.conv3d_device(new, sig, out[1], count, stream=b)
        torch.cuda.synchronize()
        new.close()
    finally:
        api.set_plan(n, api.CF_PLAN_AUTO)
    assert torch.equal(_bits(out), _bits(want))


def test_kept_memory_is_given_back(gpu):
    """trim() leaves neither destroyed spectra nor transform workspaces; both are
    made again."""
    import torch
    n = 256
    print("case trim", flush=True)
    x = torch.empty((2, n ** 3), dtype=torch.complex64, device="cuda")
    gpu.api.fill_uniform(x, 2 * x.numel(), 68001)
    want, out = torch.empty_like(x), torch.empty_like(x)

    def calls(y):
        gpu.fft3d_device(n, x[0], y[0])
        spec = gpu.Spectrum(n, x[1])
        gpu.conv3d_device(spec, x[0], y[1])
        spec.close()
    calls(want)
    gpu.api.trim()
    free0 = torch.cuda.mem_get_info()[0]
    calls(out)
    kept = torch.cuda.mem_get_info()[0]
    gpu.api.trim()
    assert free0 - kept >= 2 * 8 * n ** 3 and torch.cuda.mem_get_info()[0] >= free0
    assert torch.equal(_bits(out), _bits(want))
