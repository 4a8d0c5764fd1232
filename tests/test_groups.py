"""Batches whose cubes go through the passes in groups (pass_group, engine.cpp):
each cube's result is, bit for bit, that of a call on the cube alone, whatever
the group it falls in, for counts around the points where the grouping changes."""
import pytest

pytestmark = pytest.mark.gpu


def _same(a, b):
    import torch
    torch.cuda.synchronize()
    return torch.equal(torch.view_as_real(a).view(torch.int32), torch.view_as_real(b).view(torch.int32))


# the largest groups: 8 (own filters) and 9 (one filter) cubes of 128^3, 72 and 88 of
# 64^3, 1 of 256^3
@pytest.mark.parametrize("n,count", [(128, 9), (128, 10), (128, 15), (128, 17), (64, 73), (64, 89), (64, 130), (256, 2),
                                     (256, 3)])
@pytest.mark.parametrize("in_place", [False, True])
def test_groups_equal_single_cubes(gpu, n, count, in_place):
    import torch
    api = gpu.api
    print("case groups N=%d count=%d in_place=%s" % (n, count, in_place), flush=True)
    P = n ** 3
    sig = torch.empty((count, P), dtype=torch.complex64, device="cuda")
    filt = torch.empty_like(sig)
    api.fill_uniform(sig, 2 * sig.numel(), 61000 + n + count)
    api.fill_uniform(filt, 2 * filt.numel(), 62000 + n + count)
    own, shared = gpu.Spectrum(n, filt, count), gpu.Spectrum(n, filt)
    tr = torch.empty_like(sig)
    gpu.fft3d_device(n, sig, tr, count, inverse=in_place)
    out, out_sh = (sig.clone(), sig.clone()) if in_place else (torch.empty_like(sig), torch.empty_like(sig))
    gpu.conv3d_device(own, out if in_place else sig, out, count)
    gpu.conv3d_device(shared, out_sh if in_place else sig, out_sh, count)
    batch_out = torch.empty_like(sig)
    views = [own.view(k) for k in range(count)]
    batch = api.Batch([(sig[k], batch_out[k], views[k]) for k in range(count)], mode=api.CF_BATCH_GRAPH)
    batch.launch()
    batch.check()
    one = torch.empty_like(sig[0])
    for k in range(count):
        alone = gpu.Spectrum(n, filt[k])
        gpu.conv3d_device(alone, sig[k], one)
        assert _same(one, out[k]) and _same(one, batch_out[k]), k
        gpu.conv3d_device(shared, sig[k], one)
        assert _same(one, out_sh[k]), k
        gpu.fft3d_device(n, sig[k], one, inverse=in_place)
        assert _same(one, tr[k]), k
        alone.close()
    batch.close()


def test_timed_and_profiled_calls_run_the_groups(gpu):
    """cf_conv3d_device_timed and cf_profile_* sum a pass over the groups of a
    call: the bytes of 17 single cubes, the same output."""
    import torch
    api = gpu.api
    n, count = 128, 17
    print("case timed groups N=%d count=%d" % (n, count), flush=True)
    sig = torch.empty((count, n ** 3), dtype=torch.complex64, device="cuda")
    api.fill_uniform(sig, 2 * sig.numel(), 63001)
    spec = gpu.Spectrum(n, sig, count)
    alone = gpu.Spectrum(n, sig[0])
    want, out = torch.empty_like(sig), torch.empty_like(sig)
    gpu.conv3d_device(spec, sig, want, count)
    one = gpu.conv3d_device_timed(alone, sig[0], out[0])
    many = gpu.conv3d_device_timed(spec, sig, out, count)
    assert _same(out, want)
    assert [p["name"] for p in many] == [p["name"] for p in one]
    assert all(m["bytes"] == count * o["bytes"] and m["ms"] > o["ms"] > 0 for m, o in zip(many, one))
    out.zero_()
    api.profile_begin(4, 2)
    for _ in range(5):
        gpu.conv3d_device(spec, sig, out, count)
    passes, calls = api.profile_end()
    assert calls == 2 and _same(out, want)
    assert all(p["bytes"] == m["bytes"] and p["ms"] > 0 for p, m in zip(passes, many))


@pytest.mark.parametrize("n", [16, 64, 128])
@pytest.mark.parametrize("step", [1, 2, -1])
def test_graph_keeps_order_along_one_buffer(gpu, n, step):
    """Graph instances whose signals and outputs follow each other in one buffer,
    the output `step` cubes behind the signal: each reads what an earlier one
    wrote (or writes what an earlier one has read), in the given order."""
    import torch
    api = gpu.api
    print("case graph chain N=%d step=%d" % (n, step), flush=True)
    P, count = n ** 3, 5
    lead = max(0, -step)
    buf = torch.empty((count + abs(step), P), dtype=torch.complex64, device="cuda")
    api.fill_uniform(buf, 2 * buf.numel(), 65001 + n)
    filt = torch.empty(P, dtype=torch.complex64, device="cuda")
    api.fill_uniform(filt, 2 * P, 65002 + n)
    spec = gpu.Spectrum(n, filt)
    want = buf.clone()
    for k in range(count):
        gpu.conv3d_device(spec, want[lead + k], want[lead + k + step])
    batch = api.Batch([(buf[lead + k], buf[lead + k + step], spec) for k in range(count)], mode=api.CF_BATCH_GRAPH)
    batch.launch()
    batch.check()
    batch.close()
    assert _same(buf, want)


@pytest.mark.parametrize("n32,n64", [(1, 1), (16, 8), (5, 3), (1, 9), (40, 1), (513, 2), (3, 65)])
@pytest.mark.parametrize("first", [32, 64])
@pytest.mark.parametrize("in_place", [False, True])
def test_graph_pairs_32_and_64(gpu, n32, n64, first, in_place):
    """A 32^3 and a 64^3 run next to each other share their launches (run_pair,
    engine.cpp), up to a group of each (512 and 64 cubes; one more and they run by
    themselves): the bits of calls on the cubes alone, one filter each or shared."""
    import torch
    api = gpu.api
    print("case pair 32:%d 64:%d first=%d in_place=%s" % (n32, n64, first, in_place), flush=True)
    inst, want = [], []
    for n, count in ((32, n32), (64, n64))[:: 1 if first == 32 else -1]:
        sig = torch.empty((count, n ** 3), dtype=torch.complex64, device="cuda")
        filt = torch.empty_like(sig)
        api.fill_uniform(sig, 2 * sig.numel(), 64000 + n + count)
        api.fill_uniform(filt, 2 * filt.numel(), 65000 + n + count)
        spec = gpu.Spectrum(n, filt, count if n == 32 else 1)
        ref = torch.empty_like(sig)
        gpu.conv3d_device(spec, sig, ref, count)
        out = sig if in_place else torch.zeros_like(sig)
        inst += [(sig[k], out[k], spec.view(k) if n == 32 else spec) for k in range(count)]
        want.append((out, ref))
    batch = api.Batch(inst, mode=api.CF_BATCH_GRAPH)
    batch.launch()
    batch.check()
    for out, ref in want:
        assert _same(out, ref)
    if not in_place:
        for _ in range(2):
            for out, _ref in want:
                out.zero_()
            batch.launch()
            for out, ref in want:
                assert _same(out, ref)
    batch.close()


@pytest.mark.parametrize("overlap", ["out_sig", "out_out", "sig_out"])
def test_graph_pair_keeps_order(gpu, overlap):
    """A 64^3 and a 32^3 instance that meet in memory run one after the other."""
    import torch
    api = gpu.api
    print("case pair order %s" % overlap, flush=True)
    a, c = 64 ** 3, 32 ** 3
    buf = torch.empty(4 * a, dtype=torch.complex64, device="cuda")
    big, small = torch.empty(a, dtype=torch.complex64, device="cuda"), torch.empty(c, dtype=torch.complex64, device="cuda")
    for k, t in enumerate((buf, big, small)):
        api.fill_uniform(t, 2 * t.numel(), 66000 + k)
    hb, hs = gpu.Spectrum(64, big), gpu.Spectrum(32, small)

    def at(b, off, n):
        return b[off:off + n]

    def insts(b):
        lo, mid, tail = a - c, a + c, 2 * a
        if overlap == "out_sig":      # the second reads the end of the first's output
            return [(at(b, tail, a), at(b, 0, a), hb), (at(b, lo, c), at(b, 3 * a, c), hs)]
        if overlap == "out_out":      # both write the end of the first's output
            return [(at(b, tail, a), at(b, 0, a), hb), (at(b, 3 * a, c), at(b, lo, c), hs)]
        return [(at(b, mid, a), at(b, tail, a), hb), (at(b, 3 * a, c), at(b, mid, c), hs)]  # writes what the first read
    ref = buf.clone()
    for s, o, h in insts(ref):
        gpu.conv3d_device(h, s, o)
    batch = api.Batch(insts(buf), mode=api.CF_BATCH_GRAPH)
    batch.launch()
    batch.check()
    assert _same(buf, ref)
    batch.close()


@pytest.mark.parametrize("in_place", [False, True])
def test_slabs_equal_axis_passes(gpu, in_place):
    """One 512^3 convolution runs its y and z passes by slabs of x (conv_passes,
    engine.cpp): the bits of the plan with whole-cube passes in natural order, and
    five passes with the cube's own bytes in a timed call."""
    import torch
    api = gpu.api
    n = 512
    print("case slabs N=%d in_place=%s" % (n, in_place), flush=True)
    sig = torch.empty(n ** 3, dtype=torch.complex64, device="cuda")
    filt = torch.empty_like(sig)
    api.fill_uniform(sig, 2 * sig.numel(), 67001)
    api.fill_uniform(filt, 2 * filt.numel(), 67002)
    ref = torch.empty_like(sig)
    try:
        api.set_plan(n, api.CF_PLAN_AXIS5)
        natural = gpu.Spectrum(n, filt)
        gpu.conv3d_device(natural, sig, ref)
        natural.close()
        api.set_plan(n, api.CF_PLAN_AXIS5Z)
        spec = gpu.Spectrum(n, filt)
    finally:
        api.set_plan(n, api.CF_PLAN_AUTO)
    out = sig.clone() if in_place else torch.zeros_like(sig)
    gpu.conv3d_device(spec, out if in_place else sig, out)
    assert _same(out, ref)
    if not in_place:
        out.zero_()
        passes = gpu.conv3d_device_timed(spec, sig, out)
        assert _same(out, ref)
        assert [p["name"] for p in passes] == ["x_fwd", "y_fwd", "z_fwd_mul_z_inv", "y_inv", "x_inv"]
        assert [p["bytes"] for p in passes] == [k * 8 * n ** 3 for k in (2, 2, 3, 2, 2)]
        assert all(p["ms"] > 0 for p in passes)
    spec.close()


@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("n", [128, 256])
def test_batches_of_the_wide_plan(gpu, n, in_place):
    """A batch of 128^3 cubes with a spectrum of split3_g28m4 runs the passes of
    split3_g24 (conv_passes, engine.cpp), a single cube its own: the bits of single
    cubes, and of 256^3 batches, which keep them."""
    import torch
    api = gpu.api
    count = 3
    print("case wide plan N=%d in_place=%s" % (n, in_place), flush=True)
    sig = torch.empty((count, n ** 3), dtype=torch.complex64, device="cuda")
    filt = torch.empty_like(sig)
    api.fill_uniform(sig, 2 * sig.numel(), 68000 + n)
    api.fill_uniform(filt, 2 * filt.numel(), 69000 + n)
    try:
        api.set_plan(n, api.CF_PLAN_SPLIT3_G28M4)
        spec, shared = gpu.Spectrum(n, filt, count), gpu.Spectrum(n, filt)
        singles = [gpu.Spectrum(n, filt[k]) for k in range(count)]
    finally:
        api.set_plan(n, api.CF_PLAN_AUTO)
    want = torch.empty_like(sig)
    want_sh = torch.empty_like(sig)
    for k in range(count):
        gpu.conv3d_device(singles[k], sig[k], want[k])
        gpu.conv3d_device(shared, sig[k], want_sh[k])
    for h, ref in ((spec, want), (shared, want_sh)):
        out = sig.clone() if in_place else torch.empty_like(sig)
        gpu.conv3d_device(h, out if in_place else sig, out, count)
        assert _same(out, ref)
    for h in [spec, shared] + singles:
        h.close()


@pytest.mark.parametrize("n,count", [(128, 20), (256, 3)])
@pytest.mark.parametrize("shift", [1, -1, 2.5])
@pytest.mark.parametrize("own", [False, True])
def test_groups_with_overlapping_output(gpu, n, count, shift, own):
    """The output of a batch lies `shift` cubes from its signal in the same memory: a
    plan that takes the signals into the workspace gives the bits of a call with
    buffers of their own, as if all cubes were one group."""
    import torch
    api = gpu.api
    print("case overlap N=%d count=%d shift=%s own=%s" % (n, count, shift, own), flush=True)
    P = n ** 3
    buf = torch.empty((count + 6) * P, dtype=torch.complex64, device="cuda")
    api.fill_uniform(buf, 2 * buf.numel(), 70001 + n)
    filt = torch.empty((count if own else 1, P), dtype=torch.complex64, device="cuda")
    api.fill_uniform(filt, 2 * filt.numel(), 70002 + n)
    try:
        api.set_plan(n, api.CF_PLAN_SPLIT3_G24)
        spec = gpu.Spectrum(n, filt, count if own else 1)
    finally:
        api.set_plan(n, api.CF_PLAN_AUTO)
    at = 3 * P
    to = at + int(shift * P)
    sig, out = buf[at:at + count * P], buf[to:to + count * P]
    want = torch.empty_like(sig)
    gpu.conv3d_device(spec, sig, want, count)
    gpu.conv3d_device(spec, sig, out, count)
    assert _same(out, want)
    spec.close()
