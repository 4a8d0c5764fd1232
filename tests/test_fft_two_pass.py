"""The plain 256^3 and 512^3 transforms' two routes: through the workspace (256^3 in
two passes, 512^3 by slabs), and, recorded into a graph, in one pass per axis
without it.  The 256^3 routes are held to the FP32 bound of the other transform
tests against the transform in 64 bits, the 512^3 ones to the same bits."""
import pytest

pytestmark = pytest.mark.gpu


def _rel(a, b):
    import torch
    return float(torch.linalg.vector_norm(a.to(torch.complex128) - b) / torch.linalg.vector_norm(b))


@pytest.mark.parametrize("inverse", [False, True])
@pytest.mark.parametrize("in_place", [False, True])
def test_fft256_routes_agree(gpu, inverse, in_place):
    import torch
    n = 256
    print("case fft 256 routes inverse=%s in_place=%s" % (inverse, in_place), flush=True)
    x = torch.empty((n, n, n), dtype=torch.complex64, device="cuda")
    gpu.api.fill_uniform(x, 2 * x.numel(), 71001)
    y = x.clone() if in_place else torch.empty_like(x)
    gpu.fft3d_device(n, y if in_place else x, y, 1, inverse)
    want = torch.fft.ifftn(x.to(torch.complex128)) * n ** 3 if inverse else torch.fft.fftn(x.to(torch.complex128))
    assert _rel(y, want) <= 1e-5
    src, dst = x.clone(), torch.empty_like(x)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        gpu.fft3d_device(n, src, dst, 1, inverse, stream=torch.cuda.current_stream())
    for _ in range(3):
        dst.fill_(float("nan"))
        graph.replay()
        gpu.fft3d_device(n, x, y, 1, inverse)  # eager work that uses the workspace
        torch.cuda.synchronize()
        assert _rel(dst, want) <= 1e-5


@pytest.mark.parametrize("inverse", [False, True])
@pytest.mark.parametrize("count", [1, 2])
def test_fft512_slabs_equal_axis_passes(gpu, inverse, count):
    import torch
    n = 512
    print("case fft 512 routes inverse=%s count=%d" % (inverse, count), flush=True)
    x = torch.empty((count, n, n, n), dtype=torch.complex64, device="cuda")
    gpu.api.fill_uniform(x, 2 * x.numel(), 72001)
    axis = torch.empty_like(x)
    gpu.fft3d_device(n, x[0], axis[0], 1, inverse)  # sets the edge up, which a capture cannot
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        gpu.fft3d_device(n, x, axis, count, inverse, stream=torch.cuda.current_stream())
    graph.replay()
    torch.cuda.synchronize()
    for y in (torch.empty_like(x), x):  # out of place, then in place
        gpu.fft3d_device(n, x, y, count, inverse)
        torch.cuda.synchronize()
        assert torch.equal(torch.view_as_real(y).view(torch.int32), torch.view_as_real(axis).view(torch.int32))
