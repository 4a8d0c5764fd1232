"""The plain 256^3 transform's two routes: through the workspace in two passes,
and, recorded into a graph, in one pass per axis without it.  Both are held to
the FP32 bound of the other transform tests against the transform in 64 bits."""
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
