"""What orders the library's launches on several streams and threads, on the CPU:
the host library linked to a HIP runtime that records calls instead of running
them (tests/native/hip_recorder.h, stream_order_check.cpp)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
CHECKS = ["fft_per_thread", "fft_streams", "fft_beside_capture", "fft_first_call", "conv_per_thread",
          "spectrum_reuse", "conv_overlap", "trim"]

needs_gxx = pytest.mark.skipif(shutil.which("g++") is None or not os.path.exists(os.path.join(ROCM, "include", "hip")),
                               reason="needs g++ and the HIP headers")


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = tmp_path_factory.mktemp("order") / "stream_order_check"
    csrc = os.path.join(ROOT, "convfpga_amd", "csrc")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-fopenmp", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I" + os.path.join(ROCM, "include"), "-I" + os.path.join(ROOT, "include"), "-I" + csrc,
                    os.path.join(ROOT, "tests", "native", "stream_order_check.cpp"),
                    os.path.join(csrc, "engine.cpp"), os.path.join(csrc, "capi.cpp"), "-o", str(exe)], check=True)
    return str(exe)


@needs_gxx
@pytest.mark.parametrize("name", CHECKS)
def test_stream_order(check, name):
    r = subprocess.run([check, name], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.endswith("ok %s\n" % name), r.stdout


@pytest.fixture
def fresh(gpu):
    """the library as a program that has just started finds it: no stream has a workspace"""
    gpu.fpga_final()
    assert gpu.fpga_initialize("gfx950", gpu.CODE_OBJECT, True) == 0
    return gpu


def _transforms(n, k):
    """k inputs and what one call on each gives, by whichever route"""
    import torch
    import convfpga_amd as C
    x = torch.empty((k, n, n, n), dtype=torch.complex64, device="cuda")
    C.api.fill_uniform(x, 2 * x.numel(), 73001 + n)
    want = torch.stack([torch.fft.fftn(v.to(torch.complex128)) for v in x])
    return x, torch.empty_like(x), want


def _rel(a, b):
    import torch
    return max(float(torch.linalg.vector_norm(p.to(torch.complex128) - q) / torch.linalg.vector_norm(q))
               for p, q in zip(a, b))


@pytest.mark.gpu
@pytest.mark.parametrize("per_thread", [True, False])
def test_transforms_of_several_threads(fresh, per_thread):
    """256^3 transforms of six threads, on hipStreamPerThread (handle 2) or on a
    stream each, held to the FP32 bound of the other transform tests."""
    import threading

    import torch
    n, k, rounds = 256, 6, 8
    print("case fft threads per_thread=%s" % per_thread, flush=True)
    x, y, want = _transforms(n, k)
    streams = [2 if per_thread else torch.cuda.Stream() for _ in range(k)]
    torch.cuda.synchronize()
    errors = []

    def work(i):
        try:
            for _ in range(rounds):
                fresh.fft3d_device(n, x[i], y[i], stream=streams[i])
            torch.cuda.synchronize()
        except Exception as e:  # shown by the assertion below
            errors.append(e)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(k)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors and _rel(y, want) <= 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("n", [256, 512])
def test_transform_beside_a_capture(fresh, n):
    """A stream that ran a transform is recorded into a graph while another stream
    runs one: that one runs at once, and the graph is whole."""
    import torch
    print("case fft beside capture N=%d" % n, flush=True)
    x, y, want = _transforms(n, 2)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    fresh.fft3d_device(n, x[1], y[1], stream=b)
    fresh.fft3d_device(n, x[0], y[0], stream=a)
    torch.cuda.synchronize()
    y.fill_(float("nan"))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=a, capture_error_mode="relaxed"):
        fresh.fft3d_device(n, x[0], y[0], stream=a)
        fresh.fft3d_device(n, x[1], y[1], stream=b)
    torch.cuda.synchronize()
    assert bool(torch.isnan(y[0]).all()) and _rel(y[1:], want[1:]) <= 1e-5
    for _ in range(3):
        y.fill_(float("nan"))
        graph.replay()
        fresh.fft3d_device(n, x[1], y[1])
        torch.cuda.synchronize()
        assert _rel(y, want) <= 1e-5


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["global", "thread_local", "relaxed"])
def test_first_transform_of_a_stream_beside_a_capture(fresh, mode):
    """A stream's first 256^3 transform, which allocates its workspace, while
    another stream is recorded into a graph."""
    import torch
    n = 256
    print("case first fft beside capture mode=%s" % mode, flush=True)
    x, y, want = _transforms(n, 2)
    fresh.fft3d_device(n, x[0], y[0])
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()  # (as torch.cuda.graph does)
    free = torch.cuda.mem_get_info()[0]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=a, capture_error_mode=mode):
        fresh.fft3d_device(n, x[0], y[0], stream=a)
        fresh.fft3d_device(n, x[1], y[1], stream=b)
    torch.cuda.synchronize()
    assert free - torch.cuda.mem_get_info()[0] >= 8 * n ** 3  # the workspace
    for _ in range(3):
        y[0].fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert _rel(y, want) <= 1e-5


@pytest.mark.gpu
def test_convolutions_of_several_threads(fresh):
    """256^3 convolutions through the common workspace from four threads on their
    hipStreamPerThread (handle 2), with others on a stream between them: the bits of
    calls one after the other."""
    import threading

    import torch
    api, n, k, rounds = fresh.api, 256, 5, 8
    print("case conv threads", flush=True)
    x = torch.empty((k, n, n, n), dtype=torch.complex64, device="cuda")
    api.fill_uniform(x, 2 * x.numel(), 74001)
    y, want = torch.empty_like(x), torch.empty_like(x)
    api.set_plan(n, api.CF_PLAN_SPLIT3_G24)
    try:
        spec = fresh.Spectrum(n, x[0])
    finally:
        api.set_plan(n, api.CF_PLAN_AUTO)
    for i in range(k):
        fresh.conv3d_device(spec, x[i], want[i])
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    errors = []

    def work(i):
        try:
            for _ in range(rounds):
                fresh.conv3d_device(spec, x[i], y[i], stream=2 if i else stream)
            torch.cuda.synchronize()
        except Exception as e:  # shown by the assertion below
            errors.append(e)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(k)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    spec.close()
    assert not errors
    assert torch.equal(torch.view_as_real(y).view(torch.int32), torch.view_as_real(want).view(torch.int32))
