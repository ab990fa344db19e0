"""Launches with scratch between them (fft/scratch.py) on the GPU: calls, graphs and captures on
several streams at once.  Bounds: the suite's rel-L2 5e-6 / 1e-5 against FP64."""
import numpy as np
import pytest

import oracle as O
import vkdispatch_amd as vd
from tests._gpu_common import assert_close, crand

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

N, COUNT = 1 << 17, 16


def _signals(seed, copies):
    rng = np.random.default_rng(seed)
    xs = [crand(rng, (COUNT, N)) for _ in range(copies)]
    return xs, [np.fft.fft(x.astype(np.complex128), axis=1) for x in xs]


def test_graphs_on_other_streams_beside_calls():
    """Two graphs recorded on the library's stream, submitted on two others, and calls on the
    first: all under way together, three rounds."""
    print("scratch: graphs on two streams beside calls", flush=True)
    xs, refs = _signals(1, 3)
    dev = [torch.from_numpy(x).cuda() for x in xs]
    work = [torch.empty_like(d) for d in dev]
    bufs = [vd.from_cuda_array(w) for w in work]
    vd.fft.fft(bufs[2])  # loads the kernels
    vd.synchronize()
    graphs = [vd.CommandGraph() for _ in range(2)]
    for g, b in zip(graphs, bufs):
        vd.fft.fft(b, graph=g)
    streams = [torch.cuda.Stream() for _ in range(2)]
    for _ in range(3):
        for w, d in zip(work, dev):
            w.copy_(d)
        torch.cuda.synchronize()
        for g, s in zip(graphs, streams):
            g.submit(stream=s.cuda_stream)
        vd.fft.fft(bufs[2])
        torch.cuda.synchronize()
        for w, ref in zip(work, refs):
            assert_close(w.cpu().numpy(), ref)


def test_captured_calls():
    """Direct calls captured into two of torch's graphs, which replay on two streams beside
    calls on the library's; a second transform in one capture shares with the first."""
    print("scratch: captured calls", flush=True)
    xs, refs = _signals(2, 3)
    dev = [torch.from_numpy(x).cuda() for x in xs]
    work = [torch.empty_like(d) for d in dev]
    bufs = [vd.from_cuda_array(w) for w in work]
    vd.fft.fft(bufs[2])
    vd.fft.ifft(bufs[2])
    vd.synchronize()
    graphs = [torch.cuda.CUDAGraph() for _ in range(2)]
    for i, (g, b) in enumerate(zip(graphs, bufs)):
        with torch.cuda.graph(g):
            with vd.cuda_graph_capture(torch.cuda.current_stream()):
                vd.fft.fft(b)
                if i:
                    vd.fft.ifft(b)
                    vd.fft.fft(b)
    streams = [torch.cuda.Stream() for _ in range(2)]
    for _ in range(3):
        for w, d in zip(work, dev):
            w.copy_(d)
        torch.cuda.synchronize()
        for g, s in zip(graphs, streams):
            with torch.cuda.stream(s):
                g.replay()
        vd.fft.fft(bufs[2])
        torch.cuda.synchronize()
        for w, ref in zip(work, refs):
            assert_close(w.cpu().numpy(), ref)


def test_convolutions_on_two_streams():
    """Two batches of one shape with different kernels, each on a stream of its own."""
    print("scratch: convolutions on two streams", flush=True)
    rng = np.random.default_rng(3)
    xs = [rng.uniform(-1, 1, (16, 256, 256)).astype(np.float32) for _ in range(2)]
    ks = [np.fft.rfft2(rng.standard_normal((256, 256))).astype(np.complex64) for _ in range(2)]
    refs = [O.convolve2DR(x, k, kernel_inner_only=True) for x, k in zip(xs, ks)]
    bufs, kbufs = [], []
    for x, k in zip(xs, ks):
        bufs.append(vd.asrfftbuffer(x))
        kbufs.append(vd.RFFTBuffer((256, 256)))
        kbufs[-1].write_fourier(k)
    vd.fft.convolve2DR(bufs[0], kbufs[0], kernel_inner_only=True)
    streams = [torch.cuda.Stream() for _ in range(2)]
    for _ in range(3):
        for b, x in zip(bufs, xs):
            b.write_real(x)
        vd.synchronize()
        for s, b, k in zip(streams, bufs, kbufs):
            with vd.stream_scope(s):
                vd.fft.convolve2DR(b, k, kernel_inner_only=True)
        torch.cuda.synchronize()
        for b, ref in zip(bufs, refs):
            assert_close(b.read_real(0), ref, rel=1e-5)


@pytest.mark.parametrize("count", [3, 24])
def test_prime_lengths_on_two_streams(count):
    """The ragged executor's lengths: items of the persistent kernel (3), a length class on side
    streams (24)."""
    print("scratch: prime lengths on two streams", count, flush=True)
    rng = np.random.default_rng(count)
    xs = [crand(rng, (count, 20011)) for _ in range(3)]
    refs = [np.fft.fft(x.astype(np.complex128), axis=1) for x in xs]
    bufs = [vd.asbuffer(x) for x in xs]
    g = vd.CommandGraph()
    vd.fft.fft(bufs[2], graph=g)
    streams = [torch.cuda.Stream() for _ in range(3)]
    for _ in range(3):
        for b, x in zip(bufs, xs):
            b.write(x)
        vd.synchronize()
        g.submit(stream=streams[2].cuda_stream)
        for s, b in zip(streams, bufs[:2]):
            with vd.stream_scope(s):
                vd.fft.fft(b)
        torch.cuda.synchronize()
        for b, ref in zip(bufs, refs):
            assert_close(b.read(0), ref, rel=1e-5)
