"""Asynchronous calls on one stream and an extraction on another right behind them: the backward still uses the
extraction it belongs to, as do the positions and quads, and so does a second backward on a third stream."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 72
SHAPE = (N, N, N)


def sphere(r):
    t = np.linspace(-1, 1, N, dtype=np.float32)
    return (np.sqrt(t[:, None, None] ** 2 + t[None, :, None] ** 2 + t[None, None, :] ** 2) - r).astype(np.float32)


@pytest.mark.parametrize("first", ["stream", "default", "own"])
@pytest.mark.parametrize("call", ["backward", "backward_noalloc", "two backwards", "quads"])
def test_extraction_on_another_stream_waits(call, first):
    import torch

    import manifolddmc_amd as mdmc
    flags = mdmc.PAD1 | mdmc.RECORD_ADJOINT
    big, small = (torch.from_numpy(sphere(r)).cuda() for r in (0.7, 0.4))
    a, b, c = (torch.cuda.Stream() for _ in range(3))
    busy = torch.full((4096, 4096), 1e-3, device="cuda")
    d = mdmc.DualMarchingCubes()

    def extract(f):
        d.extract_raw(f.data_ptr(), SHAPE, (-1, -1, -1), (2 / (N - 1),) * 3, 0.0, flags, 0, True)
        return d.info()

    handle = {"stream": a.cuda_stream, "default": mdmc.DEFAULT_STREAM, "own": 0}[first]
    queue = {"stream": a, "default": torch.cuda.default_stream(), "own": None}[first]

    def read(stream, dpos, out, use):
        d.set_stream(handle if stream is a else stream.cuda_stream)
        if use == "quads":
            d.copy_quads(out[0].data_ptr(), out[1].data_ptr())
        elif use == "backward_noalloc":
            d.backward_noalloc(dpos.data_ptr(), out[0].data_ptr(), False)
        else:
            d.backward(dpos.data_ptr(), out[0].data_ptr(), False)

    try:
        torch.cuda.synchronize()
        d.set_stream(handle)
        V, _, F = extract(big)
        dpos = torch.randn((V, 3), device="cuda", generator=torch.Generator(device="cuda").manual_seed(5))
        make = lambda: (torch.zeros((V, 3), device="cuda"), torch.zeros((F, 4), dtype=torch.int64, device="cuda")) if call == "quads" else (torch.zeros(SHAPE, device="cuda"),)
        want, got, more = make(), make(), make()
        torch.cuda.synchronize()
        read(a, dpos, want, call)
        torch.cuda.synchronize()
        for rep in range(3):
            print("reader streams", call, first, rep, flush=True)
            d.set_stream(handle)
            assert extract(big) == (V, 4 * F, F)
            if queue is not None:
                with torch.cuda.stream(queue):  # some ms of work that the reader stands behind
                    h = busy
                    for _ in range(12):
                        h = h @ busy
            read(a, dpos, got, call)
            if call == "two backwards":
                read(c, dpos, more, call)
            d.set_stream(b.cuda_stream)
            Vs, _, _ = extract(small)
            assert 0 < Vs < V
            torch.cuda.synchronize()
            for x, y in zip(got, want):
                assert torch.equal(x, y), (call, rep)
            if call == "two backwards":
                assert torch.equal(more[0], want[0]), rep
            for x in got + more:
                x.zero_()
            torch.cuda.synchronize()
    finally:
        torch.cuda.synchronize()
        d.close()


def test_backward_in_a_graph_and_an_extraction_elsewhere():
    import torch

    import manifolddmc_amd as mdmc
    f = torch.from_numpy(sphere(0.6)).cuda()
    d = mdmc.DualMarchingCubes()
    try:
        s = torch.cuda.Stream()
        torch.cuda.synchronize()
        d.set_stream(s.cuda_stream)
        ext = lambda: d.extract_raw(f.data_ptr(), SHAPE, (-1, -1, -1), (2 / (N - 1),) * 3, 0.0, mdmc.PAD1 | mdmc.RECORD_ADJOINT, 0, True)
        ext()
        dpos = torch.ones((d.info()[0], 3), device="cuda")
        want, got = torch.zeros(SHAPE, device="cuda"), torch.zeros(SHAPE, device="cuda")
        torch.cuda.synchronize()
        d.backward_noalloc(dpos.data_ptr(), want.data_ptr(), False)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            d.backward_noalloc(dpos.data_ptr(), got.data_ptr(), False)
        for rep in range(3):
            got.fill_(float("nan"))
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(got, want), rep
        d.set_stream(0)
        ext()
        d.backward_noalloc(dpos.data_ptr(), got.data_ptr(), False)
        d.set_stream(s.cuda_stream)
        ext()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
    finally:
        d.close()


def test_stream_destroyed_behind_its_backward():
    import ctypes

    import torch

    import manifolddmc_amd as mdmc
    hip = ctypes.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line))
    f = torch.from_numpy(sphere(0.6)).cuda()
    d = mdmc.DualMarchingCubes()
    try:
        ext = lambda: d.extract_raw(f.data_ptr(), SHAPE, (-1, -1, -1), (2 / (N - 1),) * 3, 0.0, mdmc.PAD1 | mdmc.RECORD_ADJOINT, 0, True)
        torch.cuda.synchronize()
        ext()
        dpos = torch.ones((d.info()[0], 3), device="cuda")
        want, got = torch.zeros(SHAPE, device="cuda"), torch.zeros(SHAPE, device="cuda")
        torch.cuda.synchronize()
        d.backward(dpos.data_ptr(), want.data_ptr(), False)
        for rep in range(2):
            s = ctypes.c_void_p()
            assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0
            d.set_stream(s.value)
            ext()
            d.backward(dpos.data_ptr(), got.data_ptr(), False)
            assert hip.hipStreamDestroy(s) == 0
            d.set_stream(0)
            ext()
            torch.cuda.synchronize()
            assert torch.equal(got, want), rep
    finally:
        d.close()
