"""The transforms' kept scratch (StreamScratch): results do not depend on what earlier calls, streams
or threads left in the blocks, and a C2R leaves its input as it was. Transforms of every size class that
takes scratch are compared bit for bit with the first call's result."""
import threading

import numpy as np
import pytest

from tests._util import to_np

pytestmark = pytest.mark.gpu

SHAPES = [(2, (3, 512, 640)), (2, (5, 768, 1024)), (3, (2, 40, 384, 75)), (2, (1, 1000, 96)), (3, (1, 512, 32, 48))]


def _round(gx, x, ndims):
    X = gx.d_FFTR2C(x, ndims=ndims)
    return X, gx.d_IFFTC2R(X, x.shape[-1], ndims=ndims)


def test_scratch_across_sizes_and_streams(gx, cuda):
    import torch
    rng = np.random.default_rng(5)
    data = [(nd, torch.from_numpy(rng.standard_normal(s).astype(np.float32)).to(cuda)) for nd, s in SHAPES]
    want = []
    for nd, x in data:
        X, y = _round(gx, x, nd)
        ref = np.fft.rfftn(to_np(x).astype(np.float64), axes=tuple(range(-nd, 0)))
        # single-precision transforms of these lengths stay below 1e-6 normwise
        assert np.linalg.norm(to_np(X) - ref) <= 1e-6 * np.linalg.norm(ref)
        assert np.linalg.norm(to_np(y) - to_np(x)) <= 2e-6 * np.linalg.norm(to_np(x))
        want.append((to_np(X), to_np(y)))
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(3)]
    for k in range(6):
        got = []
        for i, (nd, x) in enumerate(data):
            with torch.cuda.stream(streams[(i + k) % 3]):
                X = gx.d_FFTR2C(x, ndims=nd)
                keep = X.clone()
                got.append((X, keep, gx.d_IFFTC2R(X, x.shape[-1], ndims=nd)))
        torch.cuda.synchronize()
        for (X, keep, y), (wX, wy) in zip(got, want):
            assert torch.equal(torch.view_as_real(X), torch.view_as_real(keep))
            assert np.array_equal(to_np(X), wX) and np.array_equal(to_np(y), wy)


def test_scratch_from_threads(gx, cuda):
    import torch
    rng = np.random.default_rng(6)
    data = [(nd, torch.from_numpy(rng.standard_normal(s).astype(np.float32)).to(cuda)) for nd, s in SHAPES]
    want = [tuple(map(to_np, _round(gx, x, nd))) for nd, x in data]
    torch.cuda.synchronize()
    bad = []

    def work(k):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for i in range(8):
                nd, x = data[(i + k) % len(data)]
                X, y = _round(gx, x, nd)
                s.synchronize()
                w = want[(i + k) % len(data)]
                if not (np.array_equal(to_np(X), w[0]) and np.array_equal(to_np(y), w[1])):
                    bad.append((k, i))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


CAP = 4 << 30  # include/gtomx.h


def test_kept_scratch_is_bounded_and_released(gx, cuda):
    """Two blocks of 2.02 GiB and three small ones of one call pass the cap together: what is held afterwards does
    not, on the default stream and on another, and a release gives all of it back to the device."""
    import torch
    n, p, nang = 256, 32, 32
    rng = np.random.default_rng(8)
    projft = gx.prepare_projector(torch.from_numpy(rng.standard_normal((16, 16, 16)).astype(np.float32)).to(cuda), p)
    E = gx.d_FFTR2C(torch.from_numpy(rng.standard_normal((2, n, n, n)).astype(np.float32)).to(cuda))
    ctf = torch.ones((2, n, n, n // 2 + 1), device=cuda)
    angles = rng.uniform(0, 6, (nang, 3)).astype(np.float32)
    assert 2 * nang * (n // 2 + 1) * n * n * 8 > CAP
    for stream in (torch.cuda.default_stream(), torch.cuda.Stream()):
        stream.wait_stream(torch.cuda.default_stream())
        with torch.cuda.stream(stream):
            gx.d_PickSubTomogramsDiff2(projft, p, p / n, E, ctf, (2, 2, 2), angles)
        stream.synchronize()
        held = gx.scratch_held()
        assert 0 < held <= CAP, held
    free = torch.cuda.mem_get_info()[0]
    gx.scratch_release()
    assert gx.scratch_held() == 0
    assert torch.cuda.mem_get_info()[0] >= free + held // 2
    X = gx.d_IFFTC2R(E, n)  # and the next call takes blocks again
    torch.cuda.synchronize()
    assert gx.scratch_held() > 0 and torch.isfinite(X).all()


@pytest.mark.parametrize("what", ["kept", "above the cap", "tables"])
def test_out_of_memory_gives_the_kept_scratch_back_and_tries_again(gx, cuda, what):
    """Every allocation behind a transform, told once that memory is out, is made at the second try with nothing kept;
    told twice it is refused, and the next call is well again."""
    import torch
    x = torch.from_numpy(np.random.default_rng(9).standard_normal((1, 64, 64)).astype(np.float32)).to(cuda)
    X = gx.d_FFTR2C(x, ndims=2)
    if what == "above the cap":
        X = X.expand(CAP // (8 * 64 * 33) + 1, 64, 33).contiguous()
    for tries in (1, 2):
        gx.scratch_release()
        big = gx.d_IFFTC2R(gx.d_FFTR2C(torch.zeros((1, 512, 512), device=cuda), ndims=2), 512, ndims=2)
        torch.cuda.synchronize()
        kept = gx.scratch_held()
        assert kept >= 8 * 512 * 257
        lines = torch.ones((1, 3, 467 if tries == 1 else 461), device=cuda)  # chirp-z lengths no other test takes
        gx.lib().gtomx_debug_out_of_memory(tries)
        try:
            if what == "tables":
                call = lambda: gx.d_FFTR2C(lines, ndims=2)  # takes no scratch of its own
            else:
                call = lambda: gx.d_IFFTC2R(X, 64, ndims=2)
            if tries == 2:
                with pytest.raises(gx.GtomxError, match="(?i)memory"):
                    call()
            else:
                y = call()
        finally:
            gx.lib().gtomx_debug_out_of_memory(0)
        torch.cuda.synchronize()
        assert gx.scratch_held() < kept
        if tries == 1 and what == "tables":
            assert abs(to_np(y)[0, 0, 0] - 3 * 467) <= 1e-2 and np.abs(to_np(y)[0].ravel()[1:]).max() <= 1e-2
        elif tries == 1:
            assert torch.equal(y[0], y[-1]) and (y[0] - x[0]).abs().max() <= 1e-5
        y = call()
        torch.cuda.synchronize()
        del y, big


# rows alone (native up to 256 and above), rows without a native transform, and a batch of several slices
@pytest.mark.parametrize("ndims,shape", [(1, (37, 64)), (1, (9, 4096)), (1, (6, 75)), (2, (20, 1024, 2048)),
                                         (2, (3, 64, 48))])
@pytest.mark.parametrize("at", ["start", "end"])
def test_c2r_over_its_own_input(gx, cuda, ndims, shape, at):
    """The output may lie over the spectra: at their start, and at the end of the same buffer."""
    import torch
    nx, batch = shape[-1], int(np.prod(shape[:-ndims]))
    gen = torch.Generator(device=cuda)
    gen.manual_seed(nx)
    X = gx.d_FFTR2C(torch.randn(shape, device=cuda, generator=gen), ndims=ndims)
    want = gx.d_IFFTC2R(X, nx, ndims=ndims)
    buf = torch.view_as_real(X).reshape(-1).clone()
    n = want.numel()
    o = 0 if at == "start" else (buf.numel() - n) // 2 * 2
    dims = (nx,) + tuple(reversed(shape[-ndims:-1])) + (1,) * (3 - ndims)
    gx.check(gx.lib().gtomx_ifft_c2r(gx._ptr(buf), gx._ptr(buf[o:]), ndims, gx.int3(*dims), batch, 1, gx._stream()),
             "gtomx_ifft_c2r")
    assert torch.equal(buf[o:o + n].reshape(want.shape), want)


@pytest.mark.parametrize("ndims,shape", [(2, (20, 1024, 2048)), (3, (7, 768, 16, 512)), (2, (3, 4096, 4096))])
def test_slices_of_a_batch_equal_items_alone(gx, cuda, ndims, shape):
    """Axes of two passes go through the scratch in slices of about 128 MB (15 of 20 items, 5 of 7, one by one): every item bit for bit as transformed alone, and the C2R's input as it was."""
    import torch
    gen = torch.Generator(device=cuda)
    gen.manual_seed(shape[0])
    x = torch.randn(shape, device=cuda, generator=gen)
    X = gx.d_FFTR2C(x, ndims=ndims)
    keep = X.clone()
    y = gx.d_IFFTC2R(X, shape[-1], ndims=ndims)
    assert torch.equal(torch.view_as_real(X), torch.view_as_real(keep))
    for i in range(shape[0]):
        Xi = gx.d_FFTR2C(x[i:i + 1].contiguous(), ndims=ndims)
        assert torch.equal(torch.view_as_real(X[i:i + 1]), torch.view_as_real(Xi)), i
        assert torch.equal(y[i:i + 1], gx.d_IFFTC2R(Xi, shape[-1], ndims=ndims)), i
