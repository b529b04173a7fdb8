"""mc_local_warp_noalloc (no device allocation; its tables live in a
file-scope device array) against mc_local_warp, bit for bit: two calls in a
row, the second with a smaller input, then one without bad flags after one
with them (the array keeps the previous call's contents); and the size
limit."""
import ctypes as C

import numpy as np
import pytest

from motioncor3_amd import lib as L

pytestmark = pytest.mark.gpu


def _noalloc(ctx, frames, centers, shifts, bad):
    N, H, W = frames.shape
    P = len(centers)
    out = ctx.empty(frames.shape, np.float32)
    cen = np.ascontiguousarray(centers, dtype=np.float32)
    sh = np.ascontiguousarray(shifts, dtype=np.float32)
    bp = None
    if bad is not None:
        bad = np.ascontiguousarray(bad, dtype=np.uint8)
        bp = bad.ctypes.data_as(C.POINTER(C.c_ubyte))
    rc = ctx.lib.mc_local_warp_noalloc(ctx.ptr, frames.vp(), out.vp(), W, H, N, P,
                                       cen.ctypes.data_as(C.POINTER(C.c_float)),
                                       sh.ctypes.data_as(C.POINTER(C.c_float)), bp)
    return rc, out


def _case(rng, N, H, W, P, with_bad):
    frames = rng.standard_normal((N, H, W)).astype(np.float32)
    g = int(np.sqrt(P))
    cen = np.array([[(i % g + 0.5) * W / g, (i // g + 0.5) * H / g] for i in range(P)], np.float32)
    sh = rng.uniform(-4, 4, (N, P, 2)).astype(np.float32)
    bad = (rng.uniform(0, 1, (N, P)) < 0.2).astype(np.uint8) if with_bad else None
    return frames, cen, sh, bad


def test_noalloc_warp_equals_allocating_warp(ctx):
    rng = np.random.default_rng(17)
    cases = [_case(rng, 6, 400, 520, 25, True),    # first call
             _case(rng, 3, 210, 300, 9, True),     # smaller: fewer frames, patches, pixels
             _case(rng, 4, 256, 256, 16, False)]   # no flags after flags: all cleared
    for k, (frames, cen, sh, bad) in enumerate(cases):
        print("no-alloc warp case", k, frames.shape, len(cen), flush=True)
        d = ctx.upload(frames)
        ref = ctx.local_warp(d, cen, sh, bad).numpy()
        rc, out = _noalloc(ctx, d, cen, sh, bad)
        assert rc == L.MC_OK, ctx.lib.mc_last_error(ctx.ptr)
        assert np.array_equal(out.numpy(), ref), k


def test_noalloc_warp_rejects_tables_beyond_its_scratch(ctx):
    """64 patches x 8000 frames need 4.6 MB of tables, more than the 4 MiB
    array: refused before any GPU work, with a message."""
    N, P = 8000, 64
    frames = ctx.empty((N, 2, 2), np.float32)
    cen = np.zeros((P, 2), np.float32)
    sh = np.zeros((N, P, 2), np.float32)
    rc, _ = _noalloc(ctx, frames, cen, sh, None)
    assert rc == L.MC_E_ARG
    assert b"scratch" in ctx.lib.mc_last_error(ctx.ptr)


def test_noalloc_warp_captured_reads_its_tables_at_replay(ctx):
    """A captured call copies the caller's shift table at every replay: with
    other values in it, larger and non-zero under a bad flag, each replay gives
    what a direct call with them gives."""
    hip = C.CDLL("libamdhip64.so.7")
    stream, graph, run = C.c_void_p(), C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreate(C.byref(stream)) == 0
    own = L.Context(0, stream.value)
    rng = np.random.default_rng(5)
    frames, cen, sh, bad = _case(rng, 5, 96, 128, 9, True)
    d, out = own.upload(frames), own.empty(frames.shape, np.float32)
    fp, bp = C.POINTER(C.c_float), bad.ctypes.data_as(C.POINTER(C.c_ubyte))

    def call():
        return own.lib.mc_local_warp_noalloc(own.ptr, d.vp(), out.vp(), 128, 96, 5, 9, cen.ctypes.data_as(fp),
                                             sh.ctypes.data_as(fp), bp)

    assert call() == L.MC_OK
    own.sync()
    print("capture", flush=True)
    assert hip.hipStreamBeginCapture(stream, 2) == 0
    rc = call()
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0 and rc == L.MC_OK
    assert hip.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
    for k in range(3):
        sh[:] = rng.uniform(-20 * (k + 1), 20 * (k + 1), sh.shape)
        print("replay", k, flush=True)
        assert hip.hipGraphLaunch(run, stream) == 0
        own.sync()
        assert np.array_equal(out.numpy(), own.local_warp(d, cen, sh, bad).numpy()), k
    assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
    d.free()
    out.free()
    own.close()
    assert hip.hipStreamDestroy(stream) == 0
