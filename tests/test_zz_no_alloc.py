"""The entry point that allocates nothing (asca_gemm_noalloc: split-K
partials in the library's static device scratch) against asca_gemm, through
the C ABI: two calls in a row, the second on a smaller product, each
bit-identical to asca_gemm and within the forward bar of a float64 product;
the device's free memory unchanged across such calls (and, as a control, an
asca_gemm on a new stream visibly allocating); the scratch's size bounding the
partials of every product."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FWD_TOL = 2e-5
SCRATCH_BYTES = 2 * 256 * 128 * 128 * 4   # the static scratch: the split-K bound on gfx950


def _hip_free_bytes():
    """hipMemGetInfo's free bytes from the HIP runtime the library uses."""
    hip = C.CDLL("libamdhip64.so.7")
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_gemm_noalloc_matches_gemm_on_two_calls(orc, g):
    from asca_amd import _lib
    from asca_amd.gpu import DevBuf, _vp

    rng = np.random.default_rng(77)
    # both split K (too few output tiles for the chip), the second is smaller
    for (M, N, K) in ((512, 1536, 16384), (256, 512, 8192)):
        wsb = C.c_size_t()
        _lib.call("asca_gemm_ws_bytes", 1, 0, M, N, K, C.byref(wsb))
        print(f"[noalloc] TN {M}x{N}x{K}: split-K partials {wsb.value} B", flush=True)
        assert 0 < wsb.value <= SCRATCH_BYTES
        x = rng.standard_normal((K, M)).astype(np.float32)
        d = rng.standard_normal((K, N)).astype(np.float32)
        bias = rng.standard_normal(N).astype(np.float32)
        bx, bd, bb = DevBuf.from_host(x), DevBuf.from_host(d), DevBuf.from_host(bias)
        c1, c2 = DevBuf(M * N * 4), DevBuf(M * N * 4)
        _lib.call("asca_gemm", 1, 0, M, N, K, 0.5, _vp(bx), M, _vp(bd), N, 0.0, _vp(c1), N, _vp(bb), None)
        _lib.call("asca_gemm_noalloc", 1, 0, M, N, K, 0.5, _vp(bx), M, _vp(bd), N, 0.0, _vp(c2), N, _vp(bb), None)
        _lib.call("asca_sync")
        want, got = c1.to_host((M, N)), c2.to_host((M, N))
        np.testing.assert_array_equal(got, want)
        ref = 0.5 * (x.astype(np.float64).T @ d.astype(np.float64)) + bias
        assert orc.rel_err(got, ref) <= FWD_TOL
        for b in (bx, bd, bb, c1, c2):
            b.free()


def test_gemm_noalloc_allocates_nothing(g):
    from asca_amd import _lib
    from asca_amd.gpu import DevBuf, _vp

    M, N, K = 512, 1536, 16384     # split K: 30 MiB of partials
    bx, bd, c = DevBuf(K * M * 4), DevBuf(K * N * 4), DevBuf(M * N * 4)
    args = (1, 0, M, N, K, 1.0, _vp(bx), M, _vp(bd), N, 0.0, _vp(c), N, None, None)
    _lib.call("asca_gemm_noalloc", *args)   # code objects loaded, nothing pending
    _lib.call("asca_sync")
    before = _hip_free_bytes()
    for _ in range(3):
        _lib.call("asca_gemm_noalloc", *args)
    _lib.call("asca_sync")
    after = _hip_free_bytes()
    print(f"[noalloc] device free bytes {before} -> {after}", flush=True)
    assert after == before
    # control: asca_gemm on a stream of its own takes that stream's scratch (the
    # library's pools released first, so the allocation cannot reuse memory they keep)
    _lib.call("asca_pool_release")
    base = _hip_free_bytes()
    sp = C.c_void_p()
    _lib.call("asca_stream_create", C.byref(sp))
    _lib.call("asca_gemm", *args[:-1], sp)
    _lib.call("asca_stream_sync", sp)
    ctrl = _hip_free_bytes()
    print(f"[noalloc] asca_gemm on a new stream: free bytes {base} -> {ctrl}", flush=True)
    assert ctrl < base
    _lib.call("asca_stream_destroy", sp)
    for b in (bx, bd, c):
        b.free()


def test_split_k_partials_never_exceed_the_static_scratch():
    # CPU-side sizing (asca_gemm_ws_bytes needs no device): the shapes that split
    # most, in every transpose case, stay within the static scratch
    from asca_amd import _lib

    worst = 0
    for ta in (0, 1):
        for tb in (0, 1):
            for M in (128, 256, 512, 1000, 1024, 2048):
                for N in (128, 384, 1536, 2048, 4096):
                    for K in (1024, 16384, 1 << 20):
                        wsb = C.c_size_t()
                        _lib.call("asca_gemm_ws_bytes", ta, tb, M, N, K, C.byref(wsb))
                        worst = max(worst, wsb.value)
    print(f"[noalloc] largest split-K partials {worst} B of {SCRATCH_BYTES}", flush=True)
    assert 0 < worst <= SCRATCH_BYTES


@pytest.mark.parametrize("B,T,H,dh,C_", [(2, 500, 4, 128, 32), (4, 300, 4, 96, 64), (4, 1000, 8, 64, 64), (3, 50, 2, 48, 64),
                                         (1, 17, 1, 16, 16), (2, 100, 2, 32, 32), (2, 200, 2, 128, 64), (2, 60, 2, 24, 32)])
def test_chunked_calls_take_their_workspace_and_nothing_else(g, B, T, H, dh, C_):
    """asca_chunk_fwd and _bwd on a new stream: the device's free memory stays as it
    is, the bytes behind the workspace too, and a second backward gives the same."""
    from asca_amd import _lib
    from asca_amd.gpu import DevBuf, _vp

    rng = np.random.default_rng(dh + T)
    rows, d = B * T, H * dh
    bf = lambda a: (np.ascontiguousarray(a, np.float32).view(np.uint32) >> 16).astype(np.uint16)
    q, k, v, do = (DevBuf.from_host(bf(rng.standard_normal((rows, d)) / np.sqrt(dh))) for _ in range(4))
    al, be = (DevBuf.from_host(rng.uniform(0.1, 0.9, (rows, H)).astype(np.float32)) for _ in range(2))
    wsb = C.c_size_t()
    _lib.call("asca_chunk_ws_bytes", B, T, H, dh, C_, C.byref(wsb))
    ws = DevBuf(wsb.value + 4096)
    guard = np.arange(1024, dtype=np.uint32)
    _lib.call("asca_h2d", C.c_void_p(ws.ptr + wsb.value), guard.ctypes.data_as(C.c_void_p), 4096)
    outs = [DevBuf(rows * d * 4) for _ in range(4)] + [DevBuf(rows * H * 4) for _ in range(2)]
    shapes = [(rows, d)] * 4 + [(rows, H)] * 2

    def both(st, fwd, b=B, t=T):
        if fwd:
            _lib.call("asca_chunk_fwd", _vp(q), _vp(k), _vp(v), _vp(al), _vp(be), _vp(outs[0]), _vp(ws), b, t, H, dh, C_, st)
        _lib.call("asca_chunk_bwd", _vp(q), _vp(k), _vp(v), _vp(do), _vp(ws), *[_vp(o) for o in outs[1:]], b, t, H, dh,
                  C_, st)
        _lib.call("asca_stream_sync", st)
        return [o.to_host(s) for o, s in zip(outs, shapes)]

    _lib.call("asca_pool_release")
    sp = C.c_void_p()
    _lib.call("asca_stream_create", C.byref(sp))
    both(sp, True, 1, 1)  # code objects loaded, the stream's hardware queue set up
    before = _hip_free_bytes()
    first = both(sp, True)
    print(f"[no alloc] chunk dh={dh} C={C_} ws {wsb.value} B, free {before} -> {_hip_free_bytes()}", flush=True)
    assert _hip_free_bytes() == before
    for a, b in zip(first, both(sp, False)):
        np.testing.assert_array_equal(a, b)
    _lib.call("asca_stream_destroy", sp)
    got = np.zeros(1024, np.uint32)
    _lib.call("asca_d2h", got.ctypes.data_as(C.c_void_p), C.c_void_p(ws.ptr + wsb.value), 4096)
    np.testing.assert_array_equal(got, guard)
    for b in (q, k, v, do, al, be, ws, *outs):
        b.free()


@pytest.mark.parametrize("what", ["delta dh32", "delta dh128", "gemm"])
def test_captured_calls_keep_their_scratch(g, what):
    """A call captured as the first one on its stream: its replays give the eager
    call's results, also after larger calls on that stream have grown its scratch."""
    from asca_amd import _lib
    from asca_amd.gpu import DevBuf, _vp

    hip = C.CDLL("libamdhip64.so.7")
    ok = lambda rc: None if rc == 0 else pytest.fail(f"HIP error {rc}")
    rng = np.random.default_rng(5)
    f32 = lambda *s: DevBuf.from_host(rng.standard_normal(s).astype(np.float32))
    bufs = []

    def call(big):
        if what == "gemm":  # split K
            M, N, K = (512, 1536, 16384) if big else (256, 256, 8192)
            A, Bm, o = f32(K, M), f32(K, N), DevBuf(M * N * 4)
            bufs.extend([A, Bm, o])
            return (lambda st: _lib.call("asca_gemm", 1, 0, M, N, K, 1.0, _vp(A), M, _vp(Bm), N, 0.0, _vp(o), N, None, st),
                    [(o, (M, N))])
        dh = int(what[8:])
        B, T, H = (17, 80, 8) if big else (17, 40, 8)  # more than 128 units
        rows, d = B * T, H * dh
        q, k, v, do = (f32(rows, d) for _ in range(4))
        al, be = (DevBuf.from_host(rng.uniform(0.1, 0.9, (rows, H)).astype(np.float32)) for _ in range(2))
        for x in (q, k):
            h = x.to_host((rows, H, dh))
            x.upload(h / np.linalg.norm(h, axis=2, keepdims=True))
        wsb = C.c_size_t()
        _lib.call("asca_delta_ws_bytes", B, T, H, dh, C.byref(wsb))
        ws, o = DevBuf(wsb.value), DevBuf(rows * d * 4)
        outs = [(DevBuf(rows * d * 4), (rows, d)) for _ in range(3)] + [(DevBuf(rows * H * 4), (rows, H)) for _ in range(2)]
        bufs.extend([q, k, v, do, al, be, ws, o, *(x for x, _ in outs)])
        _lib.call("asca_delta_fwd", _vp(q), _vp(k), _vp(v), _vp(al), _vp(be), _vp(o), _vp(ws), B, T, H, dh, None)
        _lib.call("asca_sync")
        return (lambda st: _lib.call("asca_delta_bwd_raw", _vp(q), _vp(k), _vp(v), _vp(al), _vp(be), _vp(do), _vp(ws),
                                     *[_vp(x) for x, _ in outs], B, T, H, dh, st), outs)

    run, outs = call(False)
    larger, _ = call(True)
    run(None)
    _lib.call("asca_sync")
    want = [x.to_host(s) for x, s in outs]
    sp, graph, exe = C.c_void_p(), C.c_void_p(), C.c_void_p()
    _lib.call("asca_stream_create", C.byref(sp))
    ok(hip.hipStreamBeginCapture(sp, 0))
    run(sp)
    ok(hip.hipStreamEndCapture(sp, C.byref(graph)))
    ok(hip.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0)))
    for i in range(4):
        for x, s in outs:
            _lib.call("asca_memset32", _vp(x), 0x7fc00000, int(np.prod(s)), sp)
        ok(hip.hipGraphLaunch(exe, sp))
        _lib.call("asca_stream_sync", sp)
        for (x, s), w in zip(outs, want):
            np.testing.assert_array_equal(x.to_host(s), w)
        larger(sp)
        _lib.call("asca_stream_sync", sp)
    ok(hip.hipGraphExecDestroy(exe))
    ok(hip.hipGraphDestroy(graph))
    _lib.call("asca_stream_destroy", sp)
    for b in bufs:
        b.free()
