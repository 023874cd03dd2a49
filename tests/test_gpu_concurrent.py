"""Engines on separate streams at the same time: two dual-stream engines (each step's FFN-down runs as a stream-K
launch, each stream with its own partials workspace) and an SDXL engine run concurrently, and every result equals,
bit for bit, the same engine's result when it ran alone."""
import ctypes as C
import threading
import time

import numpy as np
import pytest

import mkimage as M

pytestmark = pytest.mark.gpu

D, H, F, E = 3072, 24, 12288, 3584
SDXL_B = dict(blocks=2, dim=1280, heads=20, head_dim=64, ffn=5120, text_dim=2048)


def dual_engine(seed):
    # one block of the 1024x1024 shape: 4096 image + 256 text tokens, CFG batch 2 (8704 rows: the FFN-down GEMM's
    # 408 tiles take one whole wave and a stream-K tail)
    e = M.Engine(M.FAMILY_DUAL, blocks=1, dim=D, heads=H, head_dim=128, ffn=F, text_dim=E)
    e.init_random(seed)
    rng = np.random.default_rng(seed)
    for s in (0, 1):
        e.begin(rng.standard_normal((256, E)).astype(np.float32), 64, 64, s)
    lat = M.Dev.from_array(rng.standard_normal((4096, 64)).astype(np.float32))
    return e, lat


def test_dual_and_sdxl_engines_on_separate_streams_match_their_solo_bits(gpu):
    duals = [dual_engine(s) for s in (1, 2)]
    sx = M.Engine(M.FAMILY_SDXL, **SDXL_B)
    sx.init_random(3)
    rng = np.random.default_rng(3)
    for s in (0, 1):
        sx.begin(rng.standard_normal((77, 2048)).astype(np.float32), 32, 32, s)
    n = 1024
    x = M.Dev.from_array(rng.standard_normal((2, n, 1280)).astype(np.float32))
    outs = [M.Dev(4096 * 64 * 4) for _ in duals]
    y = M.Dev(2 * n * 1280 * 4)

    def read():
        return [o.to_array(np.float32, (4096, 64)) for o in outs] + [y.to_array(np.float32, (2, n, 1280))]

    # alone: one engine at a time, each finished before the next starts
    for (e, lat), o in zip(duals, outs):
        e.step_cfg_device(lat, 0.9, 0.85, 4.0, o)
        M.call("mk_stream_synchronize", e.stream())
    sx.sdxl_forward(x, 2, n, y)
    solo = read()
    for a in solo:
        assert np.isfinite(a).all()
    for a in outs + [y]:
        M.call("mk_memset", a.p, 0, a.nbytes)
    M.sync()
    # together: both dual steps queued on their engines' streams, the SDXL pass runs (and waits for its own stream)
    # while they are in flight
    for rep in range(2):
        for (e, lat), o in zip(duals, outs):
            e.step_cfg_device(lat, 0.9, 0.85, 4.0, o)
        sx.sdxl_forward(x, 2, n, y)
        for e, _ in duals:
            M.call("mk_stream_synchronize", e.stream())
        for got, want in zip(read(), solo):
            assert np.array_equal(got, want), f"repeat {rep}"
    for e, _ in duals:
        e.close()
    sx.close()


N, K, SHAPES, GN = 256, 4096, (200, 40), (2, 1024, 640, 32)  # a grouped launch that splits its k steps; a group norm
PER_THREAD = 2  # hipStreamPerThread: one handle, a stream of its own in each thread


class Small:
    """One seed's split-K GEMM and group norm on a stream, into new buffers each launch."""

    def __init__(self, seed):
        r = np.random.default_rng(seed)
        dev = lambda a: M.Dev.from_array(a.astype(np.float32))  # noqa: E731
        bdev = lambda a: M.Dev.from_array(M.bf16_bits(a.astype(np.float32)))  # noqa: E731
        self.a = [bdev(r.standard_normal((m, K))) for m in SHAPES]
        self.w, self.b = bdev(r.standard_normal((N, K)) * 0.03), dev(r.standard_normal(N))
        self.x, self.g, self.gb = dev(r.standard_normal(GN[:3])), dev(r.standard_normal(GN[2])), dev(
            r.standard_normal(GN[2]))
        self.runs = []

    def out(self):
        c = [M.Dev(m * N * 4) for m in SHAPES]
        args = []
        for a, m, o in zip(self.a, SHAPES, c):
            g = M.GemmArgs()
            g.a, g.w, g.bias, g.c = a.p, self.w.p, self.b.p, o.p
            g.M, g.N, g.K, g.lda, g.ldc, g.batch = m, N, K, K, N, 1
            g.w_dtype, g.c_dtype, g.epilogue = M.BF16, M.F32, M.EPI_STORE
            args.append(g)
        return (M.GemmArgs * 2)(*args), c, M.Dev(GN[0] * GN[1] * GN[2] * 2)

    def launch(self, stream, bufs):
        arr, c, y = bufs
        M.call("mk_gemm_grouped", C.cast(arr, C.c_void_p), 2, stream)
        M.call("mk_group_norm", self.x.p, *GN, self.g.p, self.gb.p, 1e-6, y.p, stream)
        self.runs.append(bufs)

    def read(self):
        got = [[d.to_array(np.float32, (m, N)) for d, m in zip(c, SHAPES)] + [y.to_array(np.uint16, GN[:3])]
               for _, c, y in self.runs]
        self.runs = []
        return got


def test_threads_on_their_per_thread_streams_match_their_solo_bits(gpu):
    # hipStreamPerThread is the same handle in every thread: the workspaces of one thread's launches are not another's
    work = [Small(s) for s in range(4)]
    solo = []
    for w in work:
        w.launch(None, w.out())
        M.sync()
        solo.append(w.read()[0])
    start, errors = threading.Barrier(len(work)), []

    def run(w, bufs):
        try:
            start.wait()
            for b in bufs:
                w.launch(PER_THREAD, b)
            M.call("mk_stream_synchronize", PER_THREAD)
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=run, args=(w, [w.out() for _ in range(20)])) for w in work]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    for w, want in zip(work, solo):
        for i, got in enumerate(w.read()):
            assert all(np.array_equal(a, b) for a, b in zip(got, want)), f"launch {i}"


def test_streams_destroyed_by_their_caller_match_their_solo_bits(gpu):
    # a stream that its caller made and destroys with work in flight, and the next one, which may get its handle
    hip = C.CDLL("libamdhip64.so.7")
    work = [Small(s) for s in range(2)]
    solo = []
    for w in work:
        w.launch(None, w.out())
        M.sync()
        solo.append(w.read()[0])
    bufs = [[w.out() for w in work] for _ in range(12)]
    for pair in bufs:
        for w, b in zip(work, pair):
            s = C.c_void_p()
            assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0  # non-blocking
            w.launch(s.value, b)
            assert hip.hipStreamDestroy(s) == 0
    M.sync()
    for w, want in zip(work, solo):
        for i, got in enumerate(w.read()):
            assert all(np.array_equal(a, b) for a, b in zip(got, want)), f"launch {i}"


def test_split_launches_on_more_streams_than_slab_buffers_do_not_wait_for_the_device(gpu):
    # 11 streams take turns with 8 buffers while another one works: the launches return, and have their solo bits
    work = Small(0)
    work.launch(None, work.out())
    M.sync()
    want = work.read()[0]
    streams = []
    for _ in range(11):
        h = C.c_void_p()
        M.call("mk_stream_create", C.byref(h))
        streams.append(h.value)
    rows = 8192
    a, w, c = M.Dev(rows * K * 2), M.Dev(rows * K * 2), M.Dev(rows * rows * 4)
    for d in (a, w):
        M.call("mk_memset", d.p, 0, d.nbytes)
    g = M.GemmArgs()
    g.a, g.w, g.c = a.p, w.p, c.p
    g.M, g.N, g.K, g.lda, g.ldc, g.batch = rows, rows, K, K, rows, 1
    g.w_dtype, g.c_dtype, g.epilogue = M.BF16, M.F32, M.EPI_STORE
    for s in streams:  # every stream has had a buffer
        work.launch(s, work.out())
    bufs = [work.out() for _ in range(3) for _ in streams]
    M.sync()
    for _ in range(300):  # 0.1 s or more
        M.call("mk_gemm", C.byref(g), streams[0])
    t0 = time.perf_counter()
    for b, s in zip(bufs, 3 * streams):
        M.call("mk_gemm_grouped", C.cast(b[0], C.c_void_p), 2, s)
    t1 = time.perf_counter()
    M.sync()
    t2 = time.perf_counter()
    assert t1 - t0 < (t2 - t0) / 2, f"{(t1 - t0) * 1e3:.1f} ms of {(t2 - t0) * 1e3:.1f} for the launches"
    for _, c, _ in bufs:
        for d, m, x in zip(c, SHAPES, want):
            assert np.array_equal(d.to_array(np.float32, (m, N)), x)
    for got in work.read():
        assert all(np.array_equal(x, y) for x, y in zip(got, want))
    for s in streams:
        M.call("mk_stream_destroy", s)


def test_streams_used_in_turn_share_a_slab_buffer(gpu):
    # a new stream's first split launch takes an idle stream's buffer instead of allocating one
    hip = C.CDLL("libamdhip64.so.7")

    def free():
        a, b = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(a), C.byref(b)) == 0
        return a.value

    work = Small(0)
    handles = [C.c_void_p() for _ in range(5)]
    for h in handles:
        M.call("mk_stream_create", C.byref(h))
    bufs = [work.out() for _ in handles]
    work.launch(handles[0].value, bufs[0])
    M.sync()
    before = free()
    for h, b in zip(handles[1:], bufs[1:]):
        work.launch(h.value, b)
        M.sync()
    assert before - free() < 32 << 20
    want, *rest = work.read()
    for got in rest:
        assert all(np.array_equal(a, b) for a, b in zip(got, want))
    for h in handles:
        M.call("mk_stream_destroy", h.value)


def test_small_gemms_during_another_streams_capture(gpu):
    # one stream is being captured while others run split launches for the first time (they need slab buffers); the
    # captured launches, of sizes that split when they are not captured, run whole tiles, the same bits every replay
    hip = C.CDLL("libamdhip64.so.7")
    work = Small(0)
    work.launch(None, work.out())
    M.sync()
    want = work.read()[0]
    handles = [C.c_void_p() for _ in range(11)]
    for h in handles:
        M.call("mk_stream_create", C.byref(h))
    cap, *others = [h.value for h in handles]
    inside, outside = work.out(), [work.out() for _ in others]
    graph, run = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(C.c_void_p(cap), 0) == 0  # global mode
    M.call("mk_gemm_grouped", C.cast(inside[0], C.c_void_p), 2, cap)
    for s, b in zip(others, outside):
        M.call("mk_gemm_grouped", C.cast(b[0], C.c_void_p), 2, s)
    assert hip.hipStreamEndCapture(C.c_void_p(cap), C.byref(graph)) == 0
    assert hip.hipGraphInstantiate(C.byref(run), graph, None, None, 0) == 0
    M.sync()
    for _, c, _ in outside:
        assert all(np.array_equal(d.to_array(np.float32, (m, N)), x) for d, m, x in zip(c, SHAPES, want))
    first = None
    for _ in range(3):
        for d in inside[1]:
            M.call("mk_memset", d.p, 0xFF, d.nbytes)
        M.sync()
        assert hip.hipGraphLaunch(run, C.c_void_p(cap)) == 0
        M.call("mk_stream_synchronize", cap)
        got = [d.to_array(np.float32, (m, N)) for d, m in zip(inside[1], SHAPES)]
        first = first or got
        for g, f, x in zip(got, first, want):
            assert np.array_equal(g, f)
            # fp32 sums of K products in another order
            assert np.abs(g - x).max() <= 1e-5 * np.abs(x).max()
        work.launch(None, outside[0])  # the program's own work between the replays
        M.sync()
        assert all(np.array_equal(a, b) for a, b in zip(work.read()[0], want))
    assert hip.hipGraphExecDestroy(run) == 0 and hip.hipGraphDestroy(graph) == 0
    for s in (cap, *others):
        M.call("mk_stream_destroy", s)


def test_group_norm_is_refused_under_capture(gpu):
    # its scratch is shared with later calls, which may free it: a graph must not keep it, also where the capturing
    # stream was the scratch's last user
    hip = C.CDLL("libamdhip64.so.7")
    work = Small(0)
    h, graph = C.c_void_p(), C.c_void_p()
    M.call("mk_stream_create", C.byref(h))
    work.launch(h.value, work.out())
    M.sync()
    want = work.read()[0][-1]
    y = M.Dev(want.nbytes)
    args = (work.x.p, *GN, work.g.p, work.gb.p, 1e-6, y.p, h.value)
    assert hip.hipStreamBeginCapture(h, 0) == 0
    status = M.lib().mk_group_norm(*args)
    assert hip.hipStreamEndCapture(h, C.byref(graph)) == 0
    assert hip.hipGraphDestroy(graph) == 0
    assert status != 0 and b"graph" in M.lib().mk_last_error()
    M.call("mk_group_norm", *args)
    M.sync()
    assert np.array_equal(y.to_array(np.uint16, want.shape), want)
    M.call("mk_stream_destroy", h.value)
