"""The no-allocation layer entry point (coli_hip_moe_forward_dev_noalloc)
against the allocating one (coli_hip_moe_forward_dev), through the C ABI:
bit-identical on two calls in a row, the second smaller, on both arms; a call
beyond the fixed scratch is refused. Collected last (it shares the device's
fixed scratch array with nothing else, but runs after the other GPU tests)."""
import ctypes as C
import sys

import numpy as np
import pytest

from peregrine_amd import qt, synth

pytestmark = pytest.mark.gpu


def say(*a):
    print("[case]", *a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def hip():
    from peregrine_amd import hip as h
    assert h.init([0]) == 1
    return h


def _layer(hip, rng, E, D, I, fmt=qt.FMT_I4G):
    gpu = []
    for _ in range(E):
        trip = synth.make_expert(rng, D, I, fmt, 32)
        gpu.append(hip.GpuExpert.upload_grouped(0, trip[0][:2], trip[1][:2], trip[2][:2], D, I, fmt))
    return gpu, hip.ExpertSet(gpu)


def _run(hip, fn, eset, x, ids, w, k, ga, arm):
    S, D = x.shape
    bx, bi, bw = (hip.DeviceBuffer.from_array(a) for a in (x, ids, w))
    bout = hip.DeviceBuffer(S * D * 4)
    fn(eset, bx.ptr, S, bi.ptr, bw.ptr, k, bout.ptr, ga, arm)
    hip.pipe_sync(0)
    return bout.download(np.float32, (S, D))


@pytest.mark.parametrize("arm,ga", [(-1, 32), (0, 0), (2, 32)])
def test_noalloc_matches_allocating_entry_point(hip, arm, ga):
    say("no-alloc", arm, ga)
    rng = np.random.default_rng(77 + arm + ga)
    E, D, I, k = 24, 1024, 512, 8
    _, eset = _layer(hip, rng, E, D, I)
    for S in (40, 3):   # the second call smaller: stale contents of the first must not leak
        x = rng.standard_normal((S, D)).astype(np.float32)
        ids, w = (np.ascontiguousarray(a) for a in synth_route(rng, S, E, k))
        want = _run(hip, hip.moe_forward_dev, eset, x, ids, w, k, ga, arm)
        got = _run(hip, hip.moe_forward_dev_noalloc, eset, x, ids, w, k, ga, arm)
        assert np.array_equal(got, want), (S, arm, ga)


def test_noalloc_decode_shape_and_limit(hip):
    """BASELINE config 2's shape (one token, top-8 of 160... here 16 resident
    experts) twice, then a batch whose scratch exceeds the fixed array."""
    say("no-alloc decode + limit")
    rng = np.random.default_rng(5120)
    E, D, I, k = 16, 5120, 1536, 8
    _, eset = _layer(hip, rng, E, D, I)
    for S in (2, 1):
        x = rng.standard_normal((S, D)).astype(np.float32)
        ids, w = synth_route(rng, S, E, k)
        want = _run(hip, hip.moe_forward_dev, eset, x, ids, w, k, 32, -1)
        got = _run(hip, hip.moe_forward_dev_noalloc, eset, x, ids, w, k, 32, -1)
        assert np.array_equal(got, want), S
    S = 400   # 3200 rows: about 90 MB of scratch at this width
    x = rng.standard_normal((S, D)).astype(np.float32)
    ids, w = synth_route(rng, S, E, k)
    with pytest.raises(hip.HipError):
        _run(hip, hip.moe_forward_dev_noalloc, eset, x, ids, w, k, 32, -1)


def test_noalloc_replayed_from_a_graph(hip):
    """What the entry point is for: a layer captured into a HIP graph with
    no allocation anywhere, replayed with new contents written into the same
    device buffers between replays; every replay equals the allocating entry
    point run eagerly on those contents."""
    say("no-alloc graph replay")
    rng = np.random.default_rng(6144)
    E, D, I, k, S = 24, 1024, 512, 8, 24
    _, eset = _layer(hip, rng, E, D, I)
    bx, bi, bw = hip.DeviceBuffer(S * D * 4), hip.DeviceBuffer(S * k * 4), hip.DeviceBuffer(S * k * 4)
    bout = hip.DeviceBuffer(S * D * 4)

    def contents():
        x = rng.standard_normal((S, D)).astype(np.float32)
        ids, w = synth_route(rng, S, E, k)
        bx.upload(x)
        bi.upload(ids)
        bw.upload(w)
        return x, ids, w

    def body():
        hip.moe_forward_dev_noalloc(eset, bx.ptr, S, bi.ptr, bw.ptr, k, bout.ptr, 32, -1)

    x, ids, w = contents()
    body()   # one eager call first, as for any captured layer
    hip.pipe_sync(0)
    # the allocating reference calls below reserve their scratch now, before
    # the capture (a later growth would make graph_launch refuse the graph)
    _run(hip, hip.moe_forward_dev, eset, x, ids, w, k, 32, -1)
    g = hip.capture(0, body)
    for rep in range(3):
        x, ids, w = contents()
        g.launch()
        hip.pipe_sync(0)
        got = bout.download(np.float32, (S, D))
        want = _run(hip, hip.moe_forward_dev, eset, x, ids, w, k, 32, -1)
        assert np.array_equal(got, want), rep


@pytest.mark.parametrize("fmt", [qt.FMT_I4, qt.FMT_I8])
@pytest.mark.parametrize("E,D,I,k,S,arm", [(9, 2048, 1900, 4, 300, -1), (9, 2048, 1900, 4, 3, 2), (9, 200, 1536, 4, 1, -1),
                                           (5, 64, 4100, 2, 1, 2), (9, 2048, 1900, 4, 6, 0)])
def test_noalloc_per_row_formats(hip, host_rules, fmt, E, D, I, k, S, arm):
    """Per-row weights and activations: the 128-row GEMM, GEMVs that quantise
    h themselves (and not, beyond 4096), one token with ids that repeat and
    leave the range."""
    say("no-alloc per row", fmt, E, D, I, k, S, arm)
    assert bool(host_rules.row_groups_c(D, I, int(fmt == qt.FMT_I4), 1, 1, S * k, E, 0)) == (S == 300)
    rng = np.random.default_rng(S + fmt)
    _, eset = _layer(hip, rng, E, D, I, fmt)
    for s in (S, max(1, S - 1)):
        x = rng.standard_normal((s, D)).astype(np.float32)
        ids = rng.integers(-1, E + 1, (s, k)).astype(np.int32)
        w = rng.uniform(0.1, 1.0, (s, k)).astype(np.float32)
        want = _run(hip, hip.moe_forward_dev, eset, x, ids, w, k, 0, arm)
        got = _run(hip, hip.moe_forward_dev_noalloc, eset, x, ids, w, k, 0, arm)
        assert np.array_equal(got, want) and np.abs(want).max() > 0, s


def test_noalloc_per_row_at_the_scratch_limit(hip, host_rules):
    """The most tokens that are accepted: the list of leading tiles (1287 words,
    under 8 tokens' scratch) no longer fits there and the 32-row GEMM runs;
    from 8 tokens fewer on it fits. The same bits on both sides."""
    say("no-alloc per row limit")
    rng = np.random.default_rng(64)
    E, D, I = 512, 64, 64
    _, eset = _layer(hip, rng, E, D, I, qt.FMT_I4)
    top = 110000
    x = rng.standard_normal((top, D)).astype(np.float32)
    ids = rng.integers(0, E, (top, 1)).astype(np.int32)
    w = rng.uniform(0.1, 1.0, (top, 1)).astype(np.float32)
    bx, bi, bw = (hip.DeviceBuffer.from_array(a) for a in (x, ids, w))
    out = hip.DeviceBuffer(top * D * 4)

    def run(fn, S):
        fn(eset, bx.ptr, S, bi.ptr, bw.ptr, 1, out.ptr, 0, 0)
        hip.pipe_sync(0)
        return out.download(np.float32, (S, D))

    lo, hi = 90000, top   # accepted, refused
    assert host_rules.row_groups_c(D, I, 1, 1, 1, lo, E, 0)
    while hi - lo > 1:
        S = (lo + hi) // 2
        try:
            hip.moe_forward_dev_noalloc(eset, bx.ptr, S, bi.ptr, bw.ptr, 1, out.ptr, 0, 0)
            lo = S
        except hip.HipError:
            hi = S
    assert lo > 90000
    for S in (lo, lo - 4, lo - 7, lo - 8, lo - 9, lo - 60):
        say("limit", S)
        want = run(hip.moe_forward_dev, S)
        got = run(hip.moe_forward_dev_noalloc, S)
        assert np.array_equal(got, want) and np.abs(want).max() > 0, S


def test_noalloc_one_token_beside_ordinary_calls(hip):
    """A captured no-allocation layer of one token, replayed on a stream of its
    own while ordinary one-token layers run on the device's: the two share no
    scratch and no counter, so both stay right."""
    say("no-alloc beside ordinary calls")
    rt = hip.lib   # resolves the HIP runtime it links

    def ck(rc):
        assert rc == 0, rc
    rng = np.random.default_rng(8)
    E, D, I, k = 16, 5120, 1536, 8
    _, eset = _layer(hip, rng, E, D, I)
    case = []
    for _ in range(2):
        x = rng.standard_normal((1, D)).astype(np.float32)
        ids, w = synth_route(rng, 1, E, k)
        want = _run(hip, hip.moe_forward_dev, eset, x, ids, w, k, 32, -1)
        case.append([hip.DeviceBuffer.from_array(a) for a in (x, ids, w)] + [hip.DeviceBuffer(D * 4), want])

    def call(fn, c):
        fn(eset, c[0].ptr, 1, c[1].ptr, c[2].ptr, k, c[3].ptr, 32, -1)
    call(hip.moe_forward_dev_noalloc, case[0])
    hip.pipe_sync(0)
    dev, own, graph, ex = C.c_void_p(hip.stream_handle(0)), C.c_void_p(), C.c_void_p(), C.c_void_p()
    ck(rt.hipStreamCreateWithFlags(C.byref(own), 1))
    ck(rt.hipStreamBeginCapture(dev, 1))
    call(hip.moe_forward_dev_noalloc, case[0])
    ck(rt.hipStreamEndCapture(dev, C.byref(graph)))
    ck(rt.hipGraphInstantiate(C.byref(ex), graph, None, None, C.c_size_t(0)))
    for rep in range(50):
        for c in case:
            c[3].fill(D, 1, 5.0, 1.0, seed=rep)
        hip.pipe_sync(0)
        for _ in range(4):
            ck(rt.hipGraphLaunch(ex, own))
            call(hip.moe_forward_dev, case[1])
        ck(rt.hipStreamSynchronize(own))
        hip.pipe_sync(0)
        for c in case:
            assert np.array_equal(c[3].download(np.float32, (1, D)), c[4]), rep
    ck(rt.hipGraphExecDestroy(ex))
    ck(rt.hipGraphDestroy(graph))
    ck(rt.hipStreamDestroy(own))


def synth_route(rng, S, E, k):
    logits = synth.normal_logits(rng, S, E)
    order = np.argsort(-logits, axis=1, kind="stable")[:, :k].astype(np.int32)
    sel = np.take_along_axis(logits, order, 1).astype(np.float64)
    w = np.exp(sel - sel[:, :1])
    w = (w / w.sum(1, keepdims=True)).astype(np.float32)
    return np.ascontiguousarray(order), np.ascontiguousarray(w)
