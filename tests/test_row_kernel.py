"""The 128-row MFMA kernel of per-row weights and activations.

On the CPU: its work items, copies and LDS layout through the index functions
that the kernel calls. On the GPU: dispatches with two or more M tiles per
expert, at the edges of its tiles, bit-identical to the oracle (the dots are
exact integers and the f32 steps are the oracle's)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from peregrine_amd import qt, synth

HERE = os.path.dirname(os.path.abspath(__file__))
MT = 32


def tiles_of(rows):
    t = [[], [], [], []]
    r = 0
    for e, n in enumerate(rows):
        t0 = len(t[0])
        for q in range(0, n, MT):
            for a, v in zip(t, (e, r + q, r + n, t0)):
                a.append(v)
        r += n
    return [np.asarray(a, np.int32) for a in t], r


@pytest.fixture(scope="module")
def chk(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("rowb") / "librow_bounds.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", os.path.join(HERE, "native", "row_bounds.cpp"),
                    "-o", out], check=True)
    lib = ctypes.CDLL(out)
    lib.check_row_dispatch.restype = ctypes.c_long
    return lib


@pytest.fixture(scope="module")
def hip():
    from peregrine_amd import hip as h
    assert h.init([0]) == 1
    yield h
    h.set_arm(-1)
    h.set_act_group(0)


def _p(a):
    return None if a is None else a.ctypes.data_as(ctypes.POINTER(ctypes.c_int))


def run_check(chk, gateup, w4, K, O, rows, lead_bound=None, row_act=None, rows_x=None, short=0):
    t, R = tiles_of(rows)
    T = len(t[0])
    Kp = -(-K // 32) * 32
    if lead_bound is None:
        lead_bound = chk.row_lead_bound_c(R, len(rows))   # the layer's bound on the leading tiles
    return chk.check_row_dispatch(int(gateup), int(w4), Kp // 32, O, T, lead_bound, _p(t[0]), _p(t[1]), _p(t[2]),
                                  _p(t[3]), R, _p(row_act), (rows_x or R) - short, Kp, len(rows))


ROWS = [[96], [70, 70, 5], [64] * 3, [200, 1, 31, 95], [129, 128, 127, 33], [1000, 64, 40]]


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("K,O", [(1536, 640), (1000, 712), (32, 33), (96, 1), (2048, 1536)])
def test_row_kernel_in_bounds(chk, rows, K, O):
    for w4 in (True, False):
        for gateup in (True, False):
            assert run_check(chk, gateup, w4, K, O, rows) == 0
            # a grid of exactly the leading tiles; rows gathered from fewer activation rows
            act = np.random.default_rng(3).integers(0, 17, sum(rows)).astype(np.int32)
            assert run_check(chk, gateup, w4, K, O, rows, lead_bound=sum(-(-n // 128) for n in rows), row_act=act,
                             rows_x=17) == 0


def test_row_checker_is_not_vacuous(chk):
    assert run_check(chk, True, True, 96, 64, [70], short=1) > 0
    assert run_check(chk, True, True, 96, 64, [40] * 9, lead_bound=8) > 0   # the last tile's item is missing


# the most rows within 4 GiB of activation codes, then the first whose offset needs a 33rd bit
EDGE_4GIB = [(524288, 8192), (524289, 8192), (838860, 5120), (838862, 5120), (2796202, 1536), (2796204, 1536)]


@pytest.mark.parametrize("rows_x,K", EDGE_4GIB)
def test_row_kernel_offsets_reach_4gib(chk, rows_x, K):
    """The kernel's 32-bit activation offsets hold exactly where its launch
    accepts them."""
    chk.off32_ok_c.argtypes = [ctypes.c_uint64]
    act = np.arange(rows_x - 70, rows_x, dtype=np.int32)   # the last rows
    for w4 in (True, False):
        bad = run_check(chk, True, w4, K, 64, [70], row_act=act, rows_x=rows_x)
        assert (bad == 0) == bool(chk.off32_ok_c(rows_x * K)) == (rows_x * K <= 1 << 32)


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [qt.FMT_I4, qt.FMT_I8])
@pytest.mark.parametrize("D,I", [(1000, 8130), (160, 8161), (96, 8192)])
@pytest.mark.parametrize("rows", [[200, 1, 31, 95], [129, 128], [64, 97, 288]])
def test_row_kernel_matches_oracle(hip, orc, host_rules, fmt, D, I, rows):
    print("row kernel", fmt, D, I, rows, flush=True)
    rng = np.random.default_rng(D + I + fmt + len(rows))
    gpu, ora = [], []
    for _ in rows:
        trip = synth.make_expert(rng, D, I, fmt, 32)
        gpu.append(hip.GpuExpert.upload_grouped(0, trip[0][:2], trip[1][:2], trip[2][:2], D, I, fmt, 32))
        ora.append(tuple(orc.Tensor(t[0], t[1], fmt, i, o, 32) for t, (o, i) in zip(trip, ((I, D), (I, D), (D, I)))))
    assert host_rules.row_groups_c(D, I, int(fmt == qt.FMT_I4), 1, 1, sum(rows), len(rows), 0)   # as the runtime decides
    x = rng.standard_normal((sum(rows), D)).astype(np.float32)
    hip.set_act_group(0)
    hip.set_arm(0)
    try:
        y, arm = hip.expert_group_tiled(gpu, rows, x, D)
    finally:
        hip.set_arm(-1)
    assert arm.value == 0
    at = 0
    for e, n in enumerate(rows):
        assert np.array_equal(y[at:at + n], orc.expert_swiglu(x[at:at + n], *ora[e], 0)), e
        at += n


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", [qt.FMT_I4, qt.FMT_I8])
@pytest.mark.parametrize("E,S,k,D,I", [(5, 64, 3, 2048, 5440), (9, 300, 4, 2048, 1900), (3, 700, 3, 96, 1800)])
def test_row_kernel_layer(hip, orc, host_rules, fmt, E, S, k, D, I):
    """The layer, whose leading tiles the device table lists (both table
    forms), with ids that skip an expert, repeat one and leave the range; at
    D = 2048 the rule's lower bound of 24 rows per expert holds too."""
    print("row layer", fmt, E, S, k, flush=True)
    assert host_rules.row_groups_c(D, I, int(fmt == qt.FMT_I4), 1, 1, S * k, E, 0)   # as the runtime decides
    rng = np.random.default_rng(E * S + fmt)
    gpu, ora = [], []
    for _ in range(E):
        trip = synth.make_expert(rng, D, I, fmt, 32)
        gpu.append(hip.GpuExpert.upload_grouped(0, trip[0][:2], trip[1][:2], trip[2][:2], D, I, fmt, 32))
        ora.append(tuple(orc.Tensor(t[0], t[1], fmt, i, o, 32) for t, (o, i) in zip(trip, ((I, D), (I, D), (D, I)))))
    eset = hip.ExpertSet(gpu)
    x = rng.standard_normal((S, D)).astype(np.float32)
    ids = np.minimum(rng.geometric(0.35, (S, k)) - 1, E - 1).astype(np.int32)   # skewed, with repeats
    w = rng.uniform(0.1, 1.0, (S, k)).astype(np.float32)
    bad = ids.copy()
    bad[::7, 0], bad[::11, k - 1] = -1, E
    b = [hip.DeviceBuffer.from_array(a) for a in (x, bad, w)]
    out = hip.DeviceBuffer(S * D * 4)
    hip.moe_forward_dev(eset, b[0].ptr, S, b[1].ptr, b[2].ptr, k, out.ptr, 0)
    hip.pipe_sync(0)
    got = out.download(np.float32, (S, D))
    ok = (bad >= 0) & (bad < E)
    # the oracle takes ids in range: a skipped slot is its expert with weight 0, taken out of the order below
    hdr = np.zeros(4, np.int32)
    assert hip.lib.coli_hip_last_table(0, hip._ipt(hdr), None, None, None, None, 0, 0) == 1
    counts = np.bincount(bad[ok], minlength=E)
    assert list(hdr) == [ok.sum(), (-(-counts // MT)).sum(), (counts > 0).sum(), 0]   # the documented header
    ref = np.zeros((S, D), np.float32)
    y = np.zeros((E, S, D), np.float32)
    for e in range(E):
        t = np.nonzero(((bad == e) & ok).any(1))[0]
        if len(t):
            y[e, t] = orc.expert_swiglu(x[t], *ora[e], 0)
    union = list(dict.fromkeys(bad[ok].tolist()))
    for e in union:
        for j in range(k):
            t = np.nonzero(ok[:, j] & (bad[:, j] == e))[0]
            ref[t] = ref[t] + w[t, j][:, None] * y[e, t]
    assert np.array_equal(got, ref)
