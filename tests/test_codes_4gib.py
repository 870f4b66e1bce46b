"""Layers whose activation codes pass 4 GiB, where the scalar-base copies of the
grouped GEMM (32-bit offsets) give way to kernels with 64-bit addresses: the
last tokens, whose rows lie past 4 GiB, equal a small batch of the same tokens
bit for bit. Codes of h (66000 tokens x 8 experts x 8192) and of x."""
import numpy as np
import pytest

from peregrine_amd import qt, synth

pytestmark = pytest.mark.gpu


def _layer(hip, rng, E, D, I, fmt):
    ex = []
    for _ in range(E):
        t = synth.make_expert(rng, D, I, fmt, 32)
        ex.append(hip.GpuExpert.upload_grouped(0, t[0][:2], t[1][:2], t[2][:2], D, I, fmt, 32))
    return hip.ExpertSet(ex)


@pytest.mark.parametrize("fmt,ga", [(qt.FMT_I8, 0), (qt.FMT_I4, 0), (qt.FMT_I4G, 0)])
def test_h_codes_past_4gib(fmt, ga):
    from peregrine_amd import hip
    assert hip.init([0]) == 1
    S, k, E, D, I, n = 66000, 8, 8, 64, 8192, 256
    assert (S * k - n) * I > 1 << 32   # the last expert's last n rows
    print("h codes past 4 GiB", fmt, ga, flush=True)
    rng = np.random.default_rng(fmt)
    eset = _layer(hip, rng, E, D, I, fmt)
    x = rng.standard_normal((S, D)).astype(np.float32)
    w = rng.uniform(0.1, 1.0, (S, k)).astype(np.float32)
    ids = np.tile(np.arange(k, dtype=np.int32), (S, 1))
    got = []
    for s in (S, n):
        b = [hip.DeviceBuffer.from_array(a[-s:]) for a in (x, ids, w)]
        out = hip.DeviceBuffer(s * D * 4)
        hip.moe_forward_dev(eset, b[0].ptr, s, b[1].ptr, b[2].ptr, k, out.ptr, ga, 0)
        hip.pipe_sync(0)
        got.append(out.download(np.float32, (s, D))[-n:])
    assert np.abs(got[1]).max() > 0 and np.array_equal(got[0], got[1])
    assert hip.init([0]) == 1   # gives the scratch back


@pytest.mark.parametrize("fmt", [qt.FMT_I8, qt.FMT_I4])
def test_x_codes_past_4gib(fmt):
    from peregrine_amd import hip
    assert hip.init([0]) == 1
    S, E, D, I, n = 525000, 2, 8192, 32, 256
    assert (S - n) * D > 1 << 32
    print("x codes past 4 GiB", fmt, flush=True)
    rng = np.random.default_rng(fmt)
    eset = _layer(hip, rng, E, D, I, fmt)
    x = hip.DeviceBuffer(S * D * 4)
    x.fill(S * D, 1, 0.0, 1.0, seed=7)
    ids = np.zeros((S, 1), np.int32)
    ids[-3000::2] = 1
    w = rng.uniform(0.1, 1.0, (S, 1)).astype(np.float32)
    bi, bw = hip.DeviceBuffer.from_array(ids), hip.DeviceBuffer.from_array(w)
    out = hip.DeviceBuffer(S * D * 4)
    small = hip.DeviceBuffer(n * D * 4)
    at = S - n
    hip.moe_forward_dev(eset, x.ptr, S, bi.ptr, bw.ptr, 1, out.ptr, 0, 0)
    hip.moe_forward_dev(eset, x.ptr + at * D * 4, n, bi.ptr + at * 4, bw.ptr + at * 4, 1, small.ptr, 0, 0)
    hip.pipe_sync(0)
    tail = hip.DeviceBuffer.__new__(hip.DeviceBuffer)   # a view of out's last n rows
    tail.device, tail.ptr, tail.nbytes = 0, out.ptr + at * D * 4, n * D * 4
    got, want = tail.download(np.float32, (n, D)), small.download(np.float32, (n, D))
    tail.ptr = 0
    assert np.abs(want).max() > 0 and np.array_equal(got, want)
    assert hip.init([0]) == 1
