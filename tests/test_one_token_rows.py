"""One token with the caller's ids on the GEMV arm: its table is built beside
the activation quantisation, per-row down projections quantise h themselves and
the last workgroup of a tile combines. Ids that repeat, leave the range or are
all invalid, 1 to 16 slots, and h rows at the edges of the in-kernel
quantisation (4096 elements; longer ones take the separate launch);
bit-identical to the oracle's expert outputs summed in union order."""
import numpy as np
import pytest

from peregrine_amd import qt, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt,gs", [(qt.FMT_I4, 0), (qt.FMT_I8, 0), (qt.FMT_I4G, 32)])
@pytest.mark.parametrize("D,I", [(96, 33), (200, 1536), (64, 4096), (64, 4100)])
def test_one_token_ids(orc, fmt, gs, D, I):
    from peregrine_amd import hip
    assert hip.init([0]) == 1
    rng = np.random.default_rng(D + I + fmt)
    E = 18
    gpu, ora = [], []
    for _ in range(E):
        trip = synth.make_expert(rng, D, I, fmt, 32)
        gpu.append(hip.GpuExpert.upload_grouped(0, trip[0][:2], trip[1][:2], trip[2][:2], D, I, fmt, gs or 32))
        ora.append(tuple(orc.Tensor(t[0], t[1], fmt, i, o, gs or 32) for t, (o, i) in zip(trip, ((I, D), (I, D), (D, I)))))
    eset = hip.ExpertSet(gpu)
    x = rng.standard_normal((1, D)).astype(np.float32)
    bx, out = hip.DeviceBuffer.from_array(x), hip.DeviceBuffer(D * 4)
    for ga in (0, 32):
        y = [orc.expert_swiglu(x, *o, ga)[0] for o in ora]
        for ids in ([3], [7, 2], [-1, E], list(range(16)), [5, 9, 5, -3, 9, 5, E + 4, 0], [4] * 16, [E] * 3, [17, 0, 17]):
            print("one token", fmt, D, I, ga, ids, flush=True)
            k = len(ids)
            w = rng.uniform(0.1, 1.0, k).astype(np.float32)
            bi, bw = hip.DeviceBuffer.from_array(np.array(ids, np.int32)), hip.DeviceBuffer.from_array(w)
            ref = np.zeros(D, np.float32)
            order = []
            for e in dict.fromkeys(i for i in ids if 0 <= i < E):
                for j in range(k):
                    if ids[j] == e:
                        ref = ref + w[j] * y[e]
                        order.append(e)
            for rep in range(2):   # the arrival counters are left clear
                out.fill(D, 1, 5.0, 1.0, seed=rep)
                hip.moe_forward_dev(eset, bx.ptr, 1, bi.ptr, bw.ptr, k, out.ptr, ga, 2)
                hip.pipe_sync(0)
                assert np.array_equal(out.download(np.float32, (D,)), ref), (ga, ids, rep)
            t = hip.last_table(0, E, k)
            union = list(dict.fromkeys(order))
            assert t["rows"] == len(order) and t["tiles"] == t["n_u"] == len(union) and list(t["uexp"]) == union
            assert list(t["off"]) == [0] + list(np.cumsum([order.count(e) for e in union]))
            assert list(t["tok_rows"]) == list(range(len(order))) + [-1] * (k - len(order))
