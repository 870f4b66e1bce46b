"""Per-row activation quantisation by whole waves: row lengths at the edges of
its 4-element groups and of what it holds in registers (8192 elements a
workgroup), few rows (four waves a row) and many (one), and rows that the
general kernel takes; layers bit-identical to the oracle."""
import numpy as np
import pytest

from peregrine_amd import qt, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,I,S", [(4, 33, 3), (36, 64, 2), (1028, 96, 5), (8192, 32, 2), (8196, 32, 2), (37, 40, 3),
                                   (36, 100, 530), (2048, 33, 601)])
def test_quant_rows_layer(orc, D, I, S):
    from peregrine_amd import hip
    assert hip.init([0]) == 1
    print("quant rows", D, I, S, flush=True)
    rng = np.random.default_rng(D + S)
    E, k, fmt = 3, 2, qt.FMT_I4
    gpu, ora = [], []
    for _ in range(E):
        trip = synth.make_expert(rng, D, I, fmt, 32)
        gpu.append(hip.GpuExpert.upload_grouped(0, trip[0][:2], trip[1][:2], trip[2][:2], D, I, fmt, 32))
        ora.append(tuple(orc.Tensor(t[0], t[1], fmt, i, o, 32) for t, (o, i) in zip(trip, ((I, D), (I, D), (D, I)))))
    eset = hip.ExpertSet(gpu)
    x = rng.standard_normal((S, D)).astype(np.float32)
    x[0] = 0.0                      # the scale's floor
    x[1, D - 1] = 300.0             # the maximum in the last element
    ids = np.stack([rng.permutation(E)[:k] for _ in range(S)]).astype(np.int32)
    w = rng.uniform(0.1, 1.0, (S, k)).astype(np.float32)
    b = [hip.DeviceBuffer.from_array(a) for a in (x, ids, w)]
    out = hip.DeviceBuffer(S * D * 4)
    for arm in (0, 2):
        hip.moe_forward_dev(eset, b[0].ptr, S, b[1].ptr, b[2].ptr, k, out.ptr, 0, arm)
        hip.pipe_sync(0)
        assert np.array_equal(out.download(np.float32, (S, D)), orc.moe_forward(x, ids, w, ora, 0)), arm
