"""SwiGLU's exp at the ends of its range through the kernels' lane-held table:
gate values from far below the underflow of exp(-g) to far above its overflow,
bit-identical to the oracle (glibc expf) on the GEMV and MFMA arms."""
import numpy as np
import pytest

from peregrine_amd import qt, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("arm", [2, 0])
@pytest.mark.parametrize("ga", [0, 32])
@pytest.mark.parametrize("fmt,gs", [(qt.FMT_I4G, 32), (qt.FMT_I8, 0)])
def test_silu_over_the_range_of_exp(orc, arm, ga, fmt, gs):
    from peregrine_amd import hip
    assert hip.init([0]) == 1
    print("silu", arm, ga, fmt, flush=True)
    rng = np.random.default_rng(5 + fmt + ga)
    D, I, n = 64, 96, 70
    trip = [list(t) for t in synth.make_expert(rng, D, I, fmt, 32)]
    g = hip.GpuExpert.upload_grouped(0, trip[0][:2], trip[1][:2], trip[2][:2], D, I, fmt, 32)
    o = tuple(orc.Tensor(t[0], t[1], fmt, i, oo, 32) for t, (oo, i) in zip(trip, ((I, D), (I, D), (D, I))))
    # row scales from 1e-6 to 1e4: |gate| from 0 to beyond 104 and 88
    x = rng.standard_normal((n, D)).astype(np.float32) * np.logspace(-6, 4, n, dtype=np.float32)[:, None]
    x[0] = 0.0
    hip.set_act_group(ga)
    hip.set_arm(arm)
    try:
        y = hip.expert_group([g], [n], x, D)
    finally:
        hip.set_arm(-1)
        hip.set_act_group(0)
    _, h = orc.expert_swiglu(x, *o, ga, want_h=True)
    assert np.isfinite(h).all() and np.abs(h).max() > 1e4 and np.abs(h[1:3]).max() < 1e-3
    assert np.array_equal(y, orc.expert_swiglu(x, *o, ga))
