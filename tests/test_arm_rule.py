"""Small batches choose their arm by rows, format and expert size. At both sides
of each format's bound, in each of the rule's three expert sizes, the automatic
choice equals the forced GEMM bit for bit, for router logits, the caller's ids
(repeated and out of range) and the host-buffer calls; for per-row weights and
activations the launches show which arm ran (only the GEMM's quantises h in a
launch of its own). The rule at every bound: test_host_rules.py."""
import numpy as np
import pytest

from peregrine_amd import qt, synth

pytestmark = pytest.mark.gpu


def check(host_rules, fmt, gs, rows, E, D, I):
    from peregrine_amd import hip
    assert hip.init([0]) == 1
    rng = np.random.default_rng(fmt + E)
    ex = []
    for _ in range(E):
        t = synth.make_expert(rng, D, I, fmt, gs or 32)
        ex.append(hip.GpuExpert.upload_grouped(0, t[0][:2], t[1][:2], t[2][:2], D, I, fmt, gs or 32))
    eset = hip.ExpertSet(ex)
    w4 = int(fmt in (qt.FMT_I4, qt.FMT_I4G))

    def ran(fn):
        """The arm that fn's one dispatch ran, by its launches (per-row weights and activations)."""
        hip.reset_stats()
        hip.set_profile(True)
        fn()
        hip.pipe_sync(0)
        hip.set_profile(False)
        return 0 if hip.kernel_stats()["quant_h"][0] else 2

    for R in rows:
        want = 2 if host_rules.gemv_pays_c(D, I, w4, w4, R) else 0
        for ga in (0, 32):
            print("arm rule", fmt, gs, R, E, D, I, ga, want, flush=True)
            k = 2 if E > 1 and R % 2 == 0 else 1
            S = R // k
            x = rng.standard_normal((S, D)).astype(np.float32)
            logits = synth.zipf_logits(rng, S, E)
            ids = rng.integers(-1, E + 1, (S, k)).astype(np.int32)
            w = rng.uniform(0.1, 1.0, (S, k)).astype(np.float32)
            bx, bl, bi, bw = [hip.DeviceBuffer.from_array(a) for a in (x, logits, ids, w)]
            ri, rw, out = hip.DeviceBuffer(S * k * 4), hip.DeviceBuffer(S * k * 4), hip.DeviceBuffer(S * D * 4)
            got = []
            for arm in (-1, 0):
                hip.moe_forward_logits_dev(eset, bx.ptr, S, bl.ptr, k, ri.ptr, rw.ptr, out.ptr, ga, arm)
                hip.pipe_sync(0)
                a = out.download(np.float32, (S, D))
                hip.moe_forward_dev(eset, bx.ptr, S, bi.ptr, bw.ptr, k, out.ptr, ga, arm)
                hip.pipe_sync(0)
                got.append((a, out.download(np.float32, (S, D))))
            assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
            n = np.diff(np.linspace(0, R, E + 1).astype(int)).tolist()
            xr = rng.standard_normal((R, D)).astype(np.float32)
            hip.set_act_group(ga)
            y = []
            for arm in (-1, 0):
                hip.set_arm(arm)
                y.append(hip.expert_group(ex, n, xr, D))
            hip.set_arm(-1)
            if gs == 0 and ga == 0:
                assert ran(lambda: hip.moe_forward_logits_dev(eset, bx.ptr, S, bl.ptr, k, ri.ptr, rw.ptr, out.ptr, ga, -1)) == want
                assert ran(lambda: hip.moe_forward_dev(eset, bx.ptr, S, bi.ptr, bw.ptr, k, out.ptr, ga, -1)) == want
                assert ran(lambda: hip.expert_group(ex, n, xr, D)) == want
                # the call that reports its arm: the GEMV only where no expert has two rows
                assert hip.expert_group_tiled(ex, n, xr, D)[1].value == 0
                assert hip.expert_group_tiled(ex, [1] * E, xr[:E], D)[1].value == 2
            hip.set_act_group(0)
            assert np.array_equal(y[0], y[1])


@pytest.mark.parametrize("fmt,gs,rows", [(qt.FMT_I4, 0, (47, 48, 49)), (qt.FMT_I4G, 64, (48, 50)), (qt.FMT_I8, 0, (23, 24, 25)),
                                         (qt.FMT_I8G, 32, (24, 26))])
@pytest.mark.parametrize("E,D,I", [(5, 200, 75), (1, 96, 64)])
def test_automatic_arm_equals_gemm(host_rules, fmt, gs, rows, E, D, I):
    check(host_rules, fmt, gs, rows, E, D, I)


@pytest.mark.parametrize("fmt,gs,D,I,rows", [
    (qt.FMT_I4, 0, 2048, 1536, (39, 40, 41)), (qt.FMT_I4G, 128, 2048, 1536, (40, 42)), (qt.FMT_I8, 0, 2048, 1536, (15, 16, 17)),
    (qt.FMT_I4, 0, 4096, 2048, (31, 32, 33)), (qt.FMT_I8, 0, 4096, 2112, (7, 8, 9)),
])
def test_automatic_arm_larger_experts(host_rules, fmt, gs, D, I, rows):
    check(host_rules, fmt, gs, rows, 2, D, I)
