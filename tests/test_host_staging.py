"""Host-buffer calls stage a large x in chunks of rows, each quantised while the
host copies the next. On the CPU: chunks cover x and start on whole cache
lines, which the host and the GPU never share. On the GPU: calls with and
without the reduce, on both arms, rows that do and do not end on a line,
bit-identical to the oracle."""
import numpy as np
import pytest

from peregrine_amd import qt, synth


@pytest.mark.parametrize("D", [1, 8, 31, 36, 1000, 1001, 5120, 70001, 600000])
def test_chunks_cover_x_on_whole_lines(host_rules, D):
    for total in (1, 2, 33, 37, 192, 531, 4099):
        for n in range(2, 9):
            at = [host_rules.chunk_row_c(total, i, n, D) for i in range(n + 1)]
            assert at[0] == 0 and at[n] == total and at == sorted(at)
            assert all(r * D * 4 % 128 == 0 for r in at[:n]), (total, n, at)
            assert all(b - a <= total / n + 33 for a, b in zip(at, at[1:])) or total < 32 * n


@pytest.mark.gpu
@pytest.mark.parametrize("fmt,ga", [(qt.FMT_I4, 0), (qt.FMT_I8G, 0), (qt.FMT_I4G, 32)])
@pytest.mark.parametrize("arm", [0, 2])
@pytest.mark.parametrize("D,rows", [(5121, [30, 1, 40, 8]), (1001, [400, 7, 131]), (15001, [9, 1, 10]), (5120, [20, 13, 66])])
def test_chunked_calls_match_oracle(orc, fmt, ga, arm, D, rows):
    from peregrine_amd import hip
    assert hip.init([0]) == 1
    total, I = sum(rows), 40
    assert total * D * 4 >= 2 << 19   # two chunks or more
    print("chunked", fmt, ga, arm, D, rows, flush=True)
    rng = np.random.default_rng(D + arm + fmt)
    gpu, ora = [], []
    for _ in rows:
        trip = synth.make_expert(rng, D, I, fmt, 32)
        gpu.append(hip.GpuExpert.upload_grouped(0, trip[0][:2], trip[1][:2], trip[2][:2], D, I, fmt, 32))
        ora.append(tuple(orc.Tensor(t[0], t[1], fmt, i, o, 32) for t, (o, i) in zip(trip, ((I, D), (I, D), (D, I)))))
    s_n = 9
    dst = rng.integers(0, s_n, total)
    rw = rng.uniform(0.1, 1.0, total).astype(np.float32)
    layout = hip.ReduceLayout.build(dst, s_n)
    hip.set_act_group(ga)
    hip.set_arm(arm)
    try:
        for rep in range(2):   # the second call overwrites the first's staging
            x = rng.standard_normal((total, D)).astype(np.float32)
            y = hip.expert_group(gpu, rows, x, D)
            out = hip.expert_group_reduce(gpu, rows, x, D, layout, rw, s_n)
            ref = np.concatenate([orc.expert_swiglu(xe, *o, ga) for xe, o in
                                  zip(np.split(x, np.cumsum(rows)[:-1]), ora)])
            assert np.array_equal(y, ref), rep
            red = np.zeros((s_n, D), np.float32)
            for j in range(total):
                red[dst[j]] = red[dst[j]] + rw[j] * ref[j]
            assert np.array_equal(out, red), rep
    finally:
        hip.set_arm(-1)
        hip.set_act_group(0)
