"""Private dendritic segments as MFMA job tiles (k44_mfma_jobs.hip): one to several k-steps per
segment, ragged segments and tokens, tiles of one job to full ones, neurons sharing segments in
clusters below 16, residuals — against the fp64 oracle and the VALU gathers."""
import numpy as np
import pytest

from snntome_amd import synth

from wave_cases import TOL, cluster_rows, run_sparse_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C,n_rows,cluster,K,S,tokens,act,residual", [
    (400, 208, 1, 3, 32, 1, "none", False),     # windows of one k-step, many jobs at one address
    (300, 48, 1, 16, 33, 64, "relu", True),     # K of two whole reduction batches
    (5000, 48, 1, 5, 100, 130, "silu", False),  # jobs far apart: tiles of one or two
    (2000, 26, 8, 9, 127, 65, "gelu", True),    # clusters: the same segment 8 times
    (3000, 64, 2, 1, 512, 300, "sigmoid", False),
    (160, 16, 1, 4, 64, 100, "relu", False),    # two tiles
])
def test_private_segments(wavec, orc, tuning, C, n_rows, cluster, K, S, tokens, act, residual):
    rng = np.random.default_rng(C + S)
    cout = n_rows * cluster
    starts = rng.integers(0, C - S + 1, (n_rows, K))
    starts[0, 0], starts[-1, -1] = 0, C - S
    w = synth.normal_f16(rng, (cout, K * S), 0.1)
    b = synth.normal_f16(rng, (cout,), 0.1)
    out = {}
    for jobs in (1, 0):
        tuning("jobs", jobs)
        y, ref, plan = run_sparse_case(wavec, orc, C=C, tokens=tokens, rows=cluster_rows(starts, S),
                                       weights=w, bias=b, cluster=cluster, act=act,
                                       residual=residual, seed=5)
        rep = plan.exec_report()
        assert rep["waves"][0]["kernel"] == ("jobs" if jobs else "gather_dot"), rep
        assert rep["launches_per_run"] == 1 + jobs
        out[jobs] = y[:, :tokens]
        assert orc.rel_err(out[jobs], ref[:, :tokens]) <= TOL
        plan.release_gpu()
    assert orc.rel_err(out[1], out[0]) <= TOL


def test_unread_infinities_stay_out(wavec, tuning):
    """Neurons meet an infinity or a NaN only where a segment of theirs reads it, whatever else
    shares their tile."""
    rng = np.random.default_rng(8)
    C, cout, K, S, tokens = 600, 96, 4, 40, 70
    starts = rng.integers(0, C - S + 1, (cout, K))
    w = np.abs(synth.normal_f16(rng, (cout, K * S), 0.1)) + np.float16(0.01)
    x = rng.random((C, 1, tokens)).astype(np.float32)
    x[300, 0, 3], x[301, 0, 69] = np.inf, np.nan
    tuning("jobs", 1)
    g = wavec.WaveGraph(kv_cache_max_seq=0)
    g.add_input("x", C, 1, tokens, is_1d=True)
    g.add_sparse_wave("w", "x", "y", cluster_rows(starts, S), w, None, cluster=1)
    plan = g.compile()
    y = plan.infer_f32(x)[0][:, 0, :]
    assert plan.exec_report()["waves"][0]["kernel"] == "jobs"
    reads = lambda r: np.any((starts <= r) & (r < starts + S), axis=1)
    assert 0 < reads(300).sum() < cout
    assert np.array_equal(np.isposinf(y[:, 3]), reads(300))
    assert np.array_equal(np.isnan(y[:, 69]), reads(301))
    rest = np.delete(y, [3, 69], axis=1)
    assert np.all(np.isfinite(rest))
    syn = (starts[:, :, None] + np.arange(S)).reshape(cout, K * S)
    xh = np.where(np.isfinite(x), x, 0).astype(np.float16).astype(np.float64)[:, 0, :]
    ref = np.einsum("js,jst->jt", w.astype(np.float64), xh[syn])
    assert np.abs(rest - np.delete(ref, [3, 69], axis=1)).max() <= 2.0 ** -10 * ref.max()


@pytest.mark.parametrize("inf_tokens", [1, 70])
def test_infinities_keep_their_signs(wavec, tuning, inf_tokens):
    """What infinities and NaNs of the rows give: +inf, -inf, NaN where both signs or a zero weight
    meet one, as the gathers give (which multiply each row of a segment by its weight)."""
    rng = np.random.default_rng(inf_tokens)
    C, cout, K, S, tokens = 400, 112, 3, 72, 70
    starts = rng.integers(0, C - S + 1, (cout, K))
    w = synth.normal_f16(rng, (cout, K * S), 0.1)
    w[rng.random(w.shape) < 0.02] = 0.0
    w[rng.random(w.shape) < 0.01] = np.float16(-0.0)
    w[0, 0], w[1, 5] = np.float16(6e-8), np.float16(-6e-8)  # subnormal
    x = rng.standard_normal((C, 1, tokens)).astype(np.float32)
    for t in range(inf_tokens):
        for v in (np.inf, -np.inf, np.nan)[:1 + t % 3]:
            x[rng.integers(0, C), 0, t] = v
    got = []
    for jobs in (1, 0):
        tuning("jobs", jobs)
        g = wavec.WaveGraph(kv_cache_max_seq=0)
        g.add_input("x", C, 1, tokens, is_1d=True)
        g.add_sparse_wave("w", "x", "y", cluster_rows(starts, S), w, None, cluster=1, act="none")
        plan = g.compile()
        got.append(plan.infer_f32(x)[0][:, 0, :])
        assert plan.exec_report()["waves"][0]["kernel"] == ("jobs" if jobs else "gather_dot")
        plan.release_gpu()
    a, b = got
    assert np.isposinf(b).any() and np.isneginf(b).any() and np.isnan(b).any()
    for kind in (np.isposinf, np.isneginf, np.isnan):
        assert np.array_equal(kind(a), kind(b))
    fin = np.isfinite(b)
    # two fp16 roundings of fp32 sums of 216 products: half an ulp (2^-11) each, and 2^-20 of the
    # largest sums between the orders
    assert np.abs(a[fin] - b[fin]).max() <= 2.0 ** -10 * np.abs(b[fin]).max()


def test_infinite_weights_stay_on_the_gathers(wavec, tuning):
    tuning("jobs", 1)
    starts = np.arange(64)[:, None] * 4
    w = np.ones((64, 64), np.float16)
    for v, kernel in ((1.0, "jobs"), (np.inf, "gather_dot"), (np.nan, "gather_dot")):
        w[3, 7] = v
        g = wavec.WaveGraph(kv_cache_max_seq=0)
        g.add_input("x", 400, 1, 64, is_1d=True)
        g.add_sparse_wave("w", "x", "y", cluster_rows(starts, 64), w, None, cluster=1)
        plan = g.compile()
        plan.init_gpu()
        assert plan.exec_report()["waves"][0]["kernel"] == kernel
        plan.release_gpu()


@pytest.mark.parametrize("C,cout,K,S,tokens,kernel", [
    (65536, 4096, 8, 64, 64, "jobs"),            # segments overlap 32 times
    (200_000, 512, 8, 128, 64, "jobs"),          # few jobs per window, 11 MiB of fragments
    (1 << 18, 2048, 4, 256, 128, "jobs"),        # 54 MB of fragments for 4 MB of weights, 67 MB of rows
    (1 << 20, 2048, 4, 256, 128, "gather_dot"),  # 109 MB: their traffic outweighs the overlap
    (1 << 20, 4096, 8, 64, 64, "gather_dot"),    # 86 MB
    (1 << 19, 2048, 8, 512, 64, "gather_dot"),   # 210 MB for 17 of weights and 67 of rows: too much memory
])
def test_automatic_choice(wavec, tuning, C, cout, K, S, tokens, kernel):
    """Job tiles where segments overlap; not where their padded fragments would
    grow without bound or cost more than the gathers."""
    rng = np.random.default_rng(S)
    starts = (rng.integers(0, (C - S) // 8 + 1, (cout, K)) * 8).astype(np.uint32)
    g = wavec.WaveGraph(kv_cache_max_seq=0)
    g.add_input("x", C, 1, tokens, is_1d=True)
    g.add_cluster_wave("w", "x", "y", starts, S, np.ones((cout, K * S), np.float16), None, cluster=1)
    plan = g.compile()
    plan.init_gpu()
    assert plan.exec_report()["waves"][0]["kernel"] == kernel
    plan.release_gpu()
