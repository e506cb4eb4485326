"""Scattered private index rows as offset lists (k44_row_list.hip): fan-ins around whole 32-position
steps, neuron counts that fill no workgroup, ragged tokens, clusters below 16, short segments, one
and four waves per neuron — against the fp64 oracle and the segment gathers."""
import numpy as np
import pytest

from snntome_amd import synth

from wave_cases import TOL, cluster_rows, random_rows, run_sparse_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [-1, 1, 4])
@pytest.mark.parametrize("n_rows,cluster,fan,S,tokens,act,residual", [
    (16, 1, 1, 1, 1, "none", False), (50, 1, 33, 1, 64, "relu", True),
    (208, 1, 257, 1, 130, "silu", False), (30, 8, 96, 1, 300, "gelu", True),
    (64, 2, 72, 3, 65, "sigmoid", False), (48, 1, 60, 15, 100, "leaky_relu", True),
    (50, 1, 64, 16, 64, "relu", True), (26, 8, 96, 24, 130, "gelu", False),
    (37, 1, 310, 31, 256, "silu", False),
])
def test_scattered_private_rows(wavec, orc, tuning, kw, n_rows, cluster, fan, S, tokens, act,
                                residual):
    rng = np.random.default_rng(fan + tokens)
    C, cout = 1500, n_rows * cluster
    rows = (random_rows(rng, n_rows, fan, C) if S == 1 else
            cluster_rows(rng.integers(0, C - S + 1, (n_rows, fan // S)), S))
    w = synth.normal_f16(rng, (cout, fan), 0.1)
    b = synth.normal_f16(rng, (cout,), 0.1)
    out = []
    for rk in (kw, 0):
        tuning("rows", rk)
        y, ref, plan = run_sparse_case(wavec, orc, C=C, tokens=tokens, rows=rows, weights=w, bias=b,
                                       cluster=cluster, act=act, residual=residual, seed=9)
        rep = plan.exec_report()["waves"][0]
        assert rep["path"] == "valu_gather_dot"
        assert rep["kernel"] == ("row_list" if rk else "gather_dot") and (rk <= 0 or rep["ksplit"] == rk)
        assert orc.rel_err(y[:, :tokens], ref[:, :tokens]) <= TOL
        out.append(y[:, :tokens])
        plan.release_gpu()
    assert orc.rel_err(out[0], out[1]) <= TOL


def test_infinities_stay_infinite(wavec, tuning):
    """The last position, which fills up the last step, adds nothing a second time."""
    rng = np.random.default_rng(3)
    C, cout, fan, tokens = 300, 48, 70, 64
    rows = random_rows(rng, cout, fan, C - 1)
    rows.sort(axis=1)
    rows[:, -1] = C - 1
    w = np.abs(synth.normal_f16(rng, (cout, fan), 0.1)) + np.float16(0.01)
    g = wavec.WaveGraph(kv_cache_max_seq=0)
    g.add_input("x", C, 1, tokens, is_1d=True)
    g.add_sparse_wave("w", "x", "y", rows, w, None, cluster=1)
    plan = g.compile()
    x = np.zeros((C, 1, tokens), np.float32)
    x[C - 1, 0, ::2] = np.inf
    y, _ = plan.infer_f32(x)
    assert plan.exec_report()["waves"][0]["kernel"] == "row_list"
    assert np.all(np.isposinf(y[:, 0, ::2])) and np.all(y[:, 0, 1::2] == 0.0)


@pytest.mark.parametrize("C,cout,K,S,tokens,kernel", [
    (131072, 2048, 16, 24, 64, "row_list"),    # few waves
    (65536, 4096, 16, 24, 64, "row_list"),     # 3/8 of the batches, rows within L2
    (131072, 4096, 16, 24, 64, "gather_dot"),  # beyond it
    (20000, 4096, 16, 15, 64, "gather_dot"),   # half of the batches
    (20000, 4096, 4, 15, 64, "row_list"),      # two steps
    (131072, 4096, 16, 8, 128, "row_list"),
    (20000, 4096, 4, 4, 256, "gather_dot"),    # 256-token gathers: few short segments
    (65536, 4096, 8, 15, 256, "row_list"),
    (131072, 4096, 8, 15, 256, "gather_dot"),
    (131072, 4096, 16, 4, 256, "row_list"),
])
def test_automatic_choice(wavec, tuning, C, cout, K, S, tokens, kernel):
    """Each line of the rule from both sides."""
    rng = np.random.default_rng(S)
    starts = (rng.integers(0, (C - S) // 8 + 1, (cout, K)) * 8).astype(np.uint32)
    g = wavec.WaveGraph(kv_cache_max_seq=0)
    g.add_input("x", C, 1, tokens, is_1d=True)
    g.add_cluster_wave("w", "x", "y", starts, S, np.ones((cout, K * S), np.float16), None, cluster=1)
    plan = g.compile()
    plan.init_gpu()
    assert plan.exec_report()["waves"][0]["kernel"] == kernel
    plan.release_gpu()
