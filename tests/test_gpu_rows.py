"""Row-table MFMA waves (k44_mfma_rows.hip): clusters sharing index rows of any positions, at the
edges of its tiles — fan-ins around whole k-steps, every block count per workgroup, ragged token
tiles — for each number of waves per tile, against the fp64 oracle and the VALU gathers."""
import numpy as np
import pytest

from oracle import cnn_oracle as co
from snntome_amd import synth

from wave_cases import TOL, random_rows, run_sparse_case, stride_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [-1, 1, 4, 8])
@pytest.mark.parametrize("cluster,fan,tokens,act,residual", [
    (16, 64, 1, "none", False), (32, 65, 64, "relu", True), (48, 95, 100, "silu", False),
    (64, 257, 300, "gelu", True), (96, 1000, 130, "sigmoid", False), (128, 96, 40, "leaky_relu", True),
    (256, 130, 320, "relu", False), (16, 1, 64, "none", False), (32, 31, 20, "relu", False),
])
def test_scattered_rows(wavec, orc, tuning, kw, cluster, fan, tokens, act, residual):
    rng = np.random.default_rng(cluster * 10 + fan)
    tuning("rows", kw)
    C, cout = 2000, 3 * cluster
    w = synth.normal_f16(rng, (cout, fan), 0.1)
    b = synth.normal_f16(rng, (cout,), 0.1)
    rows = random_rows(rng, 3, fan, C)
    y, ref, plan = run_sparse_case(wavec, orc, C=C, tokens=tokens, rows=rows, weights=w, bias=b,
                                   cluster=cluster, act=act, residual=residual, seed=31)
    rep = plan.exec_report()["waves"][0]
    assert rep["path"] == "mfma_rows" and (kw < 0 or rep["ksplit"] == kw), rep
    assert orc.rel_err(y[:, :tokens], ref[:, :tokens]) <= TOL
    tuning("rows", 0)
    v, _, plan = run_sparse_case(wavec, orc, C=C, tokens=tokens, rows=rows, weights=w, bias=b,
                                 cluster=cluster, act=act, residual=residual, seed=31)
    assert plan.exec_report()["waves"][0]["path"] == "valu_gather_dot"
    assert orc.rel_err(y[:, :tokens], v[:, :tokens]) <= TOL


def test_infinities_stay_infinite(wavec, tuning):
    """Positions that only fill up the last k-step add nothing: an infinite activation read by
    every neuron (as its last synapse, the one padding repeats) gives infinities, not NaN."""
    rng = np.random.default_rng(3)
    C, cluster, fan, tokens = 300, 32, 70, 64
    rows = random_rows(rng, 2, fan, C - 1)
    rows.sort(axis=1)
    rows[:, -1] = C - 1
    w = np.abs(synth.normal_f16(rng, (2 * cluster, fan), 0.1)) + np.float16(0.01)
    g = wavec.WaveGraph(kv_cache_max_seq=0)
    g.add_input("x", C, 1, tokens, is_1d=True)
    g.add_sparse_wave("w", "x", "y", rows, w, None, cluster=cluster)
    plan = g.compile()
    x = np.zeros((C, 1, tokens), np.float32)
    x[C - 1, 0, ::2] = np.inf
    y, _ = plan.infer_f32(x)
    assert plan.exec_report()["waves"][0]["path"] == "mfma_rows"
    assert np.all(np.isposinf(y[:, 0, ::2])) and np.all(y[:, 0, 1::2] == 0.0)


@pytest.mark.parametrize("tile,cout", [(16, 200), (64, 150)])
def test_pruned_tiles_with_empty_slots(wavec, orc, tile, cout):
    """Pattern-sorted tiles whose segments are not whole k-steps: outputs through cout_map, empty
    slots not stored."""
    rng = np.random.default_rng(cout)
    n_cl, K, S, tokens = 7, 4, 24, 70
    C = n_cl * S
    pick = np.argsort(rng.random((cout, n_cl)), axis=1)[:, :K]
    starts = (pick * S).astype(np.uint32)
    w = synth.normal_f16(rng, (cout, K * S), 0.1)
    b = synth.normal_f16(rng, (cout,), 0.1)
    g = wavec.WaveGraph(kv_cache_max_seq=0)
    g.add_input("x", C, 1, tokens, is_1d=True)
    g.add_pruned_wave("p", "x", "y", starts, S, w, b, tile=tile, act="silu")
    plan = g.compile()
    plan.init_gpu()
    assert {r["path"] for r in plan.exec_report()["waves"]} == {"mfma_rows"}
    plan.fill_input_uniform(7)
    plan.execute(1)
    st = stride_of(tokens)
    canvas = plan.read_canvas(0, int(plan.summary["canvas_elems"]))
    x0, y0 = int(plan.cmds[0]["src_off"]), int(plan.cmds[0]["y_off"])
    ref = orc.wave_f64(canvas, (x0 + starts.astype(np.uint64) * st).ravel(), w, b, None, K, S, 1,
                       st, st, st, "silu")
    y = canvas[y0:y0 + cout * st].view(np.float16).reshape(cout, st).astype(np.float64)
    assert orc.rel_err(y[:, :tokens], ref[:, :tokens]) <= TOL


@pytest.mark.parametrize("kw", [-1, 1, 4, 8])
@pytest.mark.parametrize("frames,H,W,cin,cout,res", [
    (1, 9, 20, 16, 16, True), (1, 5, 128, 8, 48, False), (3, 7, 21, 24, 24, True),
    (1, 3, 5, 12, 96, False), (1, 40, 50, 3, 16, False),
])
def test_image_convolutions(wavec, orc, tuning, kw, frames, H, W, cin, cout, res):
    """3x3 convolutions over channel counts that make no whole k-steps, on padded planes (aligned
    and masked widths, several frames), with a residual; halos of the output stay zero."""
    rng = np.random.default_rng(H * W + cin)
    tuning("rows", kw)
    w = (rng.standard_normal((cout, cin, 3, 3)) * 0.1).astype(np.float16)
    b = (rng.standard_normal(cout) * 0.1).astype(np.float16)
    g = wavec.WaveGraph(kv_cache_max_seq=0, batch_size=frames)
    g.add_input("img", cin, H, W)
    g.add_conv2d("c", "img", "y", cin, cout, 3, 3, w.astype(np.float32), b.astype(np.float32),
                 stride=1, pad=1, act="silu", res_blob="img" if res else None)
    plan = g.compile()
    plan.init_gpu()
    assert plan.exec_report()["waves"][0]["path"] == "mfma_rows"
    lay = co.Layout2D(H, W, frames)
    x = rng.standard_normal((frames, cin, H, W)).astype(np.float16)
    region = np.zeros(cin * lay.channel_stride, np.float16)
    region[lay.offsets(cin).ravel()] = x.ravel()
    c = plan.cmds[0]
    plan.write_canvas(int(c["src_off"]), region)
    plan.execute(1)
    out = plan.read_canvas(int(c["y_off"]), cout * lay.channel_stride).view(np.float16)
    ref = co.conv2d_f64(x, w, b, 1, 1, "silu", x if res else None)
    assert orc.rel_err(out[lay.offsets(cout)].astype(np.float64), ref) <= TOL
    halo = np.ones(cout * lay.channel_stride, bool)
    halo[lay.offsets(cout).ravel()] = False
    assert not out[halo].any()


@pytest.mark.parametrize("tile,tokens", [(64, 100), (64, 512), (32, 200)])
def test_grouped_dense_tiles(wavec, orc, tile, tokens):
    """Sub-waves of a pruned projection (dense tiles, several row lengths, outputs through
    cout_map) share one row-table launch; the launch equals its commands run one by one bit for
    bit and the per-neuron oracle within tolerance."""
    rng = np.random.default_rng(tile + tokens)
    n_cl, K, S, cout = 4, 2, 64, 1000
    C = n_cl * S
    pick = np.argsort(rng.random((cout, n_cl)), axis=1)[:, :K]
    starts = (pick * S).astype(np.uint32)
    w = synth.normal_f16(rng, (cout, K * S), 0.1)
    b = synth.normal_f16(rng, (cout,), 0.1)
    g = wavec.WaveGraph(kv_cache_max_seq=0)
    g.add_input("x", C, 1, tokens, is_1d=True)
    g.add_pruned_wave("p", "x", "y", starts, S, w, b, tile=tile, act="silu")
    plan = g.compile()
    plan.init_gpu()
    rep = plan.exec_report()
    assert {r["kernel"] for r in rep["waves"]} == {"rows"} and len(rep["waves"]) >= 2
    assert len(rep["groups"]) == 1 and rep["launches_per_run"] == 1
    plan.fill_input_uniform(7)
    plan.execute(1)
    st = stride_of(tokens)
    x0, y0 = int(plan.cmds[0]["src_off"]), int(plan.cmds[0]["y_off"])
    canvas = plan.read_canvas(0, int(plan.summary["canvas_elems"]))
    plan.write_canvas(y0, np.zeros(cout * st, np.uint16))
    plan.execute_range(0, len(plan.cmds))
    assert np.array_equal(plan.read_canvas(y0, cout * st), canvas[y0:y0 + cout * st])
    ref = orc.wave_f64(canvas, (x0 + starts.astype(np.uint64) * st).ravel(), w, b, None, K, S, 1,
                       st, st, st, "silu")
    y = canvas[y0:y0 + cout * st].view(np.float16).reshape(cout, st).astype(np.float64)
    assert orc.rel_err(y[:, :tokens], ref[:, :tokens]) <= TOL


def test_long_rows_keep_their_split(wavec):
    """Few tiles of very long rows stay on the register-staged kernel, wider ones do not."""
    kernels = {}
    for tokens in (64, 320):
        g = wavec.WaveGraph(kv_cache_max_seq=0)
        g.add_input("x", 8192, 1, tokens, is_1d=True)
        g.add_cluster_wave("w", "x", "y", np.zeros((16, 16), np.uint32), 512,
                           np.zeros((16 * 64, 8192), np.float16), None, cluster=64)
        plan = g.compile()
        plan.init_gpu()
        kernels[tokens] = plan.exec_report()["waves"][0]["kernel"]
        plan.release_gpu()
    assert kernels == {64: "tile", 320: "rows"}


@pytest.mark.parametrize("frames,H,W,cin,cout,kw", [
    (1, 5, 128, 8, 16, 1), (3, 7, 21, 24, 48, 4), (1, 3, 5, 16, 16, 8), (2, 40, 50, 3, 32, -1),
])
def test_halos_are_cleared(wavec, tuning, frames, H, W, cin, cout, kw):
    """Whatever the output planes held, all but the image pixels is zero after the convolution,
    and a second run gives the same bits."""
    rng = np.random.default_rng(W)
    tuning("rows", kw)
    w = rng.standard_normal((cout, cin, 3, 3)).astype(np.float32)
    g = wavec.WaveGraph(kv_cache_max_seq=0, batch_size=frames)
    g.add_input("img", cin, H, W)
    g.add_conv2d("c", "img", "y", cin, cout, 3, 3, w, np.ones(cout, np.float32), stride=1, pad=1)
    plan = g.compile()
    plan.init_gpu()
    lay = co.Layout2D(H, W, frames)
    x = np.zeros(cin * lay.channel_stride, np.float16)
    x[lay.offsets(cin).ravel()] = rng.standard_normal(frames * cin * H * W).astype(np.float16)
    plan.write_canvas(int(plan.cmds[0]["src_off"]), x)
    plan.execute(1)
    y0, n = int(plan.cmds[0]["y_off"]), cout * lay.channel_stride
    first = plan.read_canvas(y0, n)
    plan.write_canvas(y0, np.full(n, 0x3c00, np.uint16))
    plan.execute(1)
    out = plan.read_canvas(y0, n)
    halo = np.ones(n, bool)
    halo[lay.offsets(cout).ravel()] = False
    assert not out[halo].any() and first[~halo].any()
    assert np.array_equal(out, first)
