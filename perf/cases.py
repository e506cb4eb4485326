"""Performance cases: what users of the framework run, through its public entry points.

Families (field "kind"):
  token64   the stand-alone Token64 wave on caller-owned device memory (forward_token64_f16)
  sparse    one plan wave of neurons in clusters that share an index row of scattered synapses
            (add_sparse_wave), inputs resident on the device
  segments  one plan wave of dendritic clusters (add_cluster_wave): K runs of S consecutive
            positions per neuron, private to it (cluster 1) or shared by a tile of neurons
  chain     a plan of several private-segment waves, each reading the input and earlier outputs
  block     a gated MLP block of dense layers with RMSNorm and residual, host fp32 in and out
            (infer_f32)
  image     a convolution block (3x3, stride 2, slice, residual, concat, 5x5 pooling, 1x1) on
            one image, host fp32 in and out (infer_f32)
  prefill   the pruned decoder of snntome_amd.synth over whole prompts, token ids to logits
  decode    the same decoder, one token per request against the carried token-shift state

Plan outputs are read into page-locked memory that the caller keeps, as a serving loop does.
"""
import ctypes
import math

import numpy as np
import torch

from snntome_amd import synth, wavec


# ------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # One tile of tokens through a small layer: a single interactive request, latency bound.
        dict(name="token64_one_tile", kind="token64", Cin=4096, Cout=2048, B=512, cluster=64,
             batch=64),
        # The whitepaper's streaming shape: 512 tokens gathered from a substrate far beyond caches.
        dict(name="token64_stream", kind="token64", Cin=4_000_000, Cout=8192, B=1024,
             cluster=128, batch=512),
        # Fine clusters, an odd number of 16-synapse blocks and a ragged batch, substrate in cache.
        dict(name="token64_fine_odd", kind="token64", Cin=60_000, Cout=4080, B=720, cluster=48,
             batch=300),
        # Scattered synapses shared by clusters of 64: the connectome the plan format is made for.
        dict(name="sparse_shared", kind="sparse", cin=65536, cout=4096, fan=512, cluster=64,
             tokens=256, act="relu"),
        # The same in small, ragged sizes: a fan-in off every block size, 100 tokens, clusters of 16.
        dict(name="sparse_small_odd", kind="sparse", cin=5000, cout=992, fan=200, cluster=16,
             tokens=100, act="silu"),
        # Private dendritic clusters on a cache-resident substrate (the single-wave plumbing size).
        dict(name="segments_private", kind="segments", cin=65536, cout=4096, K=8, S=64, cluster=1,
             tokens=64, act="relu"),
        # Tiles of 64 neurons sharing long segments: the matrix-core wave, GELU.
        dict(name="segments_tiles", kind="segments", cin=262144, cout=4096, K=16, S=512,
             cluster=64, tokens=512, act="gelu"),
        # Eight dependent waves of private segments over one canvas.
        dict(name="chain_8_waves", kind="chain", cin=32768, cout=4096, K=16, S=128, waves=8,
             tokens=128),
        # A dense gated MLP block over 200 tokens, called with host arrays.
        dict(name="block_infer", kind="block", d=1024, ffn=2816, tokens=200),
        # A convolution block on one 160x160 feature map, called with host arrays.
        dict(name="image_infer", kind="image", c=32, H=160, W=160),
        # Four prompts of 512 tokens through a two-layer pruned decoder, all logits.
        dict(name="decoder_prefill", kind="prefill", layers=2, d=2048, ffn=5632, S=512,
             vocab=4096, requests=4, prompt=512),
        # One decode step for 16 requests (the host samples: ids in, logits out).
        dict(name="decoder_step", kind="decode", layers=4, d=2048, ffn=5632, S=512, vocab=4096,
             requests=16, prompt=1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["token64", "token64", "sparse", "sparse", "segments", "segments", "chain",
                       "block", "image", "prefill", "decode"])
    if kind == "token64":
        cluster = rng.choice([16, 32, 48, 64, 96, 128, 256])
        return dict(kind=kind, Cin=_log(rng, 1024, 4_000_000),
                    Cout=cluster * max(1, _log(rng, 256, 8192) // cluster),
                    B=16 * _log(rng, 4, 64), cluster=cluster, batch=_log(rng, 1, 512))
    if kind == "sparse":
        cluster = rng.choice([1, 16, 32, 64, 128])
        top = 1024 if cluster > 1 else 256
        return dict(kind=kind, cin=_log(rng, 2048, 65536),
                    cout=max(128, _log(rng, 256, 4096) // 128 * 128), fan=_log(rng, 32, top),
                    cluster=cluster, tokens=_log(rng, 4, 256),
                    act=rng.choice(["relu", "silu", "gelu", "none"]))
    if kind == "segments":
        if rng.random() < 0.5:
            return dict(kind=kind, cin=_log(rng, 8192, 131072), cout=16 * _log(rng, 32, 512),
                        K=rng.randint(2, 12), S=rng.choice([16, 24, 32, 64, 100, 128]), cluster=1,
                        tokens=_log(rng, 8, 256), act=rng.choice(["relu", "sigmoid"]))
        cluster = rng.choice([16, 32, 64, 128])
        return dict(kind=kind, cin=_log(rng, 16384, 262144), cout=128 * _log(rng, 4, 32),
                    K=rng.randint(2, 16), S=rng.choice([32, 64, 128, 256, 512]), cluster=cluster,
                    tokens=_log(rng, 8, 512), act=rng.choice(["gelu", "leaky_relu"]))
    if kind == "chain":
        return dict(kind=kind, cin=_log(rng, 8192, 32768), cout=256 * _log(rng, 2, 16),
                    K=2 * rng.randint(2, 8), S=rng.choice([32, 64, 128]), waves=rng.randint(2, 8),
                    tokens=_log(rng, 16, 128))
    if kind == "block":
        return dict(kind=kind, d=32 * _log(rng, 8, 48), ffn=32 * _log(rng, 16, 128),
                    tokens=_log(rng, 1, 512))
    if kind == "image":
        return dict(kind=kind, c=rng.choice([8, 16, 24, 32, 48]), H=2 * _log(rng, 10, 80),
                    W=2 * _log(rng, 10, 80))
    if kind == "prefill":
        d = rng.choice([1024, 2048])
        return dict(kind=kind, layers=rng.randint(1, 2), d=d, ffn=d * 11 // 4, S=d // 4,
                    vocab=128 * rng.randint(8, 32), requests=rng.randint(1, 4),
                    prompt=_log(rng, 32, 512))
    d = rng.choice([1024, 2048])
    return dict(kind="decode", layers=rng.randint(1, 4), d=d, ffn=d * 11 // 4, S=d // 4,
                vocab=128 * rng.randint(8, 32), requests=_log(rng, 1, 64), prompt=1)


# -------------------------------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _randn(g, shape, sigma):
    return torch.randn(shape, generator=g, device="cuda") * sigma


def _uniform(g, shape):
    """fp16 activations, uniform in [-1, 1), 2**28 values at a time."""
    x = torch.empty(shape, dtype=torch.float16, device="cuda")
    for part in x.view(-1).split(1 << 28):
        part.copy_(torch.rand(part.shape, generator=g, device="cuda").mul_(2.0).sub_(1.0))
    return x


def _np16(t):
    return t.half().cpu().numpy()


def _token64_inputs(c, seed):
    g = _gen(seed)
    tiles, cl, B = (c["batch"] + 63) // 64, c["cluster"], c["B"]
    return dict(
        X=_uniform(g, (tiles, c["Cin"], 64)),
        idx=torch.randint(0, c["Cin"], (c["Cout"] // cl, B), generator=g, device="cuda",
                          dtype=torch.int32),
        w=_randn(g, (c["Cout"], B), 1.0 / math.sqrt(B)).half(),
        bias=_randn(g, (c["Cout"],), 0.01).half())


def _starts(g, n, cin, S, align):
    slots = max(1, (cin - S) // align + 1)
    return (torch.randint(0, slots, (n,), generator=g, device="cuda") * align)


def _wave_inputs(c, seed):
    """Input activations [cin][tokens], synapse positions [rows][fan], weights and bias."""
    g = _gen(seed)
    x = _uniform(g, (c["cin"], c["tokens"]))
    rows = c["cout"] // c["cluster"]
    if c["kind"] == "sparse":
        fan = c["fan"]
        pos = torch.randint(0, c["cin"], (rows, fan), generator=g, device="cuda")
        starts = None
    else:
        fan = c["K"] * c["S"]
        align = 64 if c["cluster"] > 1 and c["S"] % 64 == 0 else 8
        starts = _starts(g, rows * c["K"], c["cin"], c["S"], align).view(rows, c["K"])
        pos = (starts[:, :, None] + torch.arange(c["S"], device="cuda")).view(rows, fan)
    w = _randn(g, (c["cout"], fan), 1.0 / math.sqrt(fan)).half()
    return dict(x=x, pos=pos, starts=starts, w=w, bias=_randn(g, (c["cout"],), 0.01).half())


def _chain_inputs(c, seed):
    """Wave i reads half of its segments from the tensor before it, half from all earlier ones."""
    g = _gen(seed)
    x = _uniform(g, (c["cin"], c["tokens"]))
    K, S, n = c["K"], c["S"], c["cout"]
    waves = []
    for i in range(c["waves"]):
        widths = [c["cin"]] + [n] * i
        offs = np.concatenate([[0], np.cumsum(widths)])
        prev = offs[i] + _starts(g, n * (K // 2), widths[i], S, 8)
        p = torch.tensor(widths, dtype=torch.float32, device="cuda")
        pick = torch.multinomial(p, n * (K // 2), replacement=True, generator=g)
        span = torch.tensor([max(1, (v - S) // 8 + 1) for v in widths], device="cuda")[pick]
        inside = (torch.rand(n * (K // 2), generator=g, device="cuda") * span).long()
        inside = torch.minimum(inside, span - 1) * 8
        anyw = torch.tensor(offs[:-1], device="cuda")[pick] + inside
        st = torch.cat([prev.view(n, K // 2), anyw.view(n, K // 2)], 1)
        waves.append(dict(starts=st, w=_randn(g, (n, K * S), 1.0 / math.sqrt(K * S)).half(),
                          bias=_randn(g, (n,), 0.01).half()))
    return dict(x=x, waves=waves)


def _block_inputs(c, seed):
    g = _gen(seed)
    d, f = c["d"], c["ffn"]
    return dict(x=_randn(g, (d, c["tokens"]), 1.0), gamma=1.0 + _randn(g, (d,), 0.1),
                wg=_randn(g, (f, d), 1.0 / math.sqrt(d)), wu=_randn(g, (f, d), 1.0 / math.sqrt(d)),
                wd=_randn(g, (d, f), 1.0 / math.sqrt(f)), bd=_randn(g, (d,), 0.01))


def _image_inputs(c, seed):
    g = _gen(seed)
    n = c["c"]

    def conv(cout, cin, k):
        return (_randn(g, (cout, cin, k, k), 1.4 / math.sqrt(cin * k * k)),
                _randn(g, (cout,), 0.05))

    return dict(x=_randn(g, (n, c["H"], c["W"]), 1.0), down=conv(2 * n, n, 3),
                cv1=conv(2 * n, 2 * n, 1), m1=conv(n, n, 3), m2=conv(n, n, 3),
                cv2=conv(2 * n, 3 * n, 1), cv3=conv(2 * n, 4 * n, 1))


def _decoder_inputs(c, seed):
    """The weights of synth.llm_weights, drawn on the GPU, and prompt ids."""
    g = _gen(seed)
    spec = synth.LLMSpec(layers=c["layers"], d=c["d"], ffn=c["ffn"], vocab=c["vocab"], S=c["S"],
                         requests=c["requests"], prompt=c["prompt"])

    def proj(fan_in, cout):
        K = spec.kept(fan_in)
        pick = torch.rand((cout, fan_in // spec.S), generator=g, device="cuda").argsort(1)[:, :K]
        w = _randn(g, (cout, K * spec.S), 1.0 / math.sqrt(K * spec.S)).half()
        return synth.Projection((pick * spec.S).cpu().numpy().astype(np.uint32),
                                w.cpu().numpy(), _np16(_randn(g, (cout,), 0.01)))

    embed = _np16(_randn(g, (spec.vocab, spec.d), 1.0))
    mix, layers = [], []
    for _ in range(spec.layers):
        m = torch.rand((spec.d, spec.rf), generator=g, device="cuda") + 0.05
        m[:, 0] += spec.rf
        mix.append(_np16(m / m.sum(1, keepdim=True)))
        p = {k: proj(spec.d, spec.d) for k in ("q", "k", "v", "o")}
        p["g"], p["u"] = proj(spec.d, spec.ffn), proj(spec.d, spec.ffn)
        p["dn"] = proj(spec.ffn, spec.d)
        layers.append(p)
    wts = synth.LLMWeights(embed, mix, layers, proj(spec.d, spec.vocab))
    ids = torch.randint(0, spec.vocab, (spec.requests * spec.prompt,), generator=g, device="cuda")
    return spec, wts, ids.cpu().numpy().astype(np.uint32)


# ------------------------------------------------------------------------------------- prepare
class _Output:
    """A plan's output rows, read into page-locked memory that is kept between calls."""

    def __init__(self, plan, off, rows, tokens):
        self.plan, self.off, self.rows, self.cols = plan, off, rows, tokens
        self.stride = (tokens + 63) // 64 * 64
        self.host = torch.empty((rows, tokens), dtype=torch.float16, pin_memory=True)
        self.ptr = ctypes.cast(self.host.data_ptr(), ctypes.POINTER(ctypes.c_uint16))

    def read(self):
        if wavec.get_lib().wavec_gpu_read_canvas_2d(self.plan._handle, self.off, self.rows,
                                                    self.stride, self.cols, self.ptr) != 0:
            raise RuntimeError(wavec.last_error())
        return self.host


def _rows_to_canvas(plan, x):
    """Puts [channels][tokens] fp16 into the plan input (64-token row stride)."""
    ch, tok = x.shape
    pad = torch.zeros((ch, (tok + 63) // 64 * 64), dtype=torch.float16, device="cuda")
    pad[:, :tok] = x
    plan.write_canvas(0, pad.cpu().numpy())


def _wave_plan(c, seed):
    i = _wave_inputs(c, seed)
    g = wavec.WaveGraph(kv_cache_max_seq=0)
    g.add_input("x", c["cin"], 1, c["tokens"], is_1d=True)
    w, b = i["w"].cpu().numpy(), i["bias"].cpu().numpy()
    if c["kind"] == "sparse":
        g.add_sparse_wave("wave", "x", "y", i["pos"].cpu().numpy(), w, b, cluster=c["cluster"],
                          act=c["act"])
    else:
        g.add_cluster_wave("wave", "x", "y", i["starts"].cpu().numpy(), c["S"], w, b,
                           cluster=c["cluster"], act=c["act"])
    g.set_output("y")
    plan = g.compile()
    plan.init_gpu()
    _rows_to_canvas(plan, i["x"])
    return dict(plan=plan, out=_Output(plan, int(plan.cmds[-1]["y_off"]), c["cout"], c["tokens"]))


def _chain_plan(c, seed):
    i = _chain_inputs(c, seed)
    specs = [synth.WaveSpec(f"wave{k}", c["cout"], c["K"], c["S"], 1,
                            v["starts"].cpu().numpy().astype(np.uint32), v["w"].cpu().numpy(),
                            v["bias"].cpu().numpy(), "relu",
                            ["x"] + [f"y{j}" for j in range(k)])
             for k, v in enumerate(i["waves"])]
    plan = synth.build_graph(synth.Workload("chain", c["cin"], c["tokens"], 0, specs)).compile()
    plan.init_gpu()
    _rows_to_canvas(plan, i["x"])
    return dict(plan=plan, out=_Output(plan, int(plan.cmds[-1]["y_off"]), c["cout"], c["tokens"]))


def _block_plan(c, seed):
    i = {k: v.cpu().numpy() for k, v in _block_inputs(c, seed).items()}
    d, f = c["d"], c["ffn"]
    g = wavec.WaveGraph(kv_cache_max_seq=0)
    g.add_input("x", d, 1, c["tokens"], is_1d=True)
    g.add_rmsnorm("norm", "x", "n", d, i["gamma"])
    g.add_linear("gate", "n", "g", d, f, i["wg"], act="silu")
    g.add_linear("up", "n", "u", d, f, i["wu"])
    g.add_swiglu("mul", "g", "u", "h")
    g.add_linear("down", "h", "y", f, d, i["wd"], i["bd"], res_blob="x")
    g.set_output("y")
    plan = g.compile()
    plan.init_gpu()
    return dict(plan=plan, x=i["x"])


def _image_plan(c, seed):
    i = _image_inputs(c, seed)
    n = c["c"]

    def p(name):
        return [t.cpu().numpy() for t in i[name]]

    g = wavec.WaveGraph(kv_cache_max_seq=0)
    g.add_input("img", n, c["H"], c["W"])
    g.add_conv2d("down", "img", "a", n, 2 * n, 3, 3, *p("down"), stride=2, pad=1)
    g.add_conv2d("cv1", "a", "b", 2 * n, 2 * n, 1, 1, *p("cv1"))
    g.add_slice("halves", "b", ["b0", "b1"], [n, n])
    g.add_conv2d("m1", "b1", "t", n, n, 3, 3, *p("m1"), pad=1)
    g.add_conv2d("m2", "t", "b2", n, n, 3, 3, *p("m2"), pad=1, res_blob="b1")
    g.add_concat("cat", ["b0", "b1", "b2"], "cc")
    g.add_conv2d("cv2", "cc", "e", 3 * n, 2 * n, 1, 1, *p("cv2"))
    g.add_maxpool("pool", "e", "p", kernel_size=5, stride=1, pad=2)
    g.add_concat("cat2", ["e", "p"], "ep")
    g.add_conv2d("cv3", "ep", "y", 4 * n, 2 * n, 1, 1, *p("cv3"))
    g.set_output("y")
    plan = g.compile()
    plan.init_gpu()
    return dict(plan=plan, x=i["x"].cpu().numpy())


def _decoder_plan(c, seed):
    spec, wts, ids = _decoder_inputs(c, seed)
    plan = synth.build_llm_graph(spec, wts, decode=c["kind"] == "decode").compile()
    plan.init_gpu()
    head = next(x for x in plan.cmds if x["name"].startswith("head"))
    return dict(plan=plan, ids=ids,
                out=_Output(plan, int(head["y_off"]), spec.vocab, spec.requests * spec.prompt))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "token64":
        i = _token64_inputs(case, seed)
        w = torch.empty_like(i["w"])
        wavec.interleave_weights_wmma(w, i["w"], case["Cout"], case["B"] // 8)
        tiles = i["X"].shape[0]
        Y = torch.empty((tiles, case["Cout"], 64), dtype=torch.float16, device="cuda")
        return dict(case=case, X=i["X"], idx=i["idx"], w=w, bias=i["bias"], Y=Y)
    make = dict(sparse=_wave_plan, segments=_wave_plan, chain=_chain_plan, block=_block_plan,
                image=_image_plan, prefill=_decoder_plan, decode=_decoder_plan)[kind]
    return dict(case=case, **make(case, seed))


# ----------------------------------------------------------------------------------------- run
def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "token64":
        wavec.forward_token64_f16(state["Y"], state["X"], state["idx"], state["w"], state["bias"],
                                  c["batch"], c["Cin"], c["Cout"], c["B"] // 16, c["cluster"])
        return state["Y"]
    plan = state["plan"]
    if kind in ("block", "image"):
        return plan.infer_f32(state["x"])[0]
    if kind in ("prefill", "decode"):
        plan.set_ids(state["ids"])
    plan.execute(1)
    return state["out"].read()


# ---------------------------------------------------------------------------------------- work
def _conv_layers(c):
    """(cout, cin, k*k) of the image block's layers at its half resolution."""
    n = c["c"]
    return [(2 * n, n, 9), (2 * n, 2 * n, 1), (n, n, 9), (n, n, 9), (2 * n, 3 * n, 1),
            (2 * n, 4 * n, 1)]


def _distinct(draws, of):
    """Expected distinct values of `draws` uniform draws from `of`."""
    return of * -math.expm1(-draws / of)


def work(case):
    c, kind = case, case["kind"]
    if kind == "token64":
        tok, rows = (c["batch"] + 63) // 64 * 64, c["Cout"] // c["cluster"]
        read = _distinct(rows * c["B"], c["Cin"])
        return {"bytes": 2 * read * tok + 4 * rows * c["B"] + 2 * c["Cout"] * (c["B"] + 1 + tok),
                "flops": 2 * c["Cout"] * c["B"] * tok}
    if kind in ("sparse", "segments"):
        tok, rows = c["tokens"], c["cout"] // c["cluster"]
        fan = c["fan"] if kind == "sparse" else c["K"] * c["S"]
        starts = rows * fan if kind == "sparse" else rows * c["K"]
        read = _distinct(rows * fan, c["cin"])
        return {"bytes": 2 * read * tok + 4 * starts + 2 * c["cout"] * (fan + 1 + tok),
                "flops": 2 * c["cout"] * fan * tok}
    if kind == "chain":
        tok, fan, n = c["tokens"], c["K"] * c["S"], c["waves"]
        read = _distinct(n * c["cout"] * fan / 2, c["cin"])
        return {"bytes": 2 * read * tok + n * c["cout"] * (4 * c["K"] + 2 * fan + 2 + 2 * tok),
                "flops": 2 * n * c["cout"] * fan * tok}
    if kind == "block":
        macs = 3 * c["d"] * c["ffn"]
        return {"bytes": 2 * macs + 8 * c["d"] * c["tokens"], "flops": 2 * macs * c["tokens"]}
    if kind == "image":
        px = (c["H"] // 2) * (c["W"] // 2)
        macs = sum(o * i * k for o, i, k in _conv_layers(c))
        return {"bytes": 2 * macs + 4 * c["c"] * (c["H"] * c["W"] + 2 * px), "flops": 2 * macs * px}
    spec = synth.LLMSpec(layers=c["layers"], d=c["d"], ffn=c["ffn"], vocab=c["vocab"], S=c["S"])
    tok, nnz = c["requests"] * c["prompt"], spec.nnz_per_token
    return {"bytes": 2 * nnz + 2 * tok * (c["d"] + c["vocab"]), "flops": 2 * nnz * tok}


def tolerance(case):
    kind = case["kind"]
    if kind == "token64":  # one rounding toward zero to fp16
        return {"rel": 1.6e-3, "max": 0.01}
    if kind in ("sparse", "segments"):  # one rounding to fp16
        return {"rel": 8e-4, "max": 0.01}
    if kind == "chain":  # a rounding to fp16 after every wave
        return {"rel": 1.2e-3, "max": 0.02}
    if kind == "block":
        return {"rel": 1.8e-3, "max": 0.02}
    if kind == "image":
        return {"rel": 2.1e-3, "max": 0.03}
    return {"rel": 4e-3, "max": 0.05}  # a few layers, every tensor between them in fp16


# --------------------------------------------------------------------------------------- exact
_ACTS = {
    "none": lambda v: v, "relu": torch.relu, "sigmoid": torch.sigmoid,
    "silu": torch.nn.functional.silu, "gelu": torch.nn.functional.gelu,
    "leaky_relu": lambda v: torch.maximum(v, 0.1 * v),
}


def _wave64(x, pos, w, bias, act):
    """act(bias + w . x[pos]) for neurons in groups that share a row of pos, in 64 bits."""
    rows, fan = pos.shape
    cl, tok = w.shape[0] // rows, x.shape[1]
    out = torch.empty((w.shape[0], tok), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 26) // (fan * tok))
    for r in range(0, rows, step):
        q = pos[r:r + step]
        xs = x[q.reshape(-1)].double().view(q.shape[0], fan, tok)
        ws = w[r * cl:(r + q.shape[0]) * cl].double().view(q.shape[0], cl, fan)
        v = torch.stack([a @ b for a, b in zip(ws, xs)]) if cl > 1 else \
            (ws.transpose(1, 2) * xs).sum(1, keepdim=True)
        out[r * cl:(r + q.shape[0]) * cl] = v.view(-1, tok)
    return _ACTS[act](out + bias.double()[:, None])


def _exact_chain(c, seed):
    i = _chain_inputs(c, seed)
    src = i["x"].double()
    for v in i["waves"]:
        pos = (v["starts"][:, :, None] + torch.arange(c["S"], device="cuda")).flatten(1)
        y = _wave64(src, pos, v["w"], v["bias"], "relu")
        src = torch.cat([src, y])
    return y


def _rms64(x, eps=1e-5):
    return x * torch.rsqrt(x.square().mean(0, keepdim=True) + eps)


def _exact_block(c, seed):
    i = {k: v.double() for k, v in _block_inputs(c, seed).items()}
    n = _rms64(i["x"]) * i["gamma"][:, None]
    h = _ACTS["silu"](i["wg"] @ n) * (i["wu"] @ n)
    y = i["wd"] @ h + i["bd"][:, None] + i["x"]
    return y[:, None, :].cpu().numpy()


def _exact_image(c, seed):
    i = _image_inputs(c, seed)
    F = torch.nn.functional

    def conv(x, name, stride=1):
        w, b = (t.double() for t in i[name])
        co, ci, k, _ = w.shape
        cols = F.unfold(x[None], k, padding=k // 2, stride=stride)[0]
        h, wd = ((s + 2 * (k // 2) - k) // stride + 1 for s in x.shape[1:])
        return F.silu(w.view(co, -1) @ cols + b[:, None]).view(co, h, wd)

    n = c["c"]
    b = conv(conv(i["x"].double(), "down", 2), "cv1")
    t = conv(b[n:], "m1")
    b2 = conv(t, "m2") + b[n:]  # the residual is added to the activated sum
    e = conv(torch.cat([b, b2]), "cv2")
    pooled = F.max_pool2d(e[None], 5, 1, 2)[0]
    return conv(torch.cat([e, pooled]), "cv3").cpu().numpy()


def _exact_decoder(c, seed):
    spec, wts, ids = _decoder_inputs(c, seed)

    def proj(p, x, act="none"):
        starts = torch.from_numpy(p.starts.astype(np.int64)).cuda()
        cols = (starts[:, :, None] + torch.arange(spec.S, device="cuda")).flatten(1)
        w = torch.zeros((starts.shape[0], x.shape[0]), dtype=torch.float64, device="cuda")
        w.scatter_(1, cols, torch.from_numpy(p.weights).cuda().double())
        return _ACTS[act](w @ x + torch.from_numpy(p.bias).cuda().double()[:, None])

    x = torch.from_numpy(wts.embed).cuda().double()[torch.from_numpy(ids.astype(np.int64)).cuda()].T
    for mix, p in zip(wts.mix, wts.proj):
        u = _rms64(x).view(spec.d, spec.requests, spec.prompt)
        m = torch.from_numpy(mix).cuda().double()
        s = torch.zeros_like(u)
        for k in range(min(spec.rf, spec.prompt)):  # no token before a request's first
            s[:, :, k:] += m[:, k, None, None] * u[:, :, :spec.prompt - k]
        s = s.view(spec.d, -1)
        kv = proj(p["k"], s, "silu") * proj(p["v"], s)
        x = x + proj(p["o"], proj(p["q"], s, "sigmoid") * kv)
        n = _rms64(x)
        x = x + proj(p["dn"], proj(p["g"], n, "silu") * proj(p["u"], n))
    return proj(wts.head, _rms64(x)).cpu()


def exact(case, seed):
    kind = case["kind"]
    if kind == "token64":
        i = _token64_inputs(case, seed)
        return torch.stack([_wave64(x, i["idx"].long(), i["w"], i["bias"], "none")
                            for x in i["X"]])
    if kind in ("sparse", "segments"):
        i = _wave_inputs(case, seed)
        return _wave64(i["x"], i["pos"], i["w"], i["bias"], case["act"]).cpu()
    if kind == "chain":
        return _exact_chain(case, seed).cpu()
    return dict(block=_exact_block, image=_exact_image, prefill=_exact_decoder,
                decode=_exact_decoder)[kind](case, seed)
