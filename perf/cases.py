"""The calls that performance work on this library is measured by.

Each case is one call (or one captured decode step) of the quantised matrix
path as an inference engine makes it, at the shapes of bench.py and of the
tests: Qwen2.5-1.5B / 7B linears, int8 and int4, 1..32 activation rows for
decode, up to 1024 rows for prefill, the reference's ragged shapes, the
on-device quantiser and the embedding gather.  `draw` gives further cases of
the same ranges.

Decode steps are captured in a HIP graph and replayed, which is how a decode
engine issues them (bench.py, tests/test_gpu_capture.py); single calls are
made eagerly.

    listed()             the cases
    draw(rng)            one more case of their ranges
    prepare(case, seed)  weights, inputs and graph on the device
    run(state)           one pass; its outputs
    work(case)           bytes and operations that the call cannot do without
    tolerance(case)      how far another correct implementation may be off
    exact(case, seed)    the outputs in 64 bits, in plain torch
"""
import math

import torch

from infer_amd import chain, ops

GROUP = 128

# hidden, intermediate, query and key/value widths, heads, key/value heads,
# vocabulary (bench.py)
MODELS = {
    "1.5b": dict(H=1536, I=8960, q=1536, kv=256, heads=12, kv_heads=2, V=151936),
    "7b": dict(H=3584, I=18944, q=3584, kv=512, heads=28, kv_heads=4, V=152064),
}
EPS = 1e-6


def listed():
    return [
        # The smallest call: one linear of a 1.5B model for one token, eager.
        # Latency and launch cost count.
        dict(name="linear-int8-8960x1536-1row", op="linear", kind="int8", N=8960, K=1536, T=1, bias=False),
        # A decode step's linears for one user of a 1.5B model: many short
        # launches in a graph.
        dict(name="decode-1.5b-int4-1row", op="decode", model="1.5b", kind="int4", layers=14, rows=1),
        # The same on a 7B model, where streaming the weights counts
        # (bench.py's headline, some of its layers).
        dict(name="decode-7b-int4-1row", op="decode", model="7b", kind="int4", layers=8, rows=1),
        # A few users decoding together on int8 weights.
        dict(name="decode-7b-int8-5rows", op="decode", model="7b", kind="int8", layers=4, rows=5),
        # A full decode batch: the weight read should be shared by 16 rows.
        dict(name="decode-7b-int4-16rows", op="decode", model="7b", kind="int4", layers=8, rows=16),
        # Token to logits for one user: embedding, norms, SwiGLU and
        # residuals fused into the linears, and the int8 lm_head.
        dict(name="chain-7b-int4-1seq", op="chain", model="7b", kind="int4", layers=4, rows=1),
        # The same for a large batch on the smaller model.
        dict(name="chain-1.5b-int4-24seqs", op="chain", model="1.5b", kind="int4", layers=6, rows=24),
        # One chunk of a chunked prefill, of an odd length.
        dict(name="prefill-int8-18944x3584-201rows", op="linear", kind="int8", N=18944, K=3584, T=201, bias=False),
        # A long prompt, fp32 activations as the engine holds them, long rows.
        dict(name="prefill-int4-3584x18944-1024rows", op="linear", kind="int4", N=3584, K=18944, T=1024, bias=False),
        # A long prompt, bf16 activations, the widest layer matrix.
        dict(name="prefill-bf16-int8-18944x3584-1024rows", op="gemm_bf16", kind="int8", N=18944, K=3584, T=1024,
             bias=False),
        # Sizes that fill no tile and no 128-column group, with a bias.
        dict(name="ragged-int4-1535x2050-70rows", op="linear", kind="int4", N=1535, K=2050, T=70, bias=True),
        # Packing a layer matrix on the device (model conversion).
        dict(name="quantize-int4-18944x3584", op="quantize", kind="int4", N=18944, K=3584),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _shape(rng):
    """A layer matrix: of a model, or of generic size in whole groups."""
    if rng.random() < 0.5:
        m = MODELS[rng.choice(sorted(MODELS))]
        return rng.choice([(m["q"], m["H"]), (m["kv"], m["H"]), (m["I"], m["H"]), (m["H"], m["I"])])
    K = GROUP * _log_int(rng, 4, 148)
    return _log_int(rng, 256, max(256, min(18944, (18944 * 3584) // K))), K


def draw(rng):
    op = rng.choice(["linear", "linear", "prefill", "prefill", "gemm_bf16", "ragged", "decode", "decode", "chain",
                     "quantize", "embedding"])
    kind = rng.choice(["int8", "int4"])
    if op == "linear":
        N, K = _shape(rng)
        return dict(op="linear", kind=kind, N=N, K=K, T=rng.randint(1, 32), bias=rng.random() < 0.5)
    if op in ("prefill", "gemm_bf16"):
        N, K = _shape(rng)
        return dict(op="linear" if op == "prefill" else op, kind=kind, N=N, K=K, T=_log_int(rng, 33, 1024),
                    bias=rng.random() < 0.5)
    if op == "ragged":
        K = _log_int(rng, 130, 9000)
        K += K % 2  # int4 needs an even number of columns
        return dict(op="linear", kind=kind, N=_log_int(rng, 65, 9000), K=K, T=_log_int(rng, 1, 300),
                    bias=rng.random() < 0.5)
    if op == "decode":
        model = rng.choice(sorted(MODELS))
        return dict(op="decode", model=model, kind=kind, layers=14 if model == "1.5b" else 4, rows=rng.randint(1, 32))
    if op == "chain":
        model = rng.choice(sorted(MODELS))
        return dict(op="chain", model=model, kind=kind, layers=2 if kind == "int8" else 4, rows=rng.randint(1, 32))
    if op == "quantize":
        K = _log_int(rng, 256, 18944)
        K += K % 2
        return dict(op="quantize", kind=kind, N=_log_int(rng, 256, max(256, (18944 * 3584) // K)), K=K)
    m = MODELS[rng.choice(sorted(MODELS))]
    return dict(op="embedding", kind=kind, N=m["V"], K=m["H"], T=_log_int(rng, 16, 1024))


# ------------------------------------------------------------------ inputs
def _kind(case):
    return ops.QuantKind.kInt4 if case["kind"] == "int4" else ops.QuantKind.kInt8


def _gen(seed, i):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 1000003 + i)


def _weights(gen, N, K):
    """bf16 weights ~ N(0, 0.02)."""
    return (torch.randn(N, K, generator=gen, device="cuda") * 0.02).to(torch.bfloat16)


def _activations(gen, T, K):
    """fp32 ~ N(0, 1) with one channel in 512 thirty times larger, as the
    inputs of a language model's linears have them."""
    x = torch.randn(T, K, generator=gen, device="cuda")
    x[:, torch.randperm(K, generator=gen, device="cuda")[:max(1, K // 512)]] *= 30.0
    return x


def _bias(gen, N):
    return (torch.randn(N, generator=gen, device="cuda") * 0.5).to(torch.bfloat16)


def _pack(w, int4):
    """The packed layout (codes, bf16 scales, zero points) of bf16 weights,
    in plain torch: groups of 128 columns, int8 scale max|w| / 127, int4
    scale (max - min) / 15 with the range widened to hold 0."""
    N, K = w.shape
    G = (K + GROUP - 1) // GROUP
    wf = w.float()
    if K % GROUP:
        wf = torch.nn.functional.pad(wf, (0, G * GROUP - K))
    wf = wf.view(N, G, GROUP)
    if not int4:
        amax = wf.abs().amax(2)
        s = torch.where(amax > 0, amax / 127.0, torch.ones_like(amax)).to(torch.bfloat16)
        q = (wf.double() / s.double()[:, :, None]).round_().clamp_(-127, 127)
        q = q.to(torch.int8).view(N, G * GROUP)[:, :K].contiguous()
        return q.view(torch.uint8).view(-1), s.view(torch.int16).view(-1), None
    lo, hi = wf.amin(2).clamp(max=0.0), wf.amax(2).clamp(min=0.0)
    s = torch.where(hi > lo, (hi - lo) / 15.0, torch.ones_like(hi)).to(torch.bfloat16)
    z = (-lo.double() / s.double()).round_().clamp_(0, 15)
    q = ((wf.double() / s.double()[:, :, None]).round_() + z[:, :, None]).clamp_(0, 15)
    q = q.to(torch.uint8).view(N, G * GROUP)[:, :K].contiguous()
    q = q[:, 0::2] | (q[:, 1::2] << 4)
    return q.contiguous().view(-1), s.view(torch.int16).view(-1), z.to(torch.uint8).view(-1)


def _matrix(gen, kind, N, K):
    q, s, z = _pack(_weights(gen, N, K), kind == ops.QuantKind.kInt4)
    return ops.QuantView(kind, N, K, q, s, z)


def _dequant64(W, rows=slice(None)):
    """The matrix a QuantView holds, in float64 (its rows `rows`)."""
    N, K = W.rows, W.cols
    G = (K + GROUP - 1) // GROUP
    s = W.scales.view(torch.bfloat16).view(N, G)[rows].double().repeat_interleave(GROUP, 1)[:, :K]
    if W.zeros is None:
        return W.q.view(torch.int8).view(N, K)[rows].double().mul_(s)
    b = W.q.view(N, K // 2)[rows]
    q = torch.stack((b & 15, b >> 4), 2).view(b.shape[0], K).double()
    q.sub_(W.zeros.view(N, G)[rows].double().repeat_interleave(GROUP, 1)[:, :K])
    return q.mul_(s)


def _linear64(x64, W, bias=None):
    """x W^T (+ bias) in float64, 16384 output columns at a time."""
    y = torch.empty(x64.shape[0], W.rows, dtype=torch.float64, device="cuda")
    for n in range(0, W.rows, 16384):
        y[:, n:n + 16384] = x64 @ _dequant64(W, slice(n, n + 16384)).t().contiguous()
    return y if bias is None else y + bias.double()


def _rms64(x, w):
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * w.double()


# The linear call sites of a layer: matrices that share their input go in
# one call.
SITES = (("q", "k", "v"), ("o",), ("gate", "up"), ("down",))


def _sites(m):
    """(output widths, input width) of each call site."""
    return [([m["q"], m["kv"], m["kv"]], m["H"]), ([m["H"]], m["q"]), ([m["I"], m["I"]], m["H"]), ([m["H"]], m["I"])]


def _decode_inputs(case, seed):
    """(matrices, activations) of every call of a decode step."""
    m, kind = MODELS[case["model"]], _kind(case)
    calls = []
    for layer in range(case["layers"]):
        gen = _gen(seed, layer)
        for outs, K in _sites(m):
            calls.append(([_matrix(gen, kind, N, K) for N in outs], _activations(gen, case["rows"], K)))
    return calls


def _chain_model(case, seed):
    m, kind = MODELS[case["model"]], _kind(case)
    H, I, qo, kvo = m["H"], m["I"], m["q"], m["kv"]

    def norm(gen):
        return (1.0 + 0.1 * torch.randn(H, generator=gen, device="cuda")).to(torch.bfloat16)

    layers = []
    for layer in range(case["layers"]):
        gen = _gen(seed, layer)
        shapes = dict(q=(qo, H), k=(kvo, H), v=(kvo, H), o=(H, qo), gate=(I, H), up=(I, H), down=(H, I))
        L = {name: _matrix(gen, kind, N, K) for name, (N, K) in shapes.items()}
        L.update(input_ln=norm(gen), post_ln=norm(gen), q_b=_bias(gen, qo), k_b=_bias(gen, kvo), v_b=_bias(gen, kvo))
        layers.append(L)
    gen = _gen(seed, 1000)
    ids = torch.randint(0, m["V"], (case["rows"],), generator=gen, device="cuda")
    model = dict(cfg=dict(hidden=H, inter=I, heads=m["heads"], kv_heads=m["kv_heads"], head_dim=qo // m["heads"],
                          vocab=m["V"], layers=case["layers"], eps=EPS),
                 embed=_matrix(gen, ops.QuantKind.kInt8, m["V"], H), head=_matrix(gen, ops.QuantKind.kInt8, m["V"], H),
                 final_norm=norm(gen), layers=layers)
    return model, ids


def _linear_inputs(case, seed):
    gen = _gen(seed, 0)
    W = _matrix(gen, _kind(case), case["N"], case["K"])
    x = _activations(gen, case["T"], case["K"])
    if case["op"] == "gemm_bf16":
        x = x.to(torch.bfloat16)
    return W, x, _bias(gen, case["N"]) if case["bias"] else None


def _embedding_inputs(case, seed):
    gen = _gen(seed, 0)
    W = _matrix(gen, _kind(case), case["N"], case["K"])
    return W, torch.randint(0, case["N"], (case["T"],), generator=gen, device="cuda")


_capture_stream = None


def _capture(body):
    """A graph of body(), captured on the one stream whose workspace the
    library has reserved (a capturing stream cannot allocate one)."""
    global _capture_stream
    if _capture_stream is None:
        _capture_stream = torch.cuda.Stream()
        ops.init(torch.cuda.current_device(), _capture_stream)
    body()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=_capture_stream):
        body()
    return graph


def prepare(case, seed):
    op = case["op"]
    st = dict(case=case)
    if op in ("linear", "gemm_bf16"):
        W, x, bias = _linear_inputs(case, seed)
        y = torch.empty(case["T"], case["N"], dtype=torch.float32, device="cuda")
        st.update(W=W, x=x, bias=bias, y=y)
    elif op == "decode":
        calls = _decode_inputs(case, seed)
        sites = len(SITES)
        # every call's outputs of all layers: [layers][rows][out] per matrix
        ys = [[torch.empty(case["layers"], case["rows"], W.rows, dtype=torch.float32, device="cuda") for W in Ws]
              for Ws, _ in calls[:sites]]

        def body():
            for i, (Ws, x) in enumerate(calls):
                ops.gemv_multi(x, Ws, None, case["rows"], Ws[0].cols, [y[i // sites] for y in ys[i % sites]])

        st.update(calls=calls, ys={name: y for names, yc in zip(SITES, ys) for name, y in zip(names, yc)},
                  graph=_capture(body))
    elif op == "chain":
        model, ids = _chain_model(case, seed)
        step = chain.DecodeStep(model, rows=case["rows"])
        step.ids.copy_(ids)
        st.update(step=step, graph=_capture(step.step))
    elif op == "quantize":
        w = _weights(_gen(seed, 0), case["N"], case["K"])
        st.update(w=w, out=ops.alloc_quant(_kind(case), case["N"], case["K"]))
    else:
        W, ids = _embedding_inputs(case, seed)
        st.update(W=W, ids=ids, y=torch.empty(case["T"], case["K"], dtype=torch.float32, device="cuda"))
    return st


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "linear":
        ops.launch_linear_q(state["x"], state["W"], state["bias"], case["T"], case["K"], case["N"], state["y"])
        return state["y"]
    if op == "gemm_bf16":
        ops.launch_gemm_bf16x(state["x"], state["W"], state["bias"], case["T"], case["K"], case["N"], state["y"])
        return state["y"]
    if op == "decode":
        state["graph"].replay()
        return state["ys"]
    if op == "chain":
        state["graph"].replay()
        step, B = state["step"], case["rows"]
        return {"hidden": step.h_last.view(B, -1), "logits": step.logits.view(B, -1)}
    if op == "quantize":
        out = ops.quantize(state["w"], _kind(case), out=state["out"])
        return {"codes": out.q, "scales": out.scales} if out.zeros is None else \
            {"codes": out.q, "scales": out.scales, "zeros": out.zeros}
    ops.launch_embedding_q(state["W"], state["ids"], case["T"], case["K"], state["y"])
    return state["y"]


# ------------------------------------------------------------------ what is expected
def _packed_bytes(kind, N, K):
    G = (K + GROUP - 1) // GROUP
    return N * K // 2 + 3 * N * G if kind == "int4" else N * K + 2 * N * G


def work(case):
    op, kind = case["op"], case.get("kind")
    if op in ("linear", "gemm_bf16"):
        N, K, T = case["N"], case["K"], case["T"]
        b = _packed_bytes(kind, N, K) + (2 if op == "gemm_bf16" else 4) * T * K + 4 * T * N + (2 * N if case["bias"] else 0)
        return {"bytes": b, "flops": 2 * T * N * K}
    if op == "quantize":
        N, K = case["N"], case["K"]
        return {"bytes": 2 * N * K + _packed_bytes(kind, N, K), "flops": 2 * N * K}
    if op == "embedding":
        return {"bytes": case["T"] * (_packed_bytes(kind, 1, case["K"]) + 8 + 4 * case["K"]), "flops": case["T"] * case["K"]}
    m, B = MODELS[case["model"]], case["rows"]
    b = f = 0
    for outs, K in _sites(m):
        for N in outs:
            b += _packed_bytes(kind, N, K)
            f += 2 * B * N * K
        if op == "decode":
            b += 4 * B * (K + sum(outs))
    if op == "decode":
        return {"bytes": b * case["layers"], "flops": f * case["layers"]}
    # the chain reads its norms and biases, keeps its hidden states on the
    # way, and returns the last one and the logits
    H, V = m["H"], m["V"]
    b = case["layers"] * (b + 2 * (2 * H + m["q"] + 2 * m["kv"])) + _packed_bytes("int8", V, H) + 2 * H
    b += B * (8 + _packed_bytes("int8", 1, H)) + 4 * B * (H + V)
    return {"bytes": b, "flops": f * case["layers"] + 2 * B * H * V}


def tolerance(case):
    if case["op"] in ("quantize", "embedding"):
        return "exact"
    # fp32 sums of products of the given activations (to 22 bits and more)
    # and exact weights: 6e-8 to 2.6e-7 against 64 bits over these ranges,
    # a few times that through the layers of a chain
    return {"rel": 2e-6 if case["op"] == "chain" else 1e-6}


def exact(case, seed):
    op = case["op"]
    if op in ("linear", "gemm_bf16"):
        W, x, bias = _linear_inputs(case, seed)
        return _linear64(x.double(), W, bias)
    if op == "decode":
        calls, sites = _decode_inputs(case, seed), len(SITES)
        return {name: torch.stack([_linear64(x.double(), Ws[j]) for Ws, x in calls[i::sites]])
                for i, names in enumerate(SITES) for j, name in enumerate(names)}
    if op == "chain":
        model, ids = _chain_model(case, seed)
        m = MODELS[case["model"]]
        heads, kv, hd = m["heads"], m["kv_heads"], m["q"] // m["heads"]
        emb = model["embed"]
        G = emb.groups
        h = emb.q.view(torch.int8).view(emb.rows, emb.cols)[ids].double() * \
            emb.scales.view(torch.bfloat16).view(emb.rows, G)[ids].double().repeat_interleave(GROUP, 1)
        for L in model["layers"]:
            # one token: every query head's attention output is the value
            # row of its key/value head
            v = _linear64(_rms64(h, L["input_ln"]), L["v"], L["v_b"])
            a = v.view(-1, kv, 1, hd).expand(-1, kv, heads // kv, hd).reshape(-1, heads * hd)
            h = h + _linear64(a, L["o"])
            n = _rms64(h, L["post_ln"])
            g = _linear64(n, L["gate"])
            h = h + _linear64(g * torch.sigmoid(g) * _linear64(n, L["up"]), L["down"])
        return {"hidden": h, "logits": _linear64(_rms64(h, model["final_norm"]), model["head"])}
    if op == "quantize":
        q, s, z = _pack(_weights(_gen(seed, 0), case["N"], case["K"]), case["kind"] == "int4")
        return {"codes": q, "scales": s} if z is None else {"codes": q, "scales": s, "zeros": z}
    W, ids = _embedding_inputs(case, seed)
    sub = ops.QuantView(W.kind, case["T"], W.cols, W.q.view(W.rows, -1)[ids].contiguous().view(-1),
                        W.scales.view(W.rows, -1)[ids].contiguous().view(-1),
                        None if W.zeros is None else W.zeros.view(W.rows, -1)[ids].contiguous().view(-1))
    return _dequant64(sub)
