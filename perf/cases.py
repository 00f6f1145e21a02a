"""The work this library is timed on: what a training program has it do, through the C-ABI as ``ane_amd.bridge`` binds it.

A pass is a piece of one training step of the two models that the repository knows (Stories110M and Qwen3-0.6B shapes):
the elementwise and normalisation ops of a layer in both directions, the loss, the classifier with its three products,
the embedding and its gradient, the optimizer, the hand-over of activations in fp16 and INT8, and the drop-in calls on
host arrays.  A program knows its buffers before it steps, so ``prepare`` makes the buffers and the argument lists of
the calls once and ``run`` issues the calls.

Sizes: 256 positions per sequence is the training loops' own length; other lengths (odd ones among them) are a user's
own data.  Batches go from one sequence (the training loops' call pattern) to 32.
"""
import numpy as np
import torch

from ane_amd import bridge as br

# channels, hidden size, query heads, KV heads, head size, RoPE theta, per-head norm of Q and K, layers, vocabulary
MODELS = {
    "stories110m": dict(C=768, H=2048, heads=12, kv=12, hd=64, theta=1e4, qk_norm=False, layers=12, V=32000),
    "qwen3-0.6b": dict(C=1024, H=3072, heads=16, kv=8, hd=128, theta=1e6, qk_norm=True, layers=28, V=151936),
}
EPS = 1e-5


def listed():
    return [
        # One layer on one sequence, as the training loops call their ops: launches of 1-2 MB tensors.
        dict(name="layer_one_sequence", kind="layer", model="stories110m", batch=1, S=256, storage="f32", fused=False),
        # The layer of a batched fp32 training step, one call per op.
        dict(name="layer_batch_f32", kind="layer", model="qwen3-0.6b", batch=16, S=256, storage="f32", fused=False),
        # The same layer with activations stored as bfloat16, the residual adds riding with the norms.
        dict(name="layer_batch_bf16", kind="layer", model="qwen3-0.6b", batch=16, S=256, storage="bf16", fused=True),
        # A batch of sequences cut at a length of the user's own: rows that start at any 4-byte boundary.
        dict(name="layer_odd_length", kind="layer", model="stories110m", batch=8, S=197, storage="f32", fused=True),
        # The loss over the whole vocabulary of the larger model.
        dict(name="loss_full_vocabulary", kind="loss", V=151936, S=256, storage="f32"),
        # The loss on bfloat16 logits of a shorter sequence, smaller vocabulary.
        dict(name="loss_short_bf16", kind="loss", V=32000, S=200, storage="bf16"),
        # The classifier of a training step: logits, loss, the gradients of the activations and of the compacted
        # table.  A compacted vocabulary has as many rows as the text happens to use.
        dict(name="classifier_compact", kind="classifier", V=24573, D=1024, S=256),
        # The embedding and its ordered gradient for a batch of text.
        dict(name="embedding_batch", kind="embedding", V=32000, D=768, batch=64, S=256),
        # The same for longer sequences into the larger table.
        dict(name="embedding_long", kind="embedding", V=151936, D=1024, batch=40, S=1000),
        # Norm, clip and AdamW over every tensor of a 110 M parameter model: the end of each training step.
        dict(name="optimizer_step", kind="optimizer", model="stories110m", layers=12, embedding=True),
        # Activations handed over in fp16 and INT8, and the attention gradients taken back from fp16.
        dict(name="handover_fp16_int8", kind="handover", model="qwen3-0.6b", batch=16, S=256),
        # The drop-in calls: a training loop whose arrays stay in ordinary host memory.
        dict(name="host_arrays", kind="host", model="stories110m", S=256, V=9216),
    ]


def _spread(rng, lo, hi):
    """An integer of [lo, hi], spread over its logarithm."""
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["layer"] * 5 + ["loss"] * 2 + ["classifier"] * 2 + ["embedding"] * 2 + ["optimizer", "handover", "host"])
    model = rng.choice(sorted(MODELS))
    S = rng.choice([256, _spread(rng, 32, 1024)])
    batch = _spread(rng, 1, max(1, 8192 // S))
    if kind == "layer":
        return dict(kind=kind, model=model, batch=batch, S=S, storage=rng.choice(["f32", "bf16"]), fused=rng.random() < 0.5)
    if kind == "loss":
        return dict(kind=kind, V=_spread(rng, 2000, min(151936, 151936 * 256 // S)), S=S, storage=rng.choice(["f32", "bf16"]))
    if kind == "classifier":
        S = min(S, 512)
        return dict(kind=kind, V=_spread(rng, 2000, 24573 * 256 // max(S, 256)), D=MODELS[model]["C"], S=S)
    if kind == "embedding":
        return dict(kind=kind, V=_spread(rng, 2000, 151936), D=MODELS[model]["C"], batch=_spread(rng, 1, 40960 // S), S=S)
    if kind == "optimizer":
        return dict(kind=kind, model="stories110m", layers=rng.randint(1, 12), embedding=rng.random() < 0.5)
    if kind == "handover":
        return dict(kind=kind, model=model, batch=batch, S=S)
    return dict(kind=kind, model=model, S=min(S, 512), V=_spread(rng, 2000, 20000))


# ---- inputs ---------------------------------------------------------------------------------------------------------

class _Made:
    """Tensors on the GPU, made from one seed."""

    def __init__(self, seed):
        br.init()
        br.check(br.lib.mi355_set_stream(torch.cuda.current_stream().cuda_stream or None))
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        self.np = np.random.default_rng(seed)
        self.keep, self.calls = [], []

    def normal(self, *shape, dtype=torch.float32, std=1.0, mean=0.0):
        t = torch.empty(shape, device="cuda").normal_(mean, std, generator=self.gen).to(dtype)
        self.keep.append(t)
        return t

    def zeros(self, *shape, dtype=torch.float32):
        t = torch.zeros(shape, dtype=dtype, device="cuda")
        self.keep.append(t)
        return t

    def zipf(self, n, V):
        """Token ids as text has them: rank r with probability ~ 1/r^1.1."""
        w = np.arange(1, V + 1, dtype=np.float64) ** -1.1
        cdf = np.cumsum(w / w.sum())
        ids = np.minimum(np.searchsorted(cdf, self.np.random(n), side="right"), V - 1).astype(np.int32)
        t = torch.from_numpy(ids).cuda()
        self.keep.append(t)
        return t

    def call(self, name, *args):
        """One call of the C-ABI; tensors are passed by their device addresses, arrays by their host addresses."""
        self.calls.append((getattr(br.lib, name), tuple(a.data_ptr() if torch.is_tensor(a) else a.ctypes.data if isinstance(a, np.ndarray) else a for a in args)))


def _layer(case, m):
    mod = MODELS[case["model"]]
    C, H, heads, kv, hd = mod["C"], mod["H"], mod["heads"], mod["kv"], mod["hd"]
    B, S, n = case["batch"], case["S"], case["batch"] * case["S"]
    bf16 = case["storage"] == "bf16"
    dtype, end = (torch.bfloat16, "_bf16_dev") if bf16 else (torch.float32, "_dev")
    x, o, f, dy, dx_ffn, dx_attn = (m.normal(B, C, S, dtype=dtype) for _ in range(6))
    q, gq = (m.normal(B, heads * hd, S, dtype=dtype) for _ in range(2))
    k, gk = (m.normal(B, kv * hd, S, dtype=dtype) for _ in range(2))
    h1, h3, dsilu = (m.normal(B, H, S, dtype=dtype) for _ in range(3))
    w_att, w_ffn = (m.normal(C, std=0.02, mean=1.0) for _ in range(2))
    wq, wk = (m.normal(hd, std=0.02, mean=1.0) for _ in range(2))
    dw_att, dw_ffn, dwq, dwk = m.zeros(C), m.zeros(C), m.zeros(hd), m.zeros(hd)
    out = {}

    def new(name, like):
        out[name] = m.zeros(*like.shape, dtype=like.dtype)
        return out[name]

    cos, sin = br.rope_tables_dev(S, hd, mod["theta"])
    alpha = float(np.float32(1.0 / np.sqrt(2.0 * mod["layers"])))
    # the training loops read weight gradients at the optimizer step, so their sums are run together at the end
    br.check(br.lib.mi355_dw_defer(1))
    # forward
    x2, x2n, x_next, xn = new("x2", x), new("x2n", x), new("x_next", x), new("xn", x)
    q_rot, k_rot, gate = new("q_rot", q), new("k_rot", k), new("gate", h1)
    if not case["fused"]:
        m.call("mi355_rmsnorm_fwd" + end, xn, x, w_att, C, S, B, EPS)
    if mod["qk_norm"]:
        m.call("mi355_qknorm_rope_fwd" + end, q_rot, k_rot, q, k, wq, wk, heads, kv, hd, S, B, cos, sin, EPS)
    else:
        m.call("mi355_rope" + end, q_rot, k_rot, q, k, heads, kv, hd, S, B, cos, sin, 1)
    if case["fused"]:
        m.call("mi355_residual_rmsnorm_fwd" + end, x2, x2n, x, o, alpha, w_ffn, C, S, B, EPS)
    else:
        m.call("mi355_axpby" + end, x2, x, o, alpha, n * C, 0)
        m.call("mi355_rmsnorm_fwd" + end, x2n, x2, w_ffn, C, S, B, EPS)
    m.call("mi355_swiglu_fwd" + end, gate, h1, h3, n * H)
    if case["fused"]:       # the norm of the next layer rides with the residual that feeds it
        m.call("mi355_residual_rmsnorm_fwd" + end, x_next, xn, x2, f, alpha, w_att, C, S, B, EPS)
    else:
        m.call("mi355_axpby" + end, x_next, x2, f, alpha, n * C, 0)
    # backward
    dffn, dx2, dx2s, dx1 = new("dffn", x), new("dx2", x), new("dx2s", x), new("dx1", x)
    dh1, dh3, dq, dk = new("dh1", h1), new("dh3", h1), new("dq", q), new("dk", k)
    m.call("mi355_axpby" + end, dffn, dy, None, alpha, n * C, 1)
    m.call("mi355_swiglu_bwd" + end, dh1, dh3, dsilu, h1, h3, n * H)
    if case["fused"]:
        m.call("mi355_rmsnorm_bwd_residual" + end, dx2, dx2s, dw_ffn, dx_ffn, x2, w_ffn, dy, alpha, C, S, B, EPS, 0)
    else:
        m.call("mi355_rmsnorm_bwd" + end, dx2, dw_ffn, dx_ffn, x2, w_ffn, C, S, B, EPS, 0)
        m.call("mi355_axpby" + end, dx2, dx2, dy, 0.0, n * C, 2)
        m.call("mi355_axpby" + end, dx2s, dx2, None, alpha, n * C, 1)
    if mod["qk_norm"]:
        m.call("mi355_qknorm_rope_bwd" + end, dq, dk, dwq, dwk, gq, gk, q, k, wq, wk, heads, kv, hd, S, B, cos, sin, EPS, 0)
        out.update(dwq=dwq, dwk=dwk)
    else:
        m.call("mi355_rope" + end, dq, dk, gq, gk, heads, kv, hd, S, B, cos, sin, -1)
    if case["fused"]:
        m.call("mi355_rmsnorm_bwd_residual" + end, dx1, None, dw_att, dx_attn, x, w_att, dx2, alpha, C, S, B, EPS, 0)
    else:
        m.call("mi355_rmsnorm_bwd" + end, dx1, dw_att, dx_attn, x, w_att, C, S, B, EPS, 0)
        m.call("mi355_axpby" + end, dx1, dx1, dx2, 0.0, n * C, 2)
    m.call("mi355_dw_flush")
    out.update(dw_att=dw_att, dw_ffn=dw_ffn)
    return out


def _loss(case, m):
    V, S = case["V"], case["S"]
    dtype, end = (torch.bfloat16, "_bf16_dev") if case["storage"] == "bf16" else (torch.float32, "_dev")
    logits, targets = m.normal(V, S, dtype=dtype, std=2.0), m.zipf(S, V)
    out = dict(dlogits=m.zeros(V, S, dtype=dtype), loss=m.zeros(1))
    m.call("mi355_softmax_ce" + end, out["dlogits"], out["loss"], logits, targets, V, S, 1.0)
    return out


def _classifier(case, m):
    V, D, S = case["V"], case["D"], case["S"]
    table, x, targets = m.normal(V, D, std=0.02), m.normal(D, S), m.zipf(S, V)
    out = dict(logits=m.zeros(V, S), dlogits=m.zeros(V, S), loss=m.zeros(1), dx=m.zeros(D, S), dtable=m.zeros(V, D))
    m.call("mi355_sgemm_dev", 0, 0, V, S, D, 1.0, table, D, x, S, 0.0, out["logits"], S)
    m.call("mi355_softmax_ce_dev", out["dlogits"], out["loss"], out["logits"], targets, V, S, 256.0)
    m.call("mi355_sgemm_dev", 1, 0, D, S, V, 1.0, table, D, out["dlogits"], S, 0.0, out["dx"], S)
    m.call("mi355_sgemm_dev", 0, 1, V, D, S, 1.0, out["dlogits"], S, x, S, 1.0, out["dtable"], D)
    return out


def _embedding(case, m):
    V, D, B, S = case["V"], case["D"], case["batch"], case["S"]
    table, ids, dx = m.normal(V, D, std=0.02), m.zipf(B * S, V), m.normal(B, D, S)
    out = dict(x=m.zeros(B, D, S), dtable=m.zeros(V, D))
    m.call("mi355_embed_gather_dev", out["x"], table, ids, V, D, S, B)
    m.call("mi355_embed_scatter_add_dev", out["dtable"], dx, ids, V, D, S, B)
    return out


def _tensor_sizes(case):
    mod = MODELS[case["model"]]
    C, H, q, kv = mod["C"], mod["H"], mod["heads"] * mod["hd"], mod["kv"] * mod["hd"]
    sizes = [C * q, C * kv, C * kv, q * C, H * C, C * H, H * C, C, C] * case["layers"] + [C]
    return sizes + ([mod["V"] * C] if case["embedding"] else [])


def _optimizer(case, m):
    import ctypes
    sizes = _tensor_sizes(case)
    at = np.concatenate([[0], np.cumsum(sizes)])
    n, count = int(at[-1]), len(sizes)
    w, g, mom = m.normal(n, std=0.02), m.normal(n), m.normal(n, std=0.01)
    v = m.normal(n, std=0.01).square_()
    scale, sumsq = m.zeros(1), br.DevArray(1)
    arrays = [(ctypes.c_void_p * count)(*[t.data_ptr() + 4 * int(a) for a in at[:-1]]) for t in (w, g, mom, v)]
    ns = (ctypes.c_size_t * count)(*sizes)
    decay = (ctypes.c_float * count)(*[0.1 if s > 4096 else 0.0 for s in sizes])      # no decay on the norm weights
    m.keep += arrays + [ns, decay, sumsq]
    loss_scale = 1.0 / 256.0
    m.call("mi355_buf_zero", sumsq.handle)
    m.call("mi355_sumsq_accum_multi_dev", sumsq.ptr, arrays[1], ns, count, loss_scale)
    m.call("mi355_clip_scale_dev", scale, sumsq.ptr, 1.0)
    m.call("mi355_adam_update_multi_dev", *arrays, ns, decay, count, 100, 3e-4, 0.9, 0.95, 1e-8, loss_scale, scale, 1)
    return dict(w=w, m=mom, v=v, g=g, scale=scale)


def _handover(case, m):
    mod = MODELS[case["model"]]
    C, H, heads, kv, hd = mod["C"], mod["H"], mod["heads"], mod["kv"], mod["hd"]
    B, S, n = case["batch"], case["S"], case["batch"] * case["S"] * mod["C"]
    x, h16 = m.normal(B, C, S), m.normal(B, H, S, dtype=torch.float16)
    dq16, dk16, dv16 = (m.normal(B, heads * hd, S, dtype=torch.float16) for _ in range(3))
    out = dict(surface=m.zeros(B, C, S + C, dtype=torch.float16), h=m.zeros(B, H, S), dq=m.zeros(B, heads * hd, S),
               dk=m.zeros(B, kv * hd, S), dv=m.zeros(B, kv * hd, S), q=m.zeros(n, dtype=torch.int8), scale=m.zeros(1),
               x_back=m.zeros(B, C, S))
    cos, sin = br.rope_tables_dev(S, hd, mod["theta"])
    # activations go into a surface whose rows hold the weights behind them, results come back packed
    m.call("mi355_cvt_f32_f16_dev", out["surface"], S + C, x, S, B * C, S)
    m.call("mi355_cvt_f16_f32_dev", out["h"], S, h16, S, B * H, S)
    m.call("mi355_attn_grads_finish_dev", out["dq"], out["dk"], out["dv"], dq16, dk16, dv16, 1, 0, 0, 0, heads, kv, hd, S, B,
           cos, sin)
    m.call("mi355_int8_quantize_dynamic_dev", out["q"], out["scale"], x, n, 0)
    m.call("mi355_int8_dequant_dev", out["x_back"], out["q"], out["scale"], n)
    return out


def _host(case, m):
    mod = MODELS[case["model"]]
    C, H, S, V, hd = mod["C"], mod["H"], case["S"], case["V"], mod["hd"]

    def normal(*shape, std=1.0):
        a = m.np.standard_normal(shape, dtype=np.float32)
        m.keep.append(a)
        return np.multiply(a, np.float32(std), out=a)

    def new(*shape):
        m.keep.append(np.zeros(shape, np.float32))
        return m.keep[-1]

    x, dy, w = normal(C, S), normal(C, S), normal(C, std=0.02) + np.float32(1)
    h1, h3, dsilu = normal(H, S), normal(H, S), normal(H, S)
    weight, grad, mom, var = normal(H, C, std=0.02), normal(H, C), normal(H, C, std=0.01), normal(H, C, std=0.01) ** 2
    logits, tokens = normal(V, S, std=2.0), m.zipf(S, V).cpu().numpy().astype(np.uint16)
    dq = normal(mod["heads"] * hd, S)
    out = dict(xn=new(C, S), x2=new(C, S), gate=new(H, S), dlogits=new(V, S), dh1=new(H, S), dh3=new(H, S), dx=new(C, S),
               dw=new(C), dq=dq, dtable=new(V, C), weight=weight, mom=mom, var=var)
    m.keep += [w, var, tokens]
    m.call("mi355_rmsnorm", out["xn"], x, w, C, S)
    m.call("mi355_axpby", out["x2"], x, dy, 0.2, C * S, 0)
    m.call("mi355_swiglu_fwd", out["gate"], h1, h3, H * S)
    m.call("mi355_cross_entropy_loss", out["dlogits"], logits, tokens, V, S)
    m.call("mi355_swiglu_bwd", out["dh1"], out["dh3"], dsilu, h1, h3, H * S)
    m.call("mi355_rmsnorm_bwd", out["dx"], out["dw"], dy, x, w, C, S)
    m.call("mi355_rope_backward_inplace", dq, S, mod["heads"] * hd, hd)
    m.call("mi355_embed_backward", out["dtable"], x, tokens, V, C, S)
    m.call("mi355_adam_update", weight, grad, mom, var, H * C, 100, 3e-4, 0.9, 0.95, 1e-8, 0.1)
    return out


_MAKERS = dict(layer=_layer, loss=_loss, classifier=_classifier, embedding=_embedding, optimizer=_optimizer,
               handover=_handover, host=_host)


# ---- what a program does ----------------------------------------------------------------------------------------------

def prepare(case, seed):
    m = _Made(seed)
    br.check(br.lib.mi355_dw_defer(0))
    out = _MAKERS[case["kind"]](case, m)
    return dict(calls=m.calls, out=out, keep=m.keep)


def run(state):
    for fn, args in state["calls"]:
        got = fn(*args)
        if got == -1:
            raise br.BridgeError("%s failed: %s" % (fn.__name__, br.last_error()))
        if type(got) is float:          # the loss, which the drop-in call returns
            state["out"]["loss"] = got
    return state["out"]


# ---- what a pass cannot do without ------------------------------------------------------------------------------------

def work(case):
    """Each input read once, each output written once (accumulated and updated tensors: both); intermediate results that
    a pass returns count as outputs only."""
    kind = case["kind"]
    if kind == "loss":
        return dict(bytes=2 * (4 if case["storage"] == "f32" else 2) * case["V"] * case["S"], flops=0)
    if kind == "classifier":
        V, D, S = case["V"], case["D"], case["S"]
        # the table and its gradient (read and written), x and its gradient, logits and their gradient out
        return dict(bytes=4 * (3 * V * D + 2 * D * S + 2 * V * S), flops=6 * V * D * S)
    if kind == "embedding":
        V, D, N = case["V"], case["D"], case["batch"] * case["S"]
        # distinct tokens expected of N draws: their rows are read once for the gather; read and written for the gradient
        p = np.arange(1, V + 1, dtype=np.float64) ** -1.1
        rows = float(np.sum(-np.expm1(N * np.log1p(-np.minimum(p / p.sum(), 1 - 1e-12)))))
        return dict(bytes=8 * D * N + 12 * D * rows + 4 * N, flops=0)
    if kind == "optimizer":
        n = sum(_tensor_sizes(case))
        return dict(bytes=32 * n, flops=0)              # read w, g, m, v; write w, m, v and the cleared g
    mod = MODELS[case["model"]]
    C, H, q, kv, S = mod["C"], mod["H"], mod["heads"] * mod["hd"], mod["kv"] * mod["hd"], case["S"]
    if kind == "host":
        return dict(bytes=4 * S * (7 * C + 8 * H + 2 * q + 2 * case["V"]) + 28 * H * C + 8 * C * S, flops=0)
    n = case["batch"] * S
    if kind == "handover":
        return dict(bytes=n * (4 * C + 2 * C + 6 * H + 6 * q + 4 * q + 8 * kv + C + 4 * C), flops=0)
    # inputs 6 C, 2 q, 2 kv, 3 H; outputs 8 C, 2 q, 2 kv, 3 H
    return dict(bytes=(4 if case["storage"] == "f32" else 2) * n * (14 * C + 4 * (q + kv) + 6 * H), flops=0)


def tolerance(case):
    """About four times what the path differs by from the same operations in 64 bits (2-norm and largest, measured):
    fp32 layers and losses 1.5e-7 and 6e-7, the classifier's products 6e-7 and 2.7e-5, bf16 results (one rounding to
    8 bits on store) 1.7e-3 and 3.9e-3."""
    kind = case["kind"]
    if kind in ("embedding", "handover"):
        return "exact"              # copies, conversions and sums in a stated order
    if case.get("storage") == "bf16":
        return {"rel": 7e-3, "max": 1.6e-2}
    if kind == "classifier":
        return {"rel": 2.5e-6, "max": 1e-4}
    return {"rel": 1e-6, "max": 1e-5}
