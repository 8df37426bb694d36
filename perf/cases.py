"""Work that users of this package have it do, as cases with inputs, a run and a check.

A case is a dict of plain values; `prepare` makes its inputs on the GPU from a seed, `run`
makes one pass over them through the package's public entry points, `work` states the bytes
and operations that the pass cannot do without, `exact` computes the same outputs in 64 bits
with plain torch, and `tolerance` bounds how far a correct implementation may lie from
another.  `listed` holds the named cases and `draw` gives further ones of the same ranges.

Kinds of work (field "kind"):

  wkv          the WKV-7 recurrence by itself: the decode step of a batch on a slot pool,
               the prefill of one prompt or of several at once, with the state in fp32 (slot
               pool) or in fp16 (dense).
  time_mix     one layer's time mix on the torch ops, as an executor written against them
               composes it: residual add + LayerNorm + six token-shift lerps, r/k/v
               projections, the low-rank adapters, the kk/a gate, WKV-7 on the slot pool,
               GroupNorm + bonus + gate, the output projection.  A decode step (T = 1) is
               captured into a HIP graph once, as serving loops do, and replayed; a prompt,
               whose length changes from call to call, runs eagerly.
  channel_mix  one layer's channel mix on the torch ops: residual add + LayerNorm, then the
               token shift, the squared-ReLU FFN and its down projection in one op.
  head         the last LayerNorm and the vocabulary projection.
  sample       a token per row from fp32 logits, with temperature / top-k / top-p, with and
               without repetition penalties.
  decode       a whole batched decode step of the model through `DecodeEngine`, captured
               into a HIP graph and replayed.
  mixed        a whole continuous-batching step through `MixedEngine`: decode rows and
               prompt chunks together, eagerly (the batch's shape changes every step).

Sizes: heads of 64; widths 768 to 4096 with the adapter ranks of the presets where there is
one; batches of 1 to 256 sequences; prompts of 2 to 4096 tokens.
"""
import math

import torch
import torch.nn.functional as F

from vkwr._ops import sampling_ops as SMP
from vkwr._ops.v1 import v1_linear_ops as LIN
from vkwr._ops.v1 import v1_mix_ops as MIX
from vkwr._ops.v1 import v1_norm_ops as NORM
from vkwr._ops.v1 import v1_rank_ops as RANK
from vkwr._ops.v1 import v1_wkv_ops as WKV
from vkwr.model_executor import DecodeEngine, MixedEngine, RWKV7Config, RWKV7Model, RWKV7State
from vkwr_amd import capi

HEAD = 64
# Low-rank widths (w, a, v, g) per model width: the presets' at 2048 and 4096, in between generic.
RANKS = {768: (64, 64, 32, 128), 2048: (96, 96, 64, 256), 2560: (96, 96, 64, 320), 4096: (128, 128, 96, 480)}
TMIX = ("x_r", "x_w", "x_k", "x_v", "x_a", "x_g")


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # The decode step of a serving batch: 128 sequences, a pool of four times as many slots.
        {"name": "wkv decode 128 seqs", "kind": "wkv", "B": 128, "T": 1, "H": 32, "state": "fp32"},
        # One user's prompt, as a chat turn sends it: a single sequence, a length that is no
        # multiple of anything.
        {"name": "wkv prompt of 1500", "kind": "wkv", "B": 1, "T": 1500, "H": 32, "state": "fp32"},
        # Several prompts at once: batch scoring, or a prefill server.
        {"name": "wkv 8 prompts of 1024", "kind": "wkv", "B": 8, "T": 1024, "H": 32, "state": "fp32"},
        # The half-size state that memory-bound deployments keep.
        {"name": "wkv fp16 2 prompts of 300", "kind": "wkv", "B": 2, "T": 300, "H": 32, "state": "fp16"},
        # A single user generating: one row through a layer, launch latency and weights.
        {"name": "time mix decode 1 row", "kind": "time_mix", "B": 1, "T": 1, "C": 2048, "weights": "nk"},
        # Three prompts through a layer whose weights are stored [K, N], as linear_f16 takes them.
        {"name": "time mix 3 prompts of 333", "kind": "time_mix", "B": 3, "T": 333, "C": 2048, "weights": "kn"},
        # A moderate decode batch through the wide model's FFN.
        {"name": "channel mix 24 rows", "kind": "channel_mix", "B": 24, "T": 1, "C": 4096},
        # A prompt through the FFN.
        {"name": "channel mix prompt of 700", "kind": "channel_mix", "B": 1, "T": 700, "C": 2048},
        # Logits of a decode batch.
        {"name": "head 96 rows", "kind": "head", "B": 96, "C": 2048, "weights": "nk"},
        # Tokens of a decode batch with the usual truncation and penalties.
        {"name": "sample 32 rows", "kind": "sample", "B": 32, "V": 65536, "top_k": 40, "top_p": 0.9,
         "penalties": True},
        # The whole decode step of the 1.5b preset at the batch it is served with.
        {"name": "decode step 1.5b 128 rows", "kind": "decode", "B": 128, "shape": "1.5b", "layers": 24},
        # A continuous-batching step at the 7b layer shape: decode rows beside two prompt chunks.
        {"name": "mixed step 7b 4 layers", "kind": "mixed", "B": 48, "chunks": 2, "T": 500, "shape": "7b",
         "layers": 4},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["wkv", "wkv", "wkv", "time_mix", "time_mix", "channel_mix", "channel_mix", "head", "sample",
                       "decode", "mixed"])
    if kind == "wkv":
        H, state = rng.choice([12, 32, 40, 64]), rng.choice(["fp32", "fp32", "fp16"])
        if rng.random() < 0.35:
            return {"kind": kind, "B": _log_int(rng, 1, 256), "T": 1, "H": H, "state": state}
        B = _log_int(rng, 1, 12)
        T = _log_int(rng, 3, 4096 if state == "fp32" else 1500)
        T = max(3, min(T, 8 * 1024 * 64 // (B * H)))
        return {"kind": kind, "B": B, "T": T, "H": H, "state": state}
    if kind in ("time_mix", "channel_mix"):
        C = rng.choice([768, 2048, 2560, 4096])
        if rng.random() < 0.5:
            case = {"kind": kind, "B": _log_int(rng, 1, 256), "T": 1, "C": C}
        else:
            B = rng.choice([1, 1, 2, 3, 4])
            case = {"kind": kind, "B": B, "T": _log_int(rng, 5, 2000 // B), "C": C}
        if kind == "time_mix":
            case["weights"] = rng.choice(["nk", "kn"])
        return case
    if kind == "head":
        return {"kind": kind, "B": _log_int(rng, 1, 256), "C": rng.choice([768, 2048, 4096]),
                "weights": rng.choice(["nk", "kn"])}
    if kind == "sample":
        top_k, top_p = rng.choice([(-1, 1.0), (-1, 0.5), (-1, 0.9), (40, 0.9), (100, 1.0), (1, 1.0)])
        return {"kind": kind, "B": _log_int(rng, 1, 256), "V": rng.choice([50304, 65536]), "top_k": top_k,
                "top_p": top_p, "penalties": rng.random() < 0.5}
    if kind == "decode":
        return {"kind": kind, "B": _log_int(rng, 1, 160), "shape": "1.5b", "layers": rng.choice([6, 12])}
    return {"kind": kind, "B": rng.randint(1, 128), "chunks": rng.randint(1, 3), "T": _log_int(rng, 20, 500),
            "shape": rng.choice(["1.5b", "7b"]), "layers": 3}


# ---------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _n(g, *shape, s=1.0):
    return (torch.randn(*shape, generator=g, device="cuda") * s).half()


def _u(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda")


def _wkv_inputs(case, seed):
    """r, w, k, v, a, b as a layer's projections and gate give them (w before its decay
    function, from long to short memory across the channels), and the state."""
    B, T, H = case["B"], case["T"], case["H"]
    C = H * HEAD
    g = _gen(seed)
    r, v = _n(g, B, T, C), _n(g, B, T, C)
    w = (-6.0 + 5.0 * _u(g, C) + torch.randn(B, T, C, generator=g, device="cuda") * 0.5).half()
    k = torch.randn(B, T, H, HEAD, generator=g, device="cuda")
    gate = torch.sigmoid(torch.randn(B, T, H, HEAD, generator=g, device="cuda"))
    kk = F.normalize(k, dim=-1)
    ins = [r, w, (k * gate).reshape(B, T, C).half(), v, (-kk).reshape(B, T, C).half(),
           (kk * gate).reshape(B, T, C).half()]
    if case["state"] == "fp16":
        return ins, _n(g, B, H, HEAD, HEAD, s=0.1), None
    pool = torch.randn(4 * B, H, HEAD, HEAD, generator=g, device="cuda") * 0.1
    slots = torch.randperm(4 * B, generator=g, device="cuda")[:B].int()
    return ins, pool, slots


def _layer(C, ranks, g):
    """One layer's weights (nn.Linear layout [out, in]) and vectors, of a trained layer's sizes."""
    W = {m: _u(g, C).half() for m in TMIX + ("x_k_ffn",)}
    for name in ("ln1_w", "ln2_w", "lnx_w", "k_a"):
        W[name] = 1.0 + _n(g, C, s=0.1)
    for name in ("ln1_b", "ln2_b", "lnx_b", "a0", "v0", "r_k"):
        W[name] = _n(g, C, s=0.1)
    W["w0"] = (-6.0 + 5.0 * _u(g, C)).half()
    W["k_k"] = (0.85 + 0.1 * _u(g, C)).half()
    for name in ("Wr", "Wk", "Wv", "Wo"):
        W[name] = _n(g, C, C, s=0.02)
    for name, rank in zip("wavg", ranks):
        W[name + "1"], W[name + "2"] = _n(g, rank, C, s=0.02), _n(g, C, rank, s=0.1)
    return W


def _time_mix_inputs(case, seed):
    B, T, C = case["B"], case["T"], case["C"]
    H = C // HEAD
    g = _gen(seed)
    W = _layer(C, RANKS[C], g)
    s = {"W": W, "x": _n(g, B, T, C), "res": _n(g, B, T, C), "shift": _n(g, B, C), "v_first": _n(g, B, T, C),
         "pool": torch.randn(2 * B, H, HEAD, HEAD, generator=g, device="cuda") * 0.1,
         "slots": torch.randperm(2 * B, generator=g, device="cuda")[:B].int()}
    if case["weights"] == "kn":
        for name in ("Wr", "Wk", "Wv", "Wo"):
            W[name] = W[name].t().contiguous()
    return s


def _channel_mix_inputs(case, seed):
    B, T, C = case["B"], case["T"], case["C"]
    g = _gen(seed)
    return {"x": _n(g, B, T, C), "res": _n(g, B, T, C), "shift": _n(g, B, C), "ln_w": 1.0 + _n(g, C, s=0.1),
            "ln_b": _n(g, C, s=0.1), "x_k": _u(g, C).half(), "key": _n(g, 4 * C, C, s=0.02),
            "value": _n(g, 4 * C, C, s=0.02)}


VOCAB = 65536


def _head_inputs(case, seed):
    B, C = case["B"], case["C"]
    g = _gen(seed)
    s = {"x": _n(g, B, 1, C), "res": _n(g, B, 1, C), "ln_w": 1.0 + _n(g, C, s=0.1), "ln_b": _n(g, C, s=0.1),
         "head": _n(g, VOCAB, C, s=0.02)}
    if case["weights"] == "kn":
        s["head"] = s["head"].t().contiguous()
    return s


def _config(case):
    c = RWKV7Config.preset(case["shape"])
    return RWKV7Config(case["layers"], c.n_embd, c.dim_ffn, c.rank_w, c.rank_a, c.rank_v, c.rank_g, c.vocab)


def _model_inputs(case, seed):
    """The model, its state pools, and the tokens and slots of each group of sequences:
    [(tokens [B] or [B, T], slots [B]), ...], the decode rows first."""
    cfg = _config(case)
    g = _gen(seed)
    model = RWKV7Model(cfg, torch.device("cuda"), seed=seed)
    seqs = case["B"] + case.get("chunks", 0)
    layout = capi.WKV_STATE_ILV if case["kind"] == "decode" else capi.WKV_STATE_STD
    state = RWKV7State(cfg, seqs + seqs // 4 + 1, torch.device("cuda"), seed=seed + 1, layout=layout)
    for shift in (state.att_shift, state.ffn_shift):  # rows of sequences under way
        shift.normal_(generator=g)
    slots = torch.randperm(state.n_slots, generator=g, device="cuda").int()
    groups = [((_u(g, case["B"]) * cfg.vocab).int(), slots[:case["B"]])]
    if case["kind"] == "mixed":
        groups.append(((_u(g, case["chunks"], case["T"]) * cfg.vocab).int(), slots[case["B"]:seqs]))
    return model, state, groups


def _captured(call, buffers):
    """A HIP graph of call(), its result, and the buffers that the warm-up call wrote as they
    were before it."""
    saved = [b.clone() for b in buffers]
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        call()
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for b, s in zip(buffers, saved):
        b.copy_(s)
    return graph, out


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "wkv":
        s["ins"], s["state"], s["slots"] = _wkv_inputs(case, seed)
    elif kind == "time_mix":
        s.update(_time_mix_inputs(case, seed))
        if case["T"] == 1:
            s["graph"], s["out"] = _captured(lambda: _time_mix(s), [s["shift"], s["pool"]])
    elif kind == "channel_mix":
        s.update(_channel_mix_inputs(case, seed))
    elif kind == "head":
        s.update(_head_inputs(case, seed))
    elif kind == "sample":
        # a trained model's logits: a broad body and a few likely tokens
        B, V = case["B"], case["V"]
        g = _gen(seed)
        s["logits"] = torch.randn(B, V, generator=g, device="cuda") * 2.5
        s["logits"] += (_u(g, B, V) < 24 / V) * (4.0 + 8.0 * _u(g, B, V))
        s["states"] = SMP.setup_rand(seed, B)
        if case["penalties"]:  # of the tokens of a few hundred steps
            s["penalties"] = (_u(g, B, V) < 300 / V) * (0.5 * _u(g, B, V))
    elif kind == "decode":
        s["model"], s["state"], [(s["tokens"], s["slots"])] = _model_inputs(case, seed)
        engine = s["engine"] = DecodeEngine(s["model"], case["B"])
        st = s["state"]
        s["graph"], s["logits"] = _captured(lambda: engine.step(st, s["tokens"], s["slots"]),
                                            [st.wkv, st.att_shift, st.ffn_shift])
    else:
        s["model"], s["state"], s["groups"] = _model_inputs(case, seed)
        s["engine"] = MixedEngine(s["model"], max_rows=case["B"] + case["chunks"] * case["T"],
                                  max_seqs=case["B"] + case["chunks"])
    return s


# ---------------------------------------------------------------- a pass

def _time_mix(s):
    case, W = s["case"], s["W"]
    B, T, C = case["B"], case["T"], case["C"]
    H, M = C // HEAD, B * T
    Rw, Ra, Rv, Rg = RANKS[C]
    linear = LIN.linear_f16 if case["weights"] == "kn" else LIN.linear_f16_orig
    mixes = [W[m] for m in TMIX]
    if T == 1:
        res, xr, xw, xk, xv, xa, xg = NORM.add_layer_norm_tmix_mix6_f16(s["x"], s["res"], s["shift"], W["ln1_w"],
                                                                        W["ln1_b"], *mixes)
    else:
        res, y = NORM.add_layer_norm_f16(s["x"], s["res"], W["ln1_w"], W["ln1_b"])
        xr, xw, xk, xv, xa, xg = MIX.tmix_mix6(B, T, C, y, s["shift"], *mixes)
    rows = lambda t: t.view(M, C)  # noqa: E731
    btc = lambda t: t.view(B, T, C)  # noqa: E731
    r, k, v = linear(xr, W["Wr"]), linear(xk, W["Wk"]), linear(xv, W["Wv"])
    w1, a1, g1, v1 = RANK.linear_wagv_rank_in_f16(M, C, Rw, Ra, Rg, Rv, rows(xw), rows(xa), rows(xg), rows(xv),
                                                  W["w1"], W["a1"], W["g1"], W["v1"])
    w, a12, g, v = RANK.linear_wagv_rank_out_f16(M, C, Rw, Ra, Rg, Rv, w1, a1, g1, v1, W["w2"], W["a2"], W["g2"],
                                                 W["v2"], rows(v), rows(s["v_first"]), W["v0"])
    w, v = btc(MIX.add_vec(C, w, W["w0"])), btc(v)
    new_k, neg_kk, kka = MIX.tmix_kk_a_gate(B, T, C, H, k, W["k_k"], W["a0"], btc(a12), W["k_a"])
    y = WKV.wkv_forward_slots_fp32(B, T, C, H, s["pool"], s["slots"], r, w, new_k, v, neg_kk, kka, validate=False)
    o_in = MIX.tmix_lnx_rkvres_xg(B, T, C, H, y, r, new_k, v, W["r_k"], W["lnx_w"], W["lnx_b"], btc(g))
    return {"res": res, "o": linear(o_in, W["Wo"]), "shift": s["shift"], "pool": s["pool"]}


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "wkv":
        B, T, H = case["B"], case["T"], case["H"]
        if case["state"] == "fp16":
            y, _ = WKV.wkv_seq_fp16(B, T, H * HEAD, H, s["state"], *s["ins"])
        else:
            y = WKV.wkv_forward_slots_fp32(B, T, H * HEAD, H, s["state"], s["slots"], *s["ins"], validate=False)
        return {"y": y, "state": s["state"]}
    if kind == "time_mix":
        if case["T"] > 1:
            return _time_mix(s)
        s["graph"].replay()
        return s["out"]
    if kind == "channel_mix":
        B, T, C = case["B"], case["T"], case["C"]
        res, y = NORM.add_layer_norm_f16(s["x"], s["res"], s["ln_w"], s["ln_b"])
        out = MIX.cmix_sparse_rows(B, T, C, 4 * C, y, s["shift"], s["x_k"], s["key"], s["value"])
        return {"res": res, "out": out, "shift": s["shift"]}
    if kind == "head":
        h = NORM.add_last_layer_norm_f16(s["x"], s["res"], s["ln_w"], s["ln_b"])
        return {"logits": (LIN.linear_f16 if case["weights"] == "kn" else LIN.linear_f16_orig)(h, s["head"])}
    if kind == "sample":
        if case["penalties"]:
            tokens = SMP.repetition_topk_topp(s["logits"], s["penalties"], s["states"], 0.2, 0.1, 0.996, 0.9,
                                              case["top_k"], case["top_p"])
            return {"tokens": tokens, "penalties": s["penalties"], "states": s["states"]}
        return {"tokens": SMP.temperature_topk_topp(s["logits"], s["states"], 0.9, case["top_k"], case["top_p"]),
                "states": s["states"]}
    st = s["state"]
    if kind == "decode":
        s["graph"].replay()
        logits = s["logits"]
    else:
        logits = s["engine"].step(st, s["groups"][0], s["groups"][1:])
    return {"logits": logits, "wkv": st.wkv, "att_shift": st.att_shift, "ffn_shift": st.ffn_shift}


# ---------------------------------------------------------------- what a pass cannot do without

def _wkv_work(B, T, H, state_bytes):
    # state read and written, six fp16 inputs, y; per token and state element: decay (1),
    # S.a (2), the two rank-1 updates (4), S.r (2)
    return 2 * B * H * 4096 * state_bytes + 7 * 2 * B * T * H * HEAD, 9 * B * T * H * 4096


def _layer_matmul(C, F4, ranks):
    """Weight elements of a layer's time mix and channel mix."""
    return 4 * C * C + 2 * C * sum(ranks), 2 * C * F4


def work(case):
    kind, B = case["kind"], case["B"]
    if kind == "wkv":
        b, f = _wkv_work(B, case["T"], case["H"], 2 if case["state"] == "fp16" else 4)
        return {"bytes": b, "flops": f}
    if kind == "time_mix":
        T, C = case["T"], case["C"]
        M = B * T
        weights, _ = _layer_matmul(C, 4 * C, RANKS[C])
        # x, res, v_first read; res', o written; shift rows and states read and written
        return {"bytes": 2 * weights + 2 * 5 * M * C + 2 * 2 * B * C + 2 * B * C * HEAD * 4,
                "flops": 2 * M * weights + 9 * M * C * HEAD}
    if kind == "channel_mix":
        T, C = case["T"], case["C"]
        M = B * T
        return {"bytes": 2 * 8 * C * C + 2 * 4 * M * C + 2 * 2 * B * C, "flops": 2 * M * 8 * C * C}
    if kind == "head":
        C = case["C"]
        return {"bytes": 2 * VOCAB * C + 2 * 2 * B * C + 2 * B * VOCAB, "flops": 2 * B * VOCAB * C}
    if kind == "sample":
        # logits read; penalties read and written
        return {"bytes": B * case["V"] * (12 if case["penalties"] else 4), "flops": 0}
    cfg = _config(case)
    C, H = cfg.n_embd, cfg.n_head
    tm, cm = _layer_matmul(C, cfg.dim_ffn, (cfg.rank_w, cfg.rank_a, cfg.rank_v, cfg.rank_g))
    seqs = B + case.get("chunks", 0)
    rows = B + case.get("chunks", 0) * case.get("T", 0)
    # weights once; embedding rows; states and shift rows read and written; logits written
    return {"bytes": 2 * (cfg.n_layer * (tm + cm) + cfg.vocab * C) + 2 * rows * C
            + cfg.n_layer * seqs * (2 * H * 4096 * 4 + 2 * 2 * 2 * C) + 2 * seqs * cfg.vocab,
            "flops": 2 * rows * cfg.n_layer * (tm + cm) + 2 * seqs * C * cfg.vocab
            + 9 * rows * cfg.n_layer * C * HEAD}


# ---------------------------------------------------------------- the same outputs in 64 bits

def _decay(w):
    return torch.exp(-math.exp(-0.5) * torch.sigmoid(w))


def _wkv64(S, r, w, k, v, a, b):
    """[B, T, C] inputs and the states [B, H, 64, 64] in 64 bits -> y [B, T, C], the states after."""
    B, T, C = r.shape
    r, w, k, v, a, b = (x.view(B, T, C // HEAD, HEAD) for x in (r, w, k, v, a, b))
    d = _decay(w)
    y = torch.empty_like(r)
    for t in range(T):
        sa = torch.matmul(S, a[:, t, :, :, None])
        S = S * d[:, t, :, None, :] + sa * b[:, t, :, None, :] + v[:, t, :, :, None] * k[:, t, :, None, :]
        y[:, t] = torch.matmul(S, r[:, t, :, :, None])[..., 0]
    return y.view(B, T, C), S


def _shifted(y, shift):
    """The previous token's rows of y [B, T, C], shift [B, C] before the first."""
    return torch.cat([shift[:, None], y[:, :-1]], 1)


def _ln64(x, w, b):
    return F.layer_norm(x, (x.shape[-1],), w, b, 1e-5)


def _time_mix64(W, x, res, shift, S, v_first):
    """x, res, v_first (None: this is the first layer) [B, T, C], shift [B, C], S in 64 bits ->
    res', o, shift', S', v_first."""
    B, T, C = x.shape
    H = C // HEAD
    heads = lambda t: t.view(B, T, H, HEAD)  # noqa: E731
    res = x + res
    y = _ln64(res, W["ln1_w"], W["ln1_b"])
    prev = _shifted(y, shift)
    xr, xw, xk, xv, xa, xg = (y + (prev - y) * W[m] for m in TMIX)
    r, k, v = xr @ W["Wr"].t(), xk @ W["Wk"].t(), xv @ W["Wv"].t()
    w = W["w0"] + torch.tanh(xw @ W["w1"].t()) @ W["w2"].t()
    a = torch.sigmoid(W["a0"] + (xa @ W["a1"].t()) @ W["a2"].t())
    g = torch.sigmoid(xg @ W["g1"].t()) @ W["g2"].t()
    if v_first is None:
        v_first = v
    else:
        v = v + (v_first - v) * torch.sigmoid(W["v0"] + (xv @ W["v1"].t()) @ W["v2"].t())
    kk = F.normalize(heads(k * W["k_k"]), dim=-1, eps=1e-12).view(B, T, C)
    k = k * (a * W["k_a"] + (1 - W["k_a"]))
    out, S = _wkv64(S, r, w, k, v, -kk, kk * a)
    out = heads(out)
    out = ((out - out.mean(-1, keepdim=True)) / torch.sqrt(out.var(-1, unbiased=False, keepdim=True) + 64e-5)).view(
        B, T, C) * W["lnx_w"] + W["lnx_b"]
    bonus = heads(r * k * W["r_k"]).sum(-1, keepdim=True) * heads(v)
    o = ((out + bonus.view(B, T, C)) * g) @ W["Wo"].t()
    return res, o, y[:, -1], S, v_first


def _channel_mix64(x, res, shift, ln_w, ln_b, x_k, key, value_fc):
    """value_fc [F, C] -> res', out, shift'."""
    res = x + res
    y = _ln64(res, ln_w, ln_b)
    xk = y + (_shifted(y, shift) - y) * x_k
    return res, (torch.relu(xk @ key.t()) ** 2) @ value_fc, y[:, -1]


def _interleaved(wkv):
    """WKV blocks as the decode engine's pool lays them out: row i's columns 4q .. 4q + 3 at
    floats 4 (64 q + i) ..."""
    return wkv.view(*wkv.shape[:-1], 16, 4).transpose(-3, -2).reshape(wkv.shape)


def _model64(case, seed):
    model, state, groups = _model_inputs(case, seed)
    cfg = model.cfg
    H = cfg.n_head
    d = lambda t: t.double()  # noqa: E731
    wkv, att, ffn = d(state.wkv_standard()), d(state.att_shift), d(state.ffn_shift)
    xs, logits = [], []
    for tokens, _ in groups:
        tokens = tokens.view(tokens.shape[0], -1).long()
        xs.append([d(model.emb)[tokens], 0.0, None])  # block output, residual stream, v_first
    for layer, weights in enumerate(model.layers):
        W = {k: d(t) for k, t in weights.items()}
        for x, (_, slots) in zip(xs, groups):
            sl = slots.long()
            res, o, att[layer, sl], wkv[layer, sl], x[2] = _time_mix64(W, x[0], x[1], att[layer, sl],
                                                                     wkv[layer, sl].view(-1, H, HEAD, HEAD), x[2])
            x[1], x[0], ffn[layer, sl] = _channel_mix64(o, res, ffn[layer, sl], W["ln2_w"], W["ln2_b"],
                                                        W["x_k_ffn"], W["key"], W["value"].t())
    for x in xs:
        h = _ln64((x[0] + x[1])[:, -1], d(model.ln_out_w), d(model.ln_out_b))
        logits.append(h @ d(model.head).t())
    return {"logits": torch.cat(logits), "wkv": _interleaved(wkv) if case["kind"] == "decode" else wkv,
            "att_shift": att, "ffn_shift": ffn}


def exact(case, seed):
    kind = case["kind"]
    if kind == "wkv":
        ins, state, slots = _wkv_inputs(case, seed)
        ins, S = [x.double() for x in ins], state.double()
        if slots is None:
            y, S = _wkv64(S, *ins)
            return {"y": y, "state": S}
        sl = slots.long()
        y, S[sl] = _wkv64(S[sl], *ins)
        return {"y": y, "state": S}
    if kind == "time_mix":
        s = _time_mix_inputs(case, seed)
        W = {k: t.double() for k, t in s["W"].items()}
        if case["weights"] == "kn":
            for name in ("Wr", "Wk", "Wv", "Wo"):
                W[name] = W[name].t()
        sl, pool = s["slots"].long(), s["pool"].double()
        res, o, shift, pool[sl], _ = _time_mix64(W, s["x"].double(), s["res"].double(), s["shift"].double(), pool[sl],
                                                 s["v_first"].double())
        return {"res": res, "o": o, "shift": shift, "pool": pool}
    if kind == "channel_mix":
        s = {k: t.double() for k, t in _channel_mix_inputs(case, seed).items()}
        res, out, shift = _channel_mix64(s["x"], s["res"], s["shift"], s["ln_w"], s["ln_b"], s["x_k"], s["key"],
                                         s["value"])
        return {"res": res, "out": out, "shift": shift}
    if kind == "head":
        s = {k: t.double() for k, t in _head_inputs(case, seed).items()}
        h = _ln64(s["x"][:, -1] + s["res"][:, -1], s["ln_w"], s["ln_b"])
        logits = h @ (s["head"] if case["weights"] == "kn" else s["head"].t())
        return {"logits": logits.view(case["B"], VOCAB)}
    if kind == "sample":
        return None  # a draw: its law has no value of its own
    return _model64(case, seed)


# ---------------------------------------------------------------- how far another implementation may lie

# About four times the error against the 64-bit values measured for each kind, over its outputs:
# 2.1e-4 is the rounding of an fp16 output by itself; a layer or a model rounds its
# intermediates too.
REL = {"time_mix": 4e-3, "channel_mix": 2e-3, "head": 1.2e-3, "decode": 8e-3, "mixed": 8e-3}


def tolerance(case):
    if case["kind"] == "wkv":
        return {"rel": 1e-2 if case["state"] == "fp16" else 1e-3}
    if case["kind"] == "sample":  # the same draws; the penalties are 32-bit products and sums
        return {"rel": 1e-6}
    return {"rel": REL[case["kind"]]}
