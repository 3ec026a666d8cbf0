"""The work that this framework is used for, as cases to be timed and compared.

A GSPO step of the Nanopore basecaller's decoder is: encode the windows, prefill their frames, decode a group of
calls per window, score the calls, and update the policy. Each case is one call of that, or one layer of it, through
the entry points that such a program calls, at the sizes it has (the benchmark's configurations) or at small and
ragged ones. Listed by hand; `draw` gives more of the same ranges.

Kinds of case and their sizes:
  decode    one decode step, all layers, LM head included, replayed from a captured graph as the engine runs it
            B sequences, group G (1: own prefix each), prefixes lo..hi frames, own tokens so far, k-mer size k
  prefill   DecodeEngine.prefill: projector, packed prefill, first token. W windows, G calls each
  score     Basecaller.logits: teacher-forced scoring of W windows x G calls of T tokens
  train     one micro-batch of the update: train_logits, the sequence-ratio loss, backward into every parameter
  attention one layer's causal attention over packed windows, forward and backward, plain or with shared prefixes
  mlp       one layer's MLP over M packed rows: gate_up + SwiGLU, down + residual, and the next norm
  encode    DoradoEncoder.forward_varlen of n chunks of raw signal
  loss      the clipped sequence-ratio objective of B calls x T tokens and its gradient with respect to the logits
  reward    strict identity of W windows x G calls against their labels, from the engine's output tokens
"""

import math

import numpy as np
import torch
import torch.nn.functional as F

from viktor_amd import hip_ops as ops
from viktor_amd.decoder import DecoderConfig, KVCache
from viktor_amd.encoder import DoradoEncoder
from viktor_amd.engine import DecodeEngine
from viktor_amd.fast_decoder import FastDecoder
from viktor_amd.gspo import bf16_copy, sequence_ratio_loss
from viktor_amd.model import Basecaller
from viktor_amd.reward import gspo_rewards_from_tokens
from viktor_amd.synthetic import SUP_ENCODER_CFG
from viktor_amd.tokenizer import BOS, EOS, PAD, KmerTokenizer
from viktor_amd.train import HipAdamW, TrainPlan, train_logits

DEV = "cuda"
BF16 = torch.bfloat16
D_ENC, D_MODEL, LAYERS, HEADS, KV_HEADS, HEAD = 512, 512, 8, 8, 2, 64
FFN, QKV, EPS = 1536, 768, 1e-6
LAYER_WEIGHTS = D_MODEL * QKV + D_MODEL * D_MODEL + 3 * D_MODEL * FFN
ROW = 2 * KV_HEADS * HEAD * 2  # bytes of one position's keys and values in one layer
CONVS = [l for l in SUP_ENCODER_CFG["model"]["encoder"]["conv"]["sublayers"] if l["type"] == "convolution"]
GRAIN = 768  # samples: 64 frames


def listed():
    return [
        # the smallest call: four calls decoded side by side, a few tokens in; launches and latency count
        {"name": "decode_4", "kind": "decode", "B": 4, "G": 1, "lo": 2048, "hi": 2048, "own": 32, "k": 1, "mix": 1},
        # the rollout's step in the middle of a call: 64 windows x 8 calls that share their window's prefix
        {"name": "decode_rollout", "kind": "decode", "B": 512, "G": 8, "lo": 2048, "hi": 2048, "own": 512, "k": 1,
         "mix": 2},
        # basecalling with the 4-mer vocabulary: every sequence its own prefix, of its own length
        {"name": "decode_kmer", "kind": "decode", "B": 1024, "G": 1, "lo": 1200, "hi": 2048, "own": 170, "k": 4,
         "mix": 3},
        # a few ragged windows: the prefill of an interactive call
        {"name": "prefill_ragged", "kind": "prefill", "W": 3, "G": 1, "lo": 301, "hi": 1999, "k": 4, "mix": 4},
        # the rollout's prefill: 64 windows of 2048 frames, handed over eight times each
        {"name": "prefill_rollout", "kind": "prefill", "W": 64, "G": 8, "lo": 2048, "hi": 2048, "k": 1, "mix": 5},
        # scoring a slice of a rollout: 8 windows x 8 calls
        {"name": "score", "kind": "score", "W": 8, "G": 8, "lo": 2048, "hi": 2048, "T": 896, "k": 1, "mix": 6},
        # the update's micro-batch of 32 calls: 4 windows x 8 calls
        {"name": "train", "kind": "train", "W": 4, "G": 8, "lo": 2048, "hi": 2048, "T": 768, "k": 1, "mix": 7},
        # attention of ragged windows whose calls are not shared (odd lengths throughout)
        {"name": "attention", "kind": "attention", "W": 24, "G": 1, "lo": 301, "hi": 2817, "T": 0, "mix": 8},
        # the MLP of a scoring batch's packed rows on the fp32 residual stream
        {"name": "mlp", "kind": "mlp", "M": 45057, "stream": "f32"},
        # one half of a rollout's windows through the encoder, the last chunks of reads shorter than the others
        {"name": "encode", "kind": "encode", "n": 64, "lo": 4608, "hi": 12288, "mix": 10},
        # the objective over a whole rollout's calls
        {"name": "loss", "kind": "loss", "B": 512, "T": 1024, "k": 1},
        # the reward of a whole rollout
        {"name": "reward", "kind": "reward", "W": 64, "G": 8, "lo": 700, "hi": 1000, "k": 1, "mix": 12},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "score", "train", "attention", "mlp", "encode", "loss", "reward"])
    mix = rng.randrange(1, 1 << 20)
    k, G = rng.choice([1, 1, 4]), rng.choice([1, 8])
    hi = _log(rng, 64, 2048)
    lo = hi if rng.random() < 0.4 else max(33, int(hi * rng.uniform(0.4, 1.0)))
    if kind == "decode":
        B = G * _log(rng, 1, 64 if G == 8 else 1024)
        return {"kind": kind, "B": B, "G": G, "lo": lo, "hi": hi, "own": rng.randrange(0, 1000), "k": k, "mix": mix}
    if kind == "prefill":
        return {"kind": kind, "W": _log(rng, 1, 64), "G": G, "lo": lo, "hi": hi, "k": k, "mix": mix}
    if kind == "score":
        return {"kind": kind, "W": _log(rng, 1, 8), "G": G, "lo": lo, "hi": hi, "T": 128 * rng.randrange(1, 8), "k": k,
                "mix": mix}
    if kind == "train":
        return {"kind": kind, "W": _log(rng, 1, 4), "G": G, "lo": lo, "hi": hi, "T": 128 * rng.randrange(1, 7), "k": k,
                "mix": mix}
    if kind == "attention":
        T = 128 * rng.randrange(1, 7) if G == 8 else 0
        return {"kind": kind, "W": _log(rng, 1, 4 if G == 8 else 24), "G": G, "lo": lo, "hi": hi, "T": T, "mix": mix}
    if kind == "mlp":
        return {"kind": kind, "M": _log(rng, 4096, 131136), "stream": rng.choice(["f32", "bf16"])}
    if kind == "encode":
        top = GRAIN * rng.randrange(1, 17)
        return {"kind": kind, "n": _log(rng, 1, 64), "lo": GRAIN * rng.randrange(1, top // GRAIN + 1), "hi": top,
                "mix": mix}
    if kind == "loss":
        return {"kind": kind, "B": _log(rng, 8, 512 if k == 1 else 64), "T": 128 * rng.randrange(1, 9), "k": k}
    top = _log(rng, 64, 1000)
    return {"kind": kind, "W": _log(rng, 1, 64), "G": 8, "lo": max(32, top // 2), "hi": top, "k": k, "mix": mix}


# ---- inputs ---------------------------------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _lens(case, n, step=1):
    """n lengths from lo to hi (steps of `step`), both ends among them; those of a case are the same for every seed."""
    if case["lo"] == case["hi"]:
        return [case["hi"]] * n
    r = np.random.default_rng(case["mix"])
    v = (r.integers(case["lo"] // step, case["hi"] // step + 1, n) * step).tolist()
    v[0] = case["hi"]
    return v


def _vocab(k):
    return 7 if k == 1 else 343


def _model(k, seed):
    """The decoder and projector with seeded weights N(0, 1) / sqrt(fan in), made on the GPU, fp32."""
    tok = KmerTokenizer(k)
    with torch.device(DEV):
        m = Basecaller(None, tok, DecoderConfig(vocab_size=tok.vocab_size, rope_theta=1e6), d_enc=D_ENC).eval()
    g = _gen(seed)
    with torch.no_grad():
        for name, p in sorted(m.named_parameters()):
            v = torch.randn(p.shape, generator=g, device=DEV)
            if name.endswith("embed.weight"):
                p.copy_(v)
            elif p.dim() == 2:
                p.copy_(v / math.sqrt(p.shape[1]))
            elif name.endswith("bias"):
                p.copy_(0.1 * v)
            else:
                p.copy_(1 + 0.1 * v)
    return m


def _randn(shape, g, dtype=BF16):
    return torch.empty(shape, dtype=dtype, device=DEV).normal_(generator=g)


def _tokens(B, T, k, g):
    """BOS, then full k-mers."""
    t = torch.randint(3, 3 + 4 ** k, (B, T), generator=g, device=DEV)
    t[:, 0] = BOS
    return t


def _decode_inputs(case, seed):
    B, G, own = case["B"], case["G"], case["own"]
    g = _gen(seed + 7)
    inf = bf16_copy(_model(case["k"], seed))
    plens = _lens(case, B // G)
    cfg = inf.decoder.cfg
    top = case["hi"] + 1
    cap = max(own + 8, 2)
    if G == 1:
        cache, prefix = KVCache(cfg, B, top + cap, BF16, DEV), None
        cache.k.normal_(generator=g)
        cache.v.normal_(generator=g)
        at = torch.tensor(plens, device=DEV) + 1 + own
        rope = at
    else:
        cache = KVCache(cfg, B, cap, BF16, DEV, pad_rows=DecodeEngine.OWN_PAD_ROWS)
        prefix = KVCache(cfg, B // G, top, BF16, DEV, pad_rows=DecodeEngine.PREFIX_PAD_ROWS)
        for c in (cache, prefix):
            c.k.normal_(generator=g)
            c.v.normal_(generator=g)
        at = torch.full((B,), own, device=DEV)
        rope = torch.tensor(plens, device=DEV).repeat_interleave(G) + 1 + own
    tok = torch.randint(3, 3 + 4 ** case["k"], (B,), generator=g, device=DEV)
    return inf, plens, cache, prefix, at.to(torch.int32), rope.to(torch.int32), tok


def _prepare_decode(case, seed):
    inf, plens, cache, prefix, at, rope, tok = _decode_inputs(case, seed)
    B, G = case["B"], case["G"]
    fast = FastDecoder(inf.decoder)
    fast.decode_workspace = ops.decode_attention_workspace(B, HEADS, cache.max_len, DEV)
    rows = torch.arange(B, dtype=torch.int32, device=DEV)
    seqlens = at + 1
    shared = None
    if G > 1:
        plen32 = torch.tensor(plens, dtype=torch.int32, device=DEV) + 1
        shared = (prefix, plen32, G, ops.decode_attention_grouped_workspace(B, G, prefix.max_len, cache.max_len, DEV))
    s = {"keep": (inf, fast, rows, seqlens, shared, cache, at, rope, tok)}

    def step():
        if shared is None:
            h = fast.decode(None, at, rows, seqlens, cache, tok=tok)
        else:
            x = fast.decode_residual(at, rows, seqlens, cache, rope_pos=rope, tok=tok, prefix=shared)
            h = ops.add_rmsnorm(x, fast.w(inf.decoder.norm.weight), EPS)
        return h, inf.decoder.head(h)

    with torch.no_grad():
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()
            step()
        torch.cuda.current_stream().wait_stream(side)
        s["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(s["graph"]):
            s["hidden"], s["logits"] = step()
    # the token's new keys and values, where all sequences have them at the same position of the cache
    s["new"] = []
    if G > 1 or case["lo"] == case["hi"]:
        row = int(at[0])
        s["new"] = [cache.k[:, :, row], cache.v[:, :, row]]
    return s


def _prepare_prefill(case, seed):
    W, G = case["W"], case["G"]
    inf = bf16_copy(_model(case["k"], seed))
    plens = _lens(case, W)
    lens = [n for n in plens for _ in range(G)]
    one = _randn((sum(plens), D_ENC), _gen(seed + 7), torch.float32)
    frames = one if G == 1 else torch.cat([f for f in one.split(plens) for _ in range(G)])
    eng = DecodeEngine(inf, W * G, 16, case["hi"], cuda_graph=False, logprobs=True, group_size=G)
    return {"eng": eng, "frames": frames, "lens": lens, "one": one, "plens": plens}


def _prepare_score(case, seed):
    W, G = case["W"], case["G"]
    g = _gen(seed + 7)
    plens = torch.tensor(_lens(case, W), device=DEV)
    frames = _randn((W, case["hi"], D_ENC), g, torch.float32).repeat_interleave(G, 0)
    tokens = _tokens(W * G, case["T"], case["k"], g)
    return {"model": _model(case["k"], seed), "frames": frames, "plens": plens.repeat_interleave(G), "tokens": tokens,
            "G": G}


def _objective_inputs(B, T, k, g):
    """Call lengths (in tokens, EOS the last), targets, mask, bases and advantages of B calls."""
    n = torch.randint(max(2, T * 2 // 3), T + 1, (B,), generator=g, device=DEV)
    at = torch.arange(T, device=DEV)[None]
    t = torch.randint(3, 3 + 4 ** k, (B, T), generator=g, device=DEV)
    t = torch.where(at == n[:, None] - 1, EOS, torch.where(at < n[:, None], t, PAD))
    return n, t, t != PAD, (n - 1).float() * k, torch.randn(B, generator=g, device=DEV)


def _prepare_train(case, seed):
    s = _prepare_score(case, seed)
    m = s["model"].train()
    B, T = s["tokens"].shape
    n, targets, mask, bases, adv = _objective_inputs(B, T, case["k"], _gen(seed + 9))
    s["tokens"] = torch.cat([torch.full((B, 1), BOS, device=DEV), targets[:, :-1]], 1)
    s.update(opt=HipAdamW(list(m.parameters()), lr=1e-5), targets=targets, mask=mask, bases=bases, adv=adv)
    with torch.no_grad():  # the old policy's log-probs: the first step of an update starts from them
        z = train_logits(m, s["frames"], s["tokens"], s["plens"], group_size=s["G"])
        s["old"] = ops.gspo_score(z.contiguous(), targets.clamp(min=0).contiguous())["lp"]
    return s


def _attention_layout(case):
    W, G, T = case["W"], case["G"], case["T"]
    pre = _lens(case, W)
    return pre, sum(pre) + W * G * T if G > 1 else sum(pre)


def _prepare_attention(case, seed):
    pre, n = _attention_layout(case)
    g = _gen(seed)
    plan = TrainPlan(pre, DEV) if case["G"] == 1 else TrainPlan.shared(pre, case["G"], case["T"], DEV)
    q, dout = _randn((n, HEADS, HEAD), g), _randn((n, HEADS, HEAD), g)
    k, v = _randn((n, KV_HEADS, HEAD), g), _randn((n, KV_HEADS, HEAD), g)
    return {"plan": plan, "q": q, "k": k, "v": v, "dout": dout}


def _prepare_mlp(case, seed):
    g = _gen(seed)
    M = case["M"]
    w = {"gate_up": _randn((2 * FFN, D_MODEL), g) / math.sqrt(D_MODEL), "down": _randn((D_MODEL, FFN), g) / math.sqrt(FFN)}
    dt = torch.float32 if case["stream"] == "f32" else BF16
    return {"h": _randn((M, D_MODEL), g), "x": _randn((M, D_MODEL), g, dt), "norm": 1 + 0.1 * _randn((D_MODEL,), g, dt), **w}


def _encoder_weights(seed):
    g = _gen(seed)
    tx = SUP_ENCODER_CFG["model"]["encoder"]["transformer_encoder"]
    C, Fd = tx["layer"]["d_model"], tx["layer"]["dim_feedforward"]
    sd = {}

    def add(name, shape, fan=None, around=0.0):
        v = torch.randn(shape, generator=g, device=DEV)
        sd[name] = v / math.sqrt(fan) if fan else around + 0.1 * v

    for i, l in enumerate(CONVS):
        add(f"conv.{i}.conv.weight", (l["size"], l["insize"], l["winlen"]), l["insize"] * l["winlen"])
        add(f"conv.{i}.conv.bias", (l["size"],))
    for j in range(tx["depth"]):
        p = f"transformer_encoder.{j}."
        add(p + "self_attn.Wqkv.weight", (3 * C, C), C)
        add(p + "self_attn.out_proj.weight", (C, C), C)
        add(p + "self_attn.out_proj.bias", (C,))
        add(p + "ff.fc1.weight", (2 * Fd, C), C)
        add(p + "ff.fc2.weight", (C, Fd), Fd)
        add(p + "norm1.weight", (C,), around=1.0)
        add(p + "norm2.weight", (C,), around=1.0)
    return sd


def _prepare_encode(case, seed):
    lens = _lens(case, case["n"], GRAIN)
    sd = _encoder_weights(seed)
    enc = DoradoEncoder(SUP_ENCODER_CFG, DEV).load_state_dict(sd)
    return {"enc": enc, "lens": lens, "signal": _randn((sum(lens),), _gen(seed + 7), torch.float32), "weights": sd}


def _prepare_loss(case, seed):
    g = _gen(seed)
    B, T, V = case["B"], case["T"], _vocab(case["k"])
    n, targets, mask, bases, adv = _objective_inputs(B, T, case["k"], g)
    z = (1.5 * _randn((B, T, V), g, torch.float32)).to(BF16).requires_grad_()
    lp = torch.log_softmax(z.detach().float(), -1).gather(-1, targets[..., None])[..., 0]
    old = (lp + 0.05 * _randn((B, T), g, torch.float32)).contiguous()
    return {"z": z, "targets": targets, "mask": mask, "old": old, "bases": bases, "adv": adv}


def _mutate(r, label, rate):
    """A call of a label: substitutions, deletions and insertions, a third of `rate` each."""
    u = r.random(len(label))
    out = np.where(u < rate / 3, r.integers(0, 4, len(label)), label)
    out = out[(u < rate / 3) | (u >= 2 * rate / 3)]
    at = np.flatnonzero(r.random(len(out)) < rate / 3)
    return np.insert(out, at, r.integers(0, 4, len(at)))


def _prepare_reward(case, seed):
    r = np.random.default_rng(seed)
    W, G, k = case["W"], case["G"], case["k"]
    tok = KmerTokenizer(k)
    lens = _lens(case, W)
    labels = [r.integers(0, 4, n) for n in lens]
    weights = [(r.random(n) > 0.03).astype(np.float32) for n in lens]
    T = 128 * -(-(case["hi"] * 5 // 4 + 2) // (128 * k)) + 128
    tokens = np.zeros((W * G, T), dtype=np.int64)
    calls = []
    for i in range(W * G):
        c = _mutate(r, labels[i // G], r.uniform(0.02, 0.2))
        calls.append(c)
        ids = tok.encode("".join("ACGT"[b] for b in c)) + [EOS]
        tokens[i, :len(ids)] = ids
    text = ["".join("ACGT"[b] for b in l) for l in labels]
    return {"tokens": torch.from_numpy(tokens).to(DEV), "tok": tok, "labels": text, "weights": weights, "G": G,
            "raw": (calls, labels)}


_PREPARE = {"decode": _prepare_decode, "prefill": _prepare_prefill, "score": _prepare_score, "train": _prepare_train,
            "attention": _prepare_attention, "mlp": _prepare_mlp, "encode": _prepare_encode, "loss": _prepare_loss,
            "reward": _prepare_reward}


def prepare(case, seed):
    s = _PREPARE[case["kind"]](case, int(seed))
    s["kind"] = case["kind"]
    return s


# ---- one pass -------------------------------------------------------------------------------------------------------
def _run_prefill(s):
    eng = s["eng"]
    eng.prefill(s["frames"], s["lens"])
    c = eng.cache if eng.prefix_cache is None else eng.prefix_cache
    return [eng.out[:, 0], eng.logp[:, 0], c.k, c.v]


def _run_train(s):
    s["opt"].zero_grad()
    z = train_logits(s["model"], s["frames"], s["tokens"], s["plens"], group_size=s["G"])
    loss, ratio, pg, lp = sequence_ratio_loss(z, s["targets"], s["mask"], s["old"], s["bases"], s["adv"])
    loss.backward()
    return [z.detach(), s["opt"].grad]


def _run_attention(s):
    p = s["plan"]
    lse = torch.empty(s["q"].shape[:2], dtype=torch.float32, device=DEV)
    o = ops.varlen_attention(s["q"], s["k"], s["v"], p.attn, lse=lse, prefix=(s["k"], s["v"]) if p.prefixed else None)
    dq, dk, dv = ops.attention_backward(s["q"], s["k"], s["v"], o, s["dout"], lse, p.attn, p.keys)
    return [o, lse, dq, dk, dv]


def _run_mlp(s):
    y = torch.empty_like(s["x"])
    a = ops.linear(s["h"], s["gate_up"], swiglu=True)
    ss = ops.linear_residual_big(a, s["down"], s["x"], out=y)
    return [y, ops.rmsnorm_apply(y, ss, s["norm"], EPS)]


def _run_loss(s):
    s["z"].grad = None
    loss, ratio, pg, lp = sequence_ratio_loss(s["z"], s["targets"], s["mask"], s["old"], s["bases"], s["adv"])
    loss.backward()
    return [loss.detach(), ratio.detach(), lp.detach(), s["z"].grad]


def run(s):
    kind = s["kind"]
    if kind == "decode":
        s["graph"].replay()
        return [s["hidden"], s["logits"], *s["new"]]
    if kind == "prefill":
        return _run_prefill(s)
    if kind == "score":
        return [s["model"].logits(s["frames"], s["tokens"], s["plens"], group_size=s["G"])]
    if kind == "train":
        return _run_train(s)
    if kind == "attention":
        return _run_attention(s)
    if kind == "mlp":
        return _run_mlp(s)
    if kind == "encode":
        return [s["enc"].forward_varlen(s["signal"], s["lens"])]
    if kind == "loss":
        return _run_loss(s)
    r = gspo_rewards_from_tokens(s["tokens"], s["tok"], s["labels"], s["weights"], s["G"])
    return [r["reward"], r["edit_distance"], r["scored_errors"]]


# ---- what a pass cannot do without ----------------------------------------------------------------------------------
def _stack_work(rows, pairs, head_rows, k):
    """The decoder over `rows` packed rows with `pairs` visible (query, key) pairs per layer and head."""
    return 2.0 * rows * LAYERS * LAYER_WEIGHTS + 4.0 * HEAD * HEADS * LAYERS * pairs + 2.0 * head_rows * D_MODEL * _vocab(k)


def _window_pairs(plens, G, T):
    """Visible pairs of windows whose prefix runs once and whose G calls have T tokens each; and the rows."""
    pairs = sum(p * (p + 1) / 2 + G * (T * p + T * (T + 1) / 2) for p in plens)
    return pairs, sum(p + G * T for p in plens)


def work(case):
    kind = case["kind"]
    weights = LAYERS * LAYER_WEIGHTS
    if kind == "decode":
        B, G = case["B"], case["G"]
        pre = [p + 1 for p in _lens(case, B // G)]
        own = case["own"] + 1
        read = sum(pre) + B * own
        V = _vocab(case["k"])
        nb = 2 * (weights + V * D_MODEL) + LAYERS * ROW * read + 2 * B * (D_MODEL + V)
        return {"bytes": nb, "flops": _stack_work(B, G * sum(pre) + B * own, B, case["k"])}
    if kind == "prefill":
        W, G = case["W"], case["G"]
        plens = _lens(case, W)
        n = sum(plens)
        pairs = sum((p + 1) * (p + 2) / 2 for p in plens)
        fl = _stack_work(n + W, pairs, W, case["k"]) + 4.0 * n * D_MODEL * D_ENC
        # the last layer finishes one row of each window
        fl -= 2.0 * n * (LAYER_WEIGHTS - D_MODEL * 2 * KV_HEADS * HEAD) + 4.0 * HEAD * HEADS * (pairs - n - W)
        return {"bytes": 4 * G * n * D_ENC + 2 * weights + LAYERS * ROW * (n + W), "flops": fl}
    if kind in ("score", "train"):
        W, G, T, k = case["W"], case["G"], case["T"], case["k"]
        plens = _lens(case, W)
        pairs, rows = _window_pairs(plens, G, T)
        B = W * G
        fl = _stack_work(rows, pairs, B * T, k) + 4.0 * sum(plens) * D_MODEL * D_ENC
        nb = 4 * B * case["hi"] * D_ENC + 4 * weights + 8 * B * T + 2 * B * T * _vocab(k)
        if kind == "train":
            at = 4.0 * HEAD * HEADS * LAYERS * pairs
            fl = 3 * fl + 0.5 * at
            nb += 4 * weights
        return {"bytes": nb, "flops": fl}
    if kind == "attention":
        pre, n = _attention_layout(case)
        pairs, _ = _window_pairs(pre, case["G"] if case["G"] > 1 else 0, case["T"])
        return {"bytes": n * (2 * QKV + 2 * 2 * HEADS * HEAD + 4 * HEADS + 4 * QKV), "flops": 3.5 * 4.0 * HEAD * HEADS * pairs}
    if kind == "mlp":
        M, b = case["M"], 4 if case["stream"] == "f32" else 2
        return {"bytes": M * D_MODEL * (2 + 2 * b + 2) + 2 * 3 * D_MODEL * FFN, "flops": 2.0 * M * 3 * D_MODEL * FFN}
    if kind == "encode":
        lens = _lens(case, case["n"], GRAIN)
        tx = SUP_ENCODER_CFG["model"]["encoder"]["transformer_encoder"]
        C, Fd, (left, right) = tx["layer"]["d_model"], tx["layer"]["dim_feedforward"], tx["layer"]["attn_window"]
        per_row = 4 * C * C + 3 * C * Fd
        fl = 0.0
        for t in lens:
            for l in CONVS:
                t //= l["stride"]
                fl += 2.0 * t * l["size"] * l["insize"] * l["winlen"]
            keys = sum(min(t - 1, i + right) - max(0, i - left) + 1 for i in range(t))
            fl += tx["depth"] * (2.0 * per_row * t + 4.0 * keys * C)
        return {"bytes": 4 * sum(lens) + 2 * tx["depth"] * per_row + 2 * C * sum(lens) // 12, "flops": fl}
    if kind == "loss":
        n = case["B"] * case["T"]
        return {"bytes": n * (2 * _vocab(case["k"]) * 2 + 8 + 1 + 4 + 4), "flops": 10.0 * n * _vocab(case["k"])}
    lens = _lens(case, case["W"])
    cells = sum(case["G"] * n * n for n in lens)
    return {"bytes": 9.0 * case["G"] * sum(lens), "flops": 10.0 * cells}


def tolerance(case):
    """About four times the distance from the 64-bit result, measured over the listed and some drawn cases: whole
    decoder passes 0.006 to 0.012, the 18 encoder layers 0.019, single layers 0.002 and the loss's bf16 gradient
    0.0016. The reward counts whole errors."""
    if case["kind"] == "reward":
        return "exact"
    return {"rel": {"decode": 5e-2, "prefill": 4e-2, "score": 3e-2, "train": 3.5e-2, "attention": 1e-2, "mlp": 1e-2,
                    "encode": 8e-2, "loss": 7e-3}[case["kind"]]}


# ---- the same in 64 bits --------------------------------------------------------------------------------------------
def _rms(x, w, eps=EPS):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rope(x, pos, cos, sin):
    a, b = x.chunk(2, -1)
    c, s = cos[pos][:, None], sin[pos][:, None]
    return torch.cat([a * c - b * s, a * s + b * c], -1)


class _Decoder64:
    """The decoder in float64 on the parameters and rotary tables of a model."""

    def __init__(self, m, grad=False):
        self.p = {n: v.detach().double() for n, v in m.named_parameters()}
        if grad:
            self.p = {n: v.requires_grad_() for n, v in self.p.items()}
        self.cos, self.sin = m.decoder.cos.double(), m.decoder.sin.double()

    def w(self, i, name):
        return self.p[f"decoder.layers.{i}.{name}.weight"]

    def project(self, f):
        p = self.p
        return F.gelu(f.double() @ p["projector.0.weight"].t() + p["projector.0.bias"]) @ p["projector.2.weight"].t() + \
            p["projector.2.bias"]

    def qkv(self, i, x, pos):
        h = _rms(x, self.w(i, "attn_norm")) @ self.w(i, "attn.qkv_proj").t()
        q, k, v = h.split([HEADS * HEAD, KV_HEADS * HEAD, KV_HEADS * HEAD], -1)
        q, k = q.reshape(-1, HEADS, HEAD), k.reshape(-1, KV_HEADS, HEAD)
        q = _rope(_rms(q, self.w(i, "attn.q_norm")), pos, self.cos, self.sin)
        k = _rope(_rms(k, self.w(i, "attn.k_norm")), pos, self.cos, self.sin)
        return q, k, v.reshape(-1, KV_HEADS, HEAD)

    def rest(self, i, x, o):
        x = x + o.reshape(len(x), -1) @ self.w(i, "attn.o_proj").t()
        g, u = (_rms(x, self.w(i, "mlp_norm")) @ self.w(i, "gate_up").t()).chunk(2, -1)
        return x + (F.silu(g) * u) @ self.w(i, "down").t()

    def window(self, x, keep=None, on_kv=None):
        """A causal pass over one window's rows x [n, d]; the last layer for its final `keep` rows."""
        n = len(x)
        pos = torch.arange(n, device=DEV)
        for i in range(LAYERS):
            q, k, v = self.qkv(i, x, pos)
            if on_kv is not None:
                on_kv(i, k, v)
            if i == LAYERS - 1 and keep is not None:
                x, q = x[n - keep:], q[n - keep:]
            x = self.rest(i, x, _causal64(q, k, v))
        return _rms(x, self.p["decoder.norm.weight"])

    def head(self, h):
        return h @ self.p["decoder.lm_head.weight"].t()


def _causal64(q, k, v):
    """The last len(q) rows of causal attention over the keys k; 8 query heads on 2 key heads."""
    m, n = len(q), len(k)
    rep = HEADS // KV_HEADS
    kk, vv = (t.transpose(0, 1).repeat_interleave(rep, 0) for t in (k, v))
    s = q.transpose(0, 1) @ kk.transpose(1, 2).contiguous() / math.sqrt(HEAD)
    hidden = torch.arange(n, device=DEV)[None] > torch.arange(n - m, n, device=DEV)[:, None]
    return (torch.softmax(s.masked_fill(hidden, float("-inf")), -1) @ vv).transpose(0, 1)


def _exact_decode(case, seed):
    inf, plens, cache, prefix, at, rope, tok = _decode_inputs(case, seed)
    B, G = case["B"], case["G"]
    net = _Decoder64(inf)
    x = net.p["decoder.embed.weight"][tok]
    step = 32
    rep = HEADS // KV_HEADS
    new = []

    def part(q, k, v, n):
        """Softmax sums of q [b, 8, 64] over the first n[b] rows of k, v [b, S, 2, 64]."""
        kk, vv = (t.double().permute(0, 2, 1, 3) for t in (k, v))
        s = q.reshape(len(q), KV_HEADS, rep, HEAD) @ kk.transpose(2, 3).contiguous() / math.sqrt(HEAD)
        s = s.masked_fill(torch.arange(s.shape[-1], device=DEV) >= n[:, None, None, None], float("-inf"))
        return s, vv

    for i in range(LAYERS):
        q, k, v = net.qkv(i, x, rope.long())
        new.append((k, v))
        o = torch.empty_like(q)
        for lo in range(0, B, step):
            b = torch.arange(lo, min(B, lo + step), device=DEV)
            # the cached rows before the token's own, then the token's own key and value
            s, vv = part(q[b], cache.k[i, b], cache.v[i, b], at[b].long())
            own, _ = part(q[b], k[b][:, None], v[b][:, None], torch.ones(len(b), device=DEV))
            ss, vs = [s, own], [vv, v[b][:, None].permute(0, 2, 1, 3)]
            if G > 1:
                pl = torch.tensor(plens, device=DEV)[b // G] + 1
                s, vv = part(q[b], prefix.k[i, b // G], prefix.v[i, b // G], pl)
                ss.append(s)
                vs.append(vv)
            o[b] = (torch.softmax(torch.cat(ss, -1), -1) @ torch.cat(vs, 2)).reshape(len(b), HEADS, HEAD)
        x = net.rest(i, x, o)
    h = _rms(x, net.p["decoder.norm.weight"])
    if G == 1 and case["lo"] != case["hi"]:
        return [h, net.head(h)]
    return [h, net.head(h), *(torch.stack(t) for t in zip(*new))]


def _exact_prefill(case, seed):
    s = _prepare_prefill(case, seed)
    eng = s["eng"]
    net = _Decoder64(eng.model)
    c = eng.cache if eng.prefix_cache is None else eng.prefix_cache
    K, V = (torch.zeros(c.k.shape, dtype=torch.float64, device=DEV) for _ in range(2))
    lp = []
    for w, f in enumerate(s["one"].split(s["plens"])):
        def put(i, k, v):
            K[i, w, :len(k)] = k
            V[i, w, :len(v)] = v

        x = torch.cat([net.project(f), net.p["decoder.embed.weight"][BOS][None]])
        z = net.head(net.window(x, 1, put))[0] + eng.bias.double()
        lp += [torch.log_softmax(z, -1).max()] * case["G"]
    return [None, torch.stack(lp), K, V]


def _logits64(net, s, b):
    x = torch.cat([net.project(s["frames"][b, :int(s["plens"][b])]), net.p["decoder.embed.weight"][s["tokens"][b]]])
    return net.head(net.window(x, s["tokens"].shape[1]))


def _exact_score(case, seed):
    s = _prepare_score(case, seed)
    net = _Decoder64(s["model"])
    return [torch.stack([_logits64(net, s, b) for b in range(len(s["tokens"]))])]


def _exact_train(case, seed):
    s = _prepare_train(case, seed)
    net = _Decoder64(s["model"], grad=True)
    B = len(s["tokens"])
    logits = []
    for b in range(B):
        z = _logits64(net, s, b)
        lp = torch.log_softmax(z, -1).gather(-1, s["targets"][b, :, None])[:, 0]
        # the ratio's value is 1: the old log-probs are this policy's
        d = ((lp - lp.detach()) * s["mask"][b]).sum() / s["bases"][b]
        (-torch.exp(d) * s["adv"][b].double() / B).backward()
        logits.append(z.detach())
    grads = [net.p[n].grad for n, _ in s["model"].named_parameters()]
    return [torch.stack(logits), torch.cat([g.reshape(-1) for g in grads])]


def _exact_attention(case, seed):
    s = _prepare_attention(case, seed)
    pre, n = _attention_layout(case)
    q, k, v = (s[t].double().requires_grad_() for t in ("q", "k", "v"))
    lse = torch.empty(n, HEADS, dtype=torch.float64, device=DEV)
    o = torch.empty(n, HEADS, HEAD, dtype=torch.float64, device=DEV)
    G, T = (case["G"], case["T"]) if case["G"] > 1 else (0, 0)
    n_pre, at = sum(pre), 0
    for w, p in enumerate(pre):
        own = torch.arange(at, at + p, device=DEV)
        spans = [(own, own)]
        for g in range(G):
            r = torch.arange(T, device=DEV) + n_pre + (w * G + g) * T
            spans.append((r, torch.cat([own, r])))
        for rq, rk in spans:
            part = _causal64(q[rq], k[rk], v[rk])
            part.backward(s["dout"][rq].double())
            o[rq] = part.detach()
            with torch.no_grad():
                kk = k[rk].transpose(0, 1).repeat_interleave(HEADS // KV_HEADS, 0)
                sc = q[rq].transpose(0, 1) @ kk.transpose(1, 2).contiguous() / math.sqrt(HEAD)
                hid = torch.arange(len(rk), device=DEV)[None] > torch.arange(len(rk) - len(rq), len(rk), device=DEV)[:, None]
                lse[rq] = torch.logsumexp(sc.masked_fill(hid, float("-inf")), -1).t() / math.log(2)
        at += p
    return [o, lse, q.grad, k.grad, v.grad]


def _exact_mlp(case, seed):
    s = {n: t.double() for n, t in _prepare_mlp(case, seed).items()}
    g, u = (s["h"] @ s["gate_up"].t()).chunk(2, -1)
    y = s["x"] + (F.silu(g) * u) @ s["down"].t()
    return [y, _rms(y, s["norm"])]


def _exact_encode(case, seed):
    s = _prepare_encode(case, seed)
    p = {n: v.double() for n, v in s["weights"].items()}
    tx = SUP_ENCODER_CFG["model"]["encoder"]["transformer_encoder"]
    C, H, alpha = tx["layer"]["d_model"], tx["layer"]["nhead"], tx["layer"]["deepnorm_alpha"]
    left, right = tx["layer"]["attn_window"]
    cos, sin = s["enc"].cos.double(), s["enc"].sin.double()
    out = []
    for sig in s["signal"].double().split(s["lens"]):
        x = sig[:, None]  # [samples, channels]
        for i, l in enumerate(CONVS):
            w = p[f"conv.{i}.conv.weight"].permute(0, 2, 1).reshape(l["size"], -1)  # taps, then channels
            x = F.pad(x, (0, 0, l["padding"], l["padding"])).unfold(0, l["winlen"], l["stride"])
            x = F.silu(x.transpose(1, 2).reshape(len(x), -1) @ w.t() + p[f"conv.{i}.conv.bias"])
        n = len(x)
        pos = torch.arange(n, device=DEV)
        rel = pos[None] - pos[:, None]
        hidden = (rel < -left) | (rel > right)
        for j in range(tx["depth"]):
            q = f"transformer_encoder.{j}."
            a, b, c = (x @ p[q + "self_attn.Wqkv.weight"].t()).view(n, 3, H, C // H).unbind(1)
            a, b = _rope(a, pos, cos, sin), _rope(b, pos, cos, sin)
            sc = a.transpose(0, 1) @ b.permute(1, 2, 0).contiguous() / math.sqrt(C // H)
            o = torch.softmax(sc.masked_fill(hidden, float("-inf")), -1) @ c.transpose(0, 1)
            o = o.transpose(0, 1).reshape(n, C) @ p[q + "self_attn.out_proj.weight"].t() + p[q + "self_attn.out_proj.bias"]
            x = _rms(o + alpha * x, p[q + "norm1.weight"], 1e-5)
            y, g = (x @ p[q + "ff.fc1.weight"].t()).chunk(2, -1)
            x = _rms((F.silu(g) * y) @ p[q + "ff.fc2.weight"].t() + alpha * x, p[q + "norm2.weight"], 1e-5)
        out.append(x)
    return [torch.cat(out)]


def _exact_loss(case, seed):
    s = _prepare_loss(case, seed)
    z = s["z"].detach().double().requires_grad_()
    lp = torch.log_softmax(z, -1).gather(-1, s["targets"][..., None])[..., 0]
    r = torch.exp(((lp - s["old"].double()) * s["mask"]).sum(1) / s["bases"].double())
    a = s["adv"].double()
    loss = -torch.minimum(r * a, r.clamp(1 - 4e-4, 1 + 4e-4) * a).mean()
    loss.backward()
    return [loss.detach(), r.detach(), lp.detach(), z.grad]


def _exact_reward(case, seed):
    """Edit distance by anti-diagonals, every call at once. Of a cell's predecessors the first best one of diagonal,
    deletion and insertion is taken; errors are counted at scored label bases."""
    s = _prepare_reward(case, seed)
    calls, labels = s["raw"]
    G = s["G"]
    n = torch.tensor([len(c) for c in calls], device=DEV)
    m = torch.tensor([len(labels[i // G]) for i in range(len(calls))], device=DEV)
    C, wide, tall = len(calls), int(m.max()), int(n.max())
    call = torch.full((C, tall + 1), 8, device=DEV)
    ref = torch.full((C, wide + 1), 9, device=DEV)
    sc = torch.zeros((C, wide + 1), dtype=torch.int64, device=DEV)
    for i, c in enumerate(calls):
        call[i, :len(c)] = torch.from_numpy(c).to(DEV)
        ref[i, :len(labels[i // G])] = torch.from_numpy(labels[i // G]).to(DEV)
        sc[i, :len(labels[i // G])] = torch.from_numpy(s["weights"][i // G] > 0).to(DEV)
    at = torch.arange(wide + 1, device=DEV)
    prev = (at - 1).clamp(min=0)
    zero = torch.zeros((C, wide + 1), dtype=torch.int64, device=DEV)
    d1, c1, d2, c2 = zero, zero, zero, zero
    dist, errs = torch.zeros(C, dtype=torch.int64, device=DEV), torch.zeros(C, dtype=torch.int64, device=DEV)
    rows = torch.arange(C, device=DEV)
    sp = sc[:, prev]
    for k in range(wide + tall + 1):
        j = k - at
        mis = (ref[:, prev] != call[:, (j - 1).clamp(0, tall)]).long()
        dd, du, dl = d2[:, prev] + mis, d1[:, prev] + 1, d1 + 1
        d = torch.minimum(torch.minimum(dd, du), dl)
        e = torch.where(dd == d, c2[:, prev] + mis * sp, torch.where(du == d, c1[:, prev] + sp, c1 + sp))
        d = torch.where(at == 0, j, torch.where(j == 0, at, d))
        e = torch.where(at == 0, c1 + sc[:, :1] if k else zero, torch.where(j == 0, c1[:, prev] + sp, e))
        d2, c2, d1, c1 = d1, c1, d, e
        end = m + n == k
        dist = torch.where(end, d[rows, m], dist)
        errs = torch.where(end, e[rows, m], errs)
    return [1 - errs.double() / torch.maximum(m, n).double(), dist.to(torch.int32), errs.to(torch.int32)]


_EXACT = {"decode": _exact_decode, "prefill": _exact_prefill, "score": _exact_score, "train": _exact_train,
          "attention": _exact_attention, "mlp": _exact_mlp, "encode": _exact_encode, "loss": _exact_loss,
          "reward": _exact_reward}


def exact(case, seed):
    if case["kind"] in ("train", "attention"):
        return _EXACT[case["kind"]](case, int(seed))
    with torch.no_grad() if case["kind"] != "loss" else torch.enable_grad():
        return _EXACT[case["kind"]](case, int(seed))
