"""The performance cases of the paged attention path: what each stands for,
its inputs, one pass through the public entry points, the work a pass cannot
do without, and its float64 statement in plain torch.

Kinds
  block    the whole decode attention block (``attention_decode``): input
           norm, QKV projection, RoPE, attention, cache write, output
           projection
  decode   the decode attention core over a paged cache with its fused cache
           write (``paged_decode_core``)
  window   the decode core of several sliding-window layers, captured once in
           a HIP graph and replayed, as a serving loop runs short layers
  prefill  one chunk of one sequence over its paged context
           (``segmented_attention``)
  mixed    one step of decode rows and prefill sequences over one cache,
           captured in a HIP graph (``mixed_batch_attention``)
  qkv      row norm, projection, RoPE and cache write of a prefill chunk
           (``qkv_proj``)
  dense    dense attention without a cache (``flash_attention``)

Conventions: Q, K, V and hidden states ~ N(0, 1); physical blocks are a
random permutation (block 0 is the null block), table tails are -1 and the
table width makes the context a multiple of 128; per-row lengths are spread
over their range, odd ones among them, and belong to the case, every value
to the seed.
"""
import math
import os
import random
import sys

import torch

_PKG = os.path.join(os.getcwd(), "vllm-neuron_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from vllm_neuron_amd.functional import (  # noqa: E402
    attention_decode,
    flash_attention,
    mixed_batch_attention,
    qkv_proj,
    segmented_attention,
)
from vllm_neuron_amd.functional.attention.attention_decode import paged_decode_core  # noqa: E402
from vllm_neuron_amd.utils.common_types import NormType  # noqa: E402

BF = torch.bfloat16
FP8 = torch.float8_e4m3fn
DEV = "cuda:0"
WINDOW = 128  # sliding window of the GPT-OSS layers

# Head geometries of the repository's workload table.
SHAPES = {
    "llama3_1b": dict(heads=32, kv=8, d=64, bs=16, sink=False, fp8=False),
    "llama3_8b": dict(heads=32, kv=8, d=128, bs=32, sink=False, fp8=False),
    "gptoss": dict(heads=64, kv=8, d=64, bs=32, sink=True, fp8=False),
    "fp8_48q": dict(heads=48, kv=8, d=128, bs=64, sink=False, fp8=True),
}


def listed():
    return [
        # The smallest call: the decode attention block of a small model at a
        # small batch, issued eagerly; launches and host time count.
        dict(name="block_1b_b4", kind="block", shape="llama3_1b", batch=4, hidden=2048, lo=128, hi=1024),
        # The serving step of an 8B model's layer at a full batch: streams the
        # cache from HBM.
        dict(name="decode_8b_b64", kind="decode", shape="llama3_8b", batch=64, lo=512, hi=8192),
        # The full-attention layer of GPT-OSS-120B with sinks (d = 64, group 8).
        dict(name="decode_gptoss_b32", kind="decode", shape="gptoss", batch=32, lo=1024, hi=16384),
        # Long contexts in an FP8 cache with per-head scales, few rows.
        dict(name="decode_fp8_32k", kind="decode", shape="fp8_48q", batch=16, lo=16384, hi=32768),
        # GPT-OSS sliding-window layers of a captured decode step: short
        # launches, latency bound.
        dict(name="decode_window_b32", kind="window", shape="gptoss", batch=32, layers=8, lo=1024, hi=16384),
        # An ordinary prefill chunk with ragged length after some context.
        dict(name="prefill_8b_chunk", kind="prefill", shape="llama3_8b", new=777, prior=1536, window=0),
        # GPT-OSS prefill chunk, full-attention layer with sinks.
        dict(name="prefill_gptoss_full", kind="prefill", shape="gptoss", new=2048, prior=4096, window=0),
        # The same chunk in a sliding-window layer (every other layer).
        dict(name="prefill_gptoss_window", kind="prefill", shape="gptoss", new=2048, prior=4096, window=WINDOW),
        # The largest: a chunk after a long prior in an FP8 cache.
        dict(name="prefill_fp8_16k", kind="prefill", shape="fp8_48q", new=2048, prior=16384, window=0),
        # A continuous-batching step: decode rows and four prefill chunks.
        dict(name="mixed_8b", kind="mixed", shape="llama3_8b", batch=60, lo=1024, hi=8192, seqs=4, new=512,
             prior_hi=4096),
        # QKV projection of a prefill chunk with the packed FP8 cache write.
        dict(name="qkv_8b_chunk", kind="qkv", shape="fp8_48q", tokens=2048, hidden=4096),
        # Vision-encoder attention: dense, not causal, a head dim that is
        # neither of the compiled widths.
        dict(name="dense_vit_d80", kind="dense", heads=16, kv=16, d=80, tokens=4096, causal=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["block", "decode", "window", "prefill", "prefill", "mixed", "qkv", "dense"])
    if kind == "block":
        shape = rng.choice(["llama3_1b", "llama3_8b"])
        return dict(kind=kind, shape=shape, batch=_log_int(rng, 1, 32), hidden=rng.choice([2048, 4096]),
                    lo=64, hi=_log_int(rng, 128, 4096))
    if kind == "decode":
        shape = rng.choice(sorted(SHAPES))
        s = SHAPES[shape]
        batch = _log_int(rng, 1, 64)
        most = int(1.0e9 / (0.6 * batch * s["kv"] * s["d"] * 2 * (1 if s["fp8"] else 2)))
        hi = _log_int(rng, 128, min(32768, most))
        return dict(kind=kind, shape=shape, batch=batch, lo=max(1, hi // rng.choice([2, 16])), hi=hi)
    if kind == "window":
        return dict(kind=kind, shape="gptoss", batch=_log_int(rng, 1, 64), layers=rng.randint(4, 12), lo=64,
                    hi=_log_int(rng, 256, 16384))
    if kind == "prefill":
        shape = rng.choice(sorted(SHAPES))
        s = SHAPES[shape]
        window = WINDOW if shape == "gptoss" and rng.random() < 0.5 else 0
        new = _log_int(rng, 64, 2048)
        prior = 0 if rng.random() < 0.2 else _log_int(rng, 64, 16384) // s["bs"] * s["bs"]
        return dict(kind=kind, shape=shape, new=new, prior=prior, window=window)
    if kind == "mixed":
        return dict(kind=kind, shape="llama3_8b", batch=rng.randint(4, 60), lo=256, hi=_log_int(rng, 512, 8192),
                    seqs=rng.randint(1, 4), new=_log_int(rng, 64, 512), prior_hi=_log_int(rng, 64, 4096))
    if kind == "qkv":
        return dict(kind=kind, shape=rng.choice(["fp8_48q", "llama3_8b", "gptoss"]), tokens=_log_int(rng, 64, 2048),
                    hidden=rng.choice([2880, 4096]))
    heads, kv = rng.choice([(16, 16), (32, 8)])
    return dict(kind=kind, heads=heads, kv=kv, d=rng.choice([64, 80, 128]), tokens=_log_int(rng, 256, 4096),
                causal=rng.random() < 0.5)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _lens(case, n, lo, hi, salt=0):
    """Row lengths of a case: spread over [lo, hi], the same for every seed."""
    r = random.Random("%d %d %d %d" % (n, lo, hi, salt))
    return [r.randint(min(lo, hi), hi) for _ in range(n)]


class _Gen:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def normal(self, *shape, scale=1.0):
        x = torch.randn(shape, generator=self.g, device=DEV, dtype=BF)
        return x if scale == 1.0 else x.mul_(scale)

    def uniform(self, n, lo, hi):
        return torch.rand(n, generator=self.g, device=DEV) * (hi - lo) + lo

    def tables(self, lens, bs, first=1):
        """-1 padded int32 tables of rows of ``lens`` tokens over a random
        permutation of the blocks from ``first`` on; the block count."""
        per = [(n + bs - 1) // bs for n in lens]
        step = max(1, 128 // bs)
        width = (max(per) + step - 1) // step * step
        perm = torch.randperm(sum(per), generator=self.g, device=DEV).to(torch.int32) + first
        t = torch.full((len(lens), width), -1, dtype=torch.int32, device=DEV)
        at = 0
        for i, n in enumerate(per):
            t[i, :n] = perm[at:at + n]
            at += n
        return t, first + sum(per)

    def cache(self, nb, s):
        """K or V cache [nb, kv, bs, d] and its per-head dequant scale (FP8)."""
        x = self.normal(nb, s["kv"], s["bs"], s["d"])
        if not s["fp8"]:
            return x, None
        scale = self.uniform(s["kv"], 0.01, 0.1)
        return _to_fp8(x, 1.0 / scale), scale


def _to_fp8(x, inv):
    out = torch.empty(x.shape, dtype=FP8, device=x.device)
    step = max(1, (1 << 26) // max(1, x[0].numel()))
    for i in range(0, x.shape[0], step):
        out[i:i + step] = (x[i:i + step].float() * inv.view(1, -1, 1, 1)).clamp_(-448, 448).to(FP8)
    return out


def _slots(table, pos, bs):
    """Write slot of position ``pos[r]`` of each table row."""
    p = torch.as_tensor(pos, dtype=torch.int64, device=DEV)
    return table.gather(1, (p // bs).view(-1, 1)).view(-1).long() * bs + p % bs


def _decode_inputs(case, s, gen, lens):
    t, nb = gen.tables(lens, s["bs"])
    kc, kd = gen.cache(nb, s)
    vc, vd = gen.cache(nb, s)
    B = len(lens)
    pos = [n - 1 for n in lens]
    x = dict(q=gen.normal(B, 1, s["heads"], s["d"]), k=gen.normal(B, 1, s["kv"], s["d"]),
             v=gen.normal(B, 1, s["kv"], s["d"]), K=kc, V=vc, table=t, kd=kd, vd=vd, slots=_slots(t, pos, s["bs"]),
             pos=torch.tensor(pos, dtype=torch.float32, device=DEV).view(B, 1), start=None,
             sink=gen.uniform(s["heads"], -1.0, 1.0) if s["sink"] else None)
    return x


def _window_inputs(case, s, gen, lens):
    """Sliding-window layer: the table holds the window's blocks alone and the
    positions are in its frame, as the runner hands them over."""
    bs = s["bs"]
    width = (WINDOW // bs + 1 + 128 // bs - 1) // (128 // bs) * (128 // bs)
    pos, start, have = [], [], []
    for n in lens:
        off = max(0, (n - 1) // bs - width + 1) * bs
        pos.append(n - 1 - off)
        start.append(max(0, n - 1 - off - WINDOW + 1))
        have.append(n - off)
    x = _decode_inputs(case, s, gen, have)
    t = torch.full((len(lens), width), -1, dtype=torch.int32, device=DEV)
    t[:, :min(width, x["table"].shape[1])] = x["table"][:, :width]
    x.update(table=t, start=torch.tensor(start, dtype=torch.float32, device=DEV).view(-1, 1))
    return x


def _prefill_inputs(case, s, gen):
    L = case["prior"] + case["new"]
    t, nb = gen.tables([L], s["bs"])
    kc, kd = gen.cache(nb, s)
    vc, vd = gen.cache(nb, s)
    return dict(q=gen.normal(s["heads"], case["new"], s["d"]), K=kc, V=vc, table=t, kd=kd, vd=vd,
                prior=torch.tensor([[case["prior"]]], dtype=torch.int32, device=DEV),
                sink=gen.uniform(s["heads"], -1.0, 1.0) if s["sink"] else None)


def _mixed_lens(case, s):
    prior = [p // s["bs"] * s["bs"] for p in _lens(case, case["seqs"], 0, case["prior_hi"], 1)]
    return _lens(case, case["batch"], case["lo"], case["hi"]), prior


def _mixed_inputs(case, s, gen):
    rows, prior = _mixed_lens(case, s)
    bs, P, S = s["bs"], case["seqs"], case["new"]
    td, nb = gen.tables(rows, bs)
    tp, nb = gen.tables([p + S for p in prior], bs, nb)
    kc, _ = gen.cache(nb, s)
    vc, _ = gen.cache(nb, s)
    B, T = len(rows), P * S
    where = torch.cat([torch.arange(p, p + S, device=DEV) for p in prior])
    seq = torch.arange(P, device=DEV).repeat_interleave(S)
    pos = [n - 1 for n in rows]
    return dict(q=gen.normal(B, 1, s["heads"], s["d"]), k=gen.normal(B, 1, s["kv"], s["d"]),
                v=gen.normal(B, 1, s["kv"], s["d"]), K=kc, V=vc, table=td, slots=_slots(td, pos, bs).view(B, 1),
                pos=torch.tensor(pos, dtype=torch.float32, device=DEV).view(B, 1),
                qp=gen.normal(T, s["heads"], s["d"]), kp=gen.normal(T, s["kv"], s["d"]),
                vp=gen.normal(T, s["kv"], s["d"]), tp=tp,
                sp=tp[seq, where // bs].long() * bs + where % bs,
                cu=torch.arange(P + 1, dtype=torch.int32, device=DEV) * S,
                prior=torch.tensor(prior, dtype=torch.int32, device=DEV))


def _rope(tokens, d, first):
    """cos, sin [tokens, d/2] of consecutive or given positions."""
    p = first + torch.arange(tokens, device=DEV) if isinstance(first, int) else first
    a = p.double().view(-1, 1) * 10000.0 ** (-torch.arange(0, d, 2, device=DEV).double() / d)
    return a.cos().float(), a.sin().float()


def _block_inputs(case, s, gen):
    H, d = case["hidden"], s["d"]
    lens = _lens(case, case["batch"], case["lo"], case["hi"])
    x = _decode_inputs(case, s, gen, lens)
    fused = (s["heads"] + 2 * s["kv"]) * d
    c, n = _rope(len(lens), d, x["pos"].view(-1))
    x.update(X=gen.normal(len(lens), 1, H), Wqkv=gen.normal(H, fused, scale=H ** -0.5),
             Wout=gen.normal(s["heads"] * d, H, scale=(s["heads"] * d) ** -0.5),
             gamma=gen.uniform(H, 0.5, 1.5).to(BF),
             # the model keeps its tables in bf16 precision
             cos=c.to(BF).float().t().reshape(d // 2, len(lens), 1).contiguous(),
             sin=n.to(BF).float().t().reshape(d // 2, len(lens), 1).contiguous())
    return x


def _qkv_inputs(case, s, gen):
    H, T, d, bs = case["hidden"], case["tokens"], s["d"], s["bs"]
    t, nb = gen.tables([T], bs)
    p = torch.arange(T, device=DEV)
    c, n = _rope(T, d, 0)
    shape = (nb, s["kv"], bs, d)
    x = dict(X=gen.normal(1, T, H), W=gen.normal(H, (s["heads"] + 2 * s["kv"]) * d, scale=H ** -0.5),
             gamma=gen.uniform(H, 0.5, 1.5).to(BF), cos=torch.cat([c, c], -1).view(1, T, d),
             sin=torch.cat([n, n], -1).view(1, T, d), slots=(t[0, p // bs].long() * bs + p % bs).view(1, T))
    if s["fp8"]:
        x.update(K=torch.zeros((nb, s["kv"], bs // 2, d, 2), dtype=FP8, device=DEV),
                 V=torch.zeros(shape, dtype=FP8, device=DEV), ks=gen.uniform(1, 0.01, 0.1).view(1, 1),
                 vs=gen.uniform(1, 0.01, 0.1).view(1, 1))
    else:
        x.update(K=torch.zeros(shape, dtype=BF, device=DEV), V=torch.zeros(shape, dtype=BF, device=DEV))
    return x


def _dense_inputs(case, gen):
    S, d = case["tokens"], case["d"]
    return dict(q=gen.normal(case["heads"], S, d), k=gen.normal(case["kv"], d, S), v=gen.normal(case["kv"], S, d))


def _inputs(case, seed):
    s, gen, kind = SHAPES.get(case.get("shape")), _Gen(seed), case["kind"]
    if kind == "decode":
        return _decode_inputs(case, s, gen, _lens(case, case["batch"], case["lo"], case["hi"]))
    if kind == "window":
        lens = _lens(case, case["batch"], case["lo"], case["hi"])
        return [_window_inputs(case, s, gen, lens) for _ in range(case["layers"])]
    if kind == "dense":
        return _dense_inputs(case, gen)
    return {"block": _block_inputs, "prefill": _prefill_inputs, "mixed": _mixed_inputs,
            "qkv": _qkv_inputs}[kind](case, s, gen)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _decode(x, s):
    kw = {}
    if s["fp8"]:
        kw = dict(k_scale=x["kq"], v_scale=x["vq"], k_dequant_scale=x["kd"], v_dequant_scale=x["vd"])
    return paged_decode_core(x["q"], x["k"], x["v"], x["K"], x["V"], x["table"], block_len=s["bs"],
                             S_ctx=x["table"].shape[1] * s["bs"], pos_ids=x["pos"], swa_start_pos_ids=x["start"],
                             sink=x["sink"], softmax_scale=s["d"] ** -0.5, write_slots=x["slots"],
                             write_slots_private=True, **kw)


def _block(x, s):
    return attention_decode(
        X=x["X"], rmsnorm_X_enabled=True, rmsnorm_X_eps=1e-5, rmsnorm_X_gamma=x["gamma"], W_qkv=x["Wqkv"],
        cos=x["cos"], sin=x["sin"], active_blocks_table=x["table"], K_cache=x["K"], V_cache=x["V"], pos_ids=x["pos"],
        update_cache=True, kv_cache_update_idx=x["slots"], kv_cache_update_private=True, W_out=x["Wout"])


def _prefill(x, s, case):
    return segmented_attention(x["q"], x["K"], x["V"], x["table"], x["prior"], s["bs"], 0,
                               sliding_window=case["window"] or None, sink=x["sink"], k_dequant_scale=x["kd"],
                               v_dequant_scale=x["vd"])


def _mixed(x, s, case):
    return mixed_batch_attention(
        x["K"], x["V"], q_decode=x["q"], k_decode=x["k"], v_decode=x["v"], decode_block_table=x["table"],
        decode_pos_ids=x["pos"], decode_slots=x["slots"], q_prefill=x["qp"], k_prefill=x["kp"], v_prefill=x["vp"],
        prefill_slots=x["sp"], prefill_cu_seqlens=x["cu"], prefill_prior=x["prior"], prefill_block_table=x["tp"],
        max_seqlen_q=case["new"])


def _qkv(x, s):
    kw = dict(k_scale=x["ks"], v_scale=x["vs"], fp8_packed=True) if s["fp8"] else {}
    return qkv_proj(x["X"], x["W"], norm_weights=x["gamma"], norm_type=NormType.RMS_NORM, eps=1e-5, d_head=s["d"],
                    cos_cache=x["cos"], sin_cache=x["sin"], num_q_heads=s["heads"], num_kv_heads=s["kv"],
                    k_cache=x["K"], v_cache=x["V"], use_block_kv=True, block_size=s["bs"], slot_mapping=x["slots"],
                    **kw)


def _captured(call):
    """The call in a HIP graph, and its (static) outputs."""
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    return graph, out


def prepare(case, seed):
    s, kind, x = SHAPES.get(case.get("shape")), case["kind"], _inputs(case, seed)
    if kind == "decode" and s["fp8"]:
        x.update(kq=1.0 / x["kd"], vq=1.0 / x["vd"])
    state = dict(case=case, s=s, kind=kind, x=x)
    if kind == "window":
        state["graph"], state["out"] = _captured(lambda: [_decode(y, s) for y in x])
    if kind == "mixed":
        state["graph"], state["out"] = _captured(lambda: _mixed(x, s, case))
    return state


def run(state):
    case, s, kind, x = state["case"], state["s"], state["kind"], state["x"]
    if kind == "block":
        return [_block(x, s), x["K"], x["V"]]
    if kind == "decode":
        return [_decode(x, s), x["K"], x["V"]]
    if kind == "window":
        state["graph"].replay()
        return [[o, y["K"], y["V"]] for o, y in zip(state["out"], x)]
    if kind == "prefill":
        return _prefill(x, s, case)
    if kind == "mixed":
        state["graph"].replay()
        return [state["out"][0], state["out"][1], x["K"], x["V"]]
    if kind == "qkv":
        return list(_qkv(x, s))
    return flash_attention(x["q"], x["k"], x["v"], causal_mask=case["causal"])


# ---------------------------------------------------------------------------
# the work of a pass
# ---------------------------------------------------------------------------
def _decode_work(s, lens):
    """Attended K/V once, Q in, O out, the new rows in and into the cache, the
    table entries of the attended blocks; 4 d flops per query head and key."""
    e, B = (1 if s["fp8"] else 2), len(lens)
    n = sum(lens)
    kv = n * s["kv"] * s["d"] * 2 * e
    rows = B * s["heads"] * s["d"] * 4 + B * s["kv"] * s["d"] * 2 * (2 + e)
    return dict(bytes=kv + rows + 4 * sum((k + s["bs"] - 1) // s["bs"] for k in lens),
                flops=4 * s["heads"] * s["d"] * n)


def _visible(new, prior, window):
    if not window:
        return new * prior + new * (new + 1) // 2
    return sum(min(prior + i + 1, window) for i in range(new))


def _prefill_work(s, new, prior, window):
    e = 1 if s["fp8"] else 2
    keys = min(prior, window - 1) + new if window else prior + new
    return dict(bytes=keys * s["kv"] * s["d"] * 2 * e + new * s["heads"] * s["d"] * 4,
                flops=4 * s["heads"] * s["d"] * _visible(new, prior, window))


def _add(*works):
    return dict(bytes=sum(w["bytes"] for w in works), flops=sum(w["flops"] for w in works))


def work(case):
    s, kind = SHAPES.get(case.get("shape")), case["kind"]
    if kind in ("decode", "block", "window"):
        lens = _lens(case, case["batch"], case["lo"], case["hi"])
    if kind == "decode":
        return _decode_work(s, lens)
    if kind == "window":
        w = _decode_work(s, [min(n, WINDOW) for n in lens])
        return {k: v * case["layers"] for k, v in w.items()}
    if kind == "block":
        H, I, B = case["hidden"], (s["heads"] + 2 * s["kv"]) * s["d"], len(lens)
        kv = dict(bytes=sum(lens) * s["kv"] * s["d"] * 4, flops=4 * s["heads"] * s["d"] * sum(lens))
        o = s["heads"] * s["d"]
        return _add(kv, dict(bytes=2 * (H * I + o * H + 2 * B * H), flops=2 * B * (H * I + o * H)))
    if kind == "prefill":
        return _prefill_work(s, case["new"], case["prior"], case["window"])
    if kind == "mixed":
        rows, prior = _mixed_lens(case, s)
        write = dict(bytes=case["seqs"] * case["new"] * s["kv"] * s["d"] * 8, flops=0)
        return _add(_decode_work(s, rows), write, *[_prefill_work(s, case["new"], p, 0) for p in prior])
    if kind == "qkv":
        H, T, I = case["hidden"], case["tokens"], (s["heads"] + 2 * s["kv"]) * s["d"]
        e = 1 if s["fp8"] else 2
        return dict(bytes=2 * (T * H + H * I + T * s["heads"] * s["d"]) + T * s["kv"] * s["d"] * 2 * e + T * s["d"] * 8,
                    flops=2 * T * H * I)
    S = case["tokens"]
    return dict(bytes=S * case["d"] * (case["heads"] * 4 + case["kv"] * 4),
                flops=4 * case["heads"] * case["d"] * (S * (S + 1) // 2 if case["causal"] else S * S))


def tolerance(case):
    # bf16 outputs from bf16 inputs: the probabilities, the outputs and, in
    # the blocks, the projected rows are rounded to bf16 (relative 2^-9 each).
    # The kernels stand 2e-3 to 3.4e-3 from float64 (2-norm; 4.4e-3 for the
    # whole block with its two projections); another correct order of the
    # sums or roundings stands as far off on another side: about four times
    # the single-kernel distance is allowed.
    return {"rel": 1e-2, "max": 0.1}


# ---------------------------------------------------------------------------
# float64 statements
# ---------------------------------------------------------------------------
def _rows64(cache, table, n):
    """The first ``n`` tokens of a table row: [kv, n, d] float64."""
    bs = cache.shape[2]
    c = cache[table[:(n + bs - 1) // bs].long()].double()
    return c.permute(1, 0, 2, 3).reshape(cache.shape[1], -1, cache.shape[3])[:, :n]


def _attend64(q, K, V, scale, sink=None, visible=None):
    """q [kv, G, n, d] over K, V [kv, L, d]; ``visible`` [n, L] or None."""
    kv, G, n, d = q.shape
    sc = (q.reshape(kv, G * n, d) @ K.transpose(1, 2).contiguous()).view(kv, G, n, -1) * scale
    if visible is not None:
        sc.masked_fill_(~visible, -math.inf)
    top = sc.amax(-1, keepdim=True)
    if sink is not None:
        b = sink.double().view(kv, G, 1, 1)
        top = torch.maximum(top, b)
    p = sc.sub_(top).exp_()
    den = p.sum(-1, keepdim=True)
    if sink is not None:
        den = den + (b - top).exp()
    return (p.view(kv, G * n, -1) @ V).view(kv, G, n, d) / den


def _decode64(x, s, lens, starts=None):
    B, G = len(lens), s["heads"] // s["kv"]
    out = []
    ka, va = x["k"].double(), x["v"].double()
    if s["fp8"]:  # the active rows are read as the cache holds them
        f8 = lambda t, sc: _to_fp8(t.transpose(1, 2), 1.0 / sc).double().transpose(1, 2)
        ka, va = f8(x["k"], x["kd"]), f8(x["v"], x["vd"])
    for b, n in enumerate(lens):
        lo = 0 if starts is None else starts[b]
        K = torch.cat([_rows64(x["K"], x["table"][b], n - 1)[:, lo:], ka[b].transpose(0, 1)], 1)
        V = torch.cat([_rows64(x["V"], x["table"][b], n - 1)[:, lo:], va[b].transpose(0, 1)], 1)
        if s["fp8"]:
            K, V = K * x["kd"].double().view(-1, 1, 1), V * x["vd"].double().view(-1, 1, 1)
        q = x["q"][b].double().view(s["kv"], G, 1, s["d"])
        out.append(_attend64(q, K, V, s["d"] ** -0.5, x["sink"]).view(1, s["heads"], s["d"]))
    return torch.stack(out)


def _written64(cache, slots, rows):
    """The cache in float64 with ``rows`` [T, kv, d] at ``slots``."""
    nb, kv, bs, d = cache.shape
    c = cache.double()
    c[slots // bs, :, slots % bs] = rows.double()
    return c


def _decode_exact(x, s, lens, starts=None):
    if s["fp8"]:  # whole codes: no float64 value
        return [_decode64(x, s, lens, starts), None, None]
    return [_decode64(x, s, lens, starts), _written64(x["K"], x["slots"], x["k"][:, 0]),
            _written64(x["V"], x["slots"], x["v"][:, 0])]


def _rotate64(x, cos, sin):
    a, b = x.chunk(2, -1)
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _project64(X, W, gamma, s, cos, sin):
    """Norm, projection and RoPE in float64: q, k, v [T, heads, d]."""
    h = X.double().reshape(-1, X.shape[-1])
    h = h * torch.rsqrt(h.pow(2).mean(-1, keepdim=True) + 1e-5) * gamma.double()
    y = (h @ W.double()).view(h.shape[0], -1, s["d"])
    q, k, v = y.split([s["heads"], s["kv"], s["kv"]], 1)
    c, n = cos.double().unsqueeze(1), sin.double().unsqueeze(1)
    return _rotate64(q, c, n), _rotate64(k, c, n), v


def _prefill64(q, K, V, L, s, case_new, prior, window, sink, kd=None, vd=None):
    """q [heads, new, d] over K, V [kv, L, d]: [heads, new, d]."""
    G = s["heads"] // s["kv"]
    i = torch.arange(case_new, device=DEV).view(-1, 1) + prior
    j = torch.arange(L, device=DEV).view(1, -1)
    see = (j <= i) & (j > i - window) if window else j <= i
    out = []
    for h in range(s["kv"]):
        k1, v1 = K[h:h + 1], V[h:h + 1]
        if kd is not None:
            k1, v1 = k1 * kd[h].double(), v1 * vd[h].double()
        out.append(_attend64(q[h * G:(h + 1) * G].double().unsqueeze(0), k1, v1, s["d"] ** -0.5,
                             None if sink is None else sink[h * G:(h + 1) * G].view(1, G), see)[0])
    return torch.cat(out)


def exact(case, seed):
    s, kind, x = SHAPES.get(case.get("shape")), case["kind"], _inputs(case, seed)
    if kind in ("decode", "block", "window"):
        lens = _lens(case, case["batch"], case["lo"], case["hi"])
    if kind == "decode":
        return _decode_exact(x, s, lens)
    if kind == "window":
        got = []
        for y in x:
            have = [int(v) + 1 for v in y["pos"].view(-1).tolist()]
            got.append(_decode_exact(y, s, have, [int(v) for v in y["start"].view(-1).tolist()]))
        return got
    if kind == "block":
        B = len(lens)
        c, n = x["cos"].reshape(-1, B).t(), x["sin"].reshape(-1, B).t()
        q, k, v = _project64(x["X"], x["Wqkv"], x["gamma"], s, c, n)
        y = dict(x, q=q.unsqueeze(1), k=k.unsqueeze(1), v=v.unsqueeze(1))
        o, K, V = _decode_exact(y, s, lens)
        return [o.reshape(B, -1) @ x["Wout"].double(), K, V]
    if kind == "prefill":
        L = case["prior"] + case["new"]
        return _prefill64(x["q"], _rows64(x["K"], x["table"][0], L), _rows64(x["V"], x["table"][0], L), L, s,
                          case["new"], case["prior"], case["window"], x["sink"], x["kd"], x["vd"])
    if kind == "mixed":
        rows, prior = _mixed_lens(case, s)
        K, V = _written64(x["K"], x["sp"], x["kp"]), _written64(x["V"], x["sp"], x["vp"])
        S, op = case["new"], []
        for i, p in enumerate(prior):
            k1, v1 = _rows64(K, x["tp"][i], p + S), _rows64(V, x["tp"][i], p + S)
            q = x["qp"][i * S:(i + 1) * S].transpose(0, 1)
            op.append(_prefill64(q, k1, v1, p + S, s, S, p, 0, None).transpose(0, 1))
        od = _decode64(dict(x, start=None, sink=None), s, rows)
        at = x["slots"].view(-1)
        return [od, torch.cat(op), _written64(K, at, x["k"][:, 0]), _written64(V, at, x["v"][:, 0])]
    if kind == "qkv":
        d = s["d"]
        q, k, v = _project64(x["X"], x["W"], x["gamma"], s, x["cos"][0, :, :d // 2], x["sin"][0, :, :d // 2])
        q = q.reshape(1, case["tokens"], -1)
        if s["fp8"]:  # whole codes: no float64 value
            return [q, None, None]
        at = x["slots"].view(-1)
        return [q, _written64(x["K"], at, k), _written64(x["V"], at, v)]
    G = case["heads"] // case["kv"]
    S = case["tokens"]
    see = torch.ones(S, S, dtype=torch.bool, device=DEV).tril() if case["causal"] else None
    out = []
    for h in range(case["kv"]):
        out.append(_attend64(x["q"][h * G:(h + 1) * G].double().unsqueeze(0), x["k"][h:h + 1].transpose(1, 2).double(),
                             x["v"][h:h + 1].double(), case["d"] ** -0.5, None, see)[0])
    return torch.cat(out)
