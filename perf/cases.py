"""The work a user of this engine has it do, as cases that can be timed and checked one by one.

Every case is a plain dict; "kind" says what it runs:
  forward   Qwen3W8.forward over W new tokens per row, replayed as a captured graph, the way every
            decode and verify round runs (generate.py): logits of every row and the hidden-state taps
  prompt    Qwen3W8.prefill of a whole prompt on a kept cache: last logits, the taps of every
            position, and (bf16 cache) the keys and values it left there
  draft     DFlashDraftModel.block_logits, replayed as a captured graph: one drafted block
  context   DFlashDraftModel.ingest: the drafter's context keys and values of a prompt
  accept    ops.accept_sample: sampled acceptance of a drafted block
  markov    ops.markov_block: a DSpark block sampled through its Markov head
  logprobs  ops.row_logprobs: log-probabilities of the emitted tokens and their alternatives

Models keep the widths, head counts and vocabularies of the shapes in synthetic.TARGETS and have
few layers: a layer costs what it costs in the full depth (each state has weights of its own, so
that passes on alternating states read them from memory), and a rounding difference travels
through few of them. Weights are seeded N(0, 0.02), quantized affine in groups of 64.
"""

import math
import random
import sys
import zlib
from pathlib import Path

import torch

_PKG = str(Path(__file__).resolve().parents[1] / "mlx-dspark_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

PAGE = 64
WIDTHS = ("qwen3-0.6b", "qwen3-8b", "gemma-12b")
DRAFT_TAPS = 5  # target layers a DFlash drafter is conditioned on


def listed():
    return [
        # plain greedy decoding of a small model in a short chat: one row, latency counts
        dict(name="decode_q06", kind="forward", width="qwen3-0.6b", layers=4, B=1, W=1, ctx_lo=311, ctx_hi=311,
             kv_bits=0),
        # the benchmark's verify step: a 16-position DFlash block over a 4096-token 8-bit cache
        dict(name="verify_q8", kind="forward", width="qwen3-8b", layers=4, B=1, W=16, ctx_lo=4096, ctx_hi=4096,
             kv_bits=8),
        # continuous batching: four conversations of very different length, 8 drafts and a bonus each
        dict(name="batch_q8", kind="forward", width="qwen3-8b", layers=3, B=4, W=9, ctx_lo=1024, ctx_hi=12288,
             kv_bits=0),
        # a DSpark verify of the Gemma-style shape: five sliding layers and a global one, long context
        dict(name="verify_g12", kind="forward", width="gemma-12b", layers=6, B=1, W=9, ctx_lo=8192, ctx_hi=8192,
             kv_bits=0),
        # a long document as the prompt, 8-bit cache, weight rows held for prompts as a server does
        dict(name="prompt_q8_long", kind="prompt", width="qwen3-8b", layers=2, L=4096, kv_bits=8),
        # an ordinary chat turn
        dict(name="prompt_q8_short", kind="prompt", width="qwen3-8b", layers=2, L=203, kv_bits=0),
        # a page of text to the Gemma-style shape
        dict(name="prompt_g12", kind="prompt", width="gemma-12b", layers=6, L=1027, kv_bits=0),
        # one DFlash draft: 16 positions through two 4-bit layers and the target's head
        dict(name="draft_q8", kind="draft", width="qwen3-8b", layers=2, W=16, ctx=2049),
        # the drafter's context of a 2048-token piece of a prompt (the engine hands over such pieces)
        dict(name="context_q8", kind="context", width="qwen3-8b", layers=2, L=2048),
        # sampled acceptance of four rows of 16 drafts at temperature 1 with a nucleus
        dict(name="accept_4x16", kind="accept", B=4, L=16, V=151936, T=1.0, top_p=0.95, top_k=0),
        # a sampled DSpark block of 7 tokens
        dict(name="markov_7", kind="markov", B=1, L=7, V=151936, T=0.7, top_p=0.95, top_k=0),
        # a request that asks for log-probabilities with five alternatives, one 16-token round
        dict(name="logprobs_16", kind="logprobs", R=16, V=151936, top_k=5),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    kind = rng.choice(["forward", "forward", "forward", "prompt", "prompt", "draft", "context", "accept", "markov",
                       "logprobs"])
    width = rng.choice(WIDTHS)
    if kind == "forward":
        B = rng.choice([1, 1, 1, 2, 3, 5])
        W = rng.randint(1, min(17, 64 // B))
        lo = _log_int(rng, 32, 8192)
        return dict(kind=kind, width=width, layers=rng.randint(2, 3) if width != "gemma-12b" else 6, B=B, W=W,
                    ctx_lo=lo, ctx_hi=lo if B == 1 else min(12000, lo * rng.randint(1, 6)), kv_bits=rng.choice([0, 8]))
    if kind == "prompt":
        L = _log_int(rng, 20, 1024 if width == "gemma-12b" else 4000)
        return dict(kind=kind, width=width, layers=2, L=L, kv_bits=rng.choice([0, 8]))
    if kind in ("draft", "context"):
        width = rng.choice(["qwen3-0.6b", "qwen3-8b"])
        if kind == "draft":
            return dict(kind=kind, width=width, layers=2, W=rng.randint(5, 16), ctx=_log_int(rng, 16, 8000))
        return dict(kind=kind, width=width, layers=2, L=_log_int(rng, 3, 2048))
    V = rng.choice([151936, 151936, 262144])
    if kind == "logprobs":
        return dict(kind=kind, R=rng.randint(1, 16), V=V, top_k=rng.randint(0, 20))
    T = round(rng.uniform(0.3, 1.2), 2)
    top_p = rng.choice([0.8, 0.9, 0.95, 1.0])
    top_k = rng.choice([0, 0, 20, 50])
    if kind == "accept":
        B = rng.randint(1, 4)
        return dict(kind=kind, B=B, L=rng.randint(1, 9), V=V, T=T, top_p=top_p, top_k=top_k)
    return dict(kind=kind, B=1, L=rng.randint(2, 8), V=V, T=T, top_p=top_p, top_k=top_k)


# ----------------------------------------------------------------------------- inputs
def _gen(seed, name):
    g = torch.Generator(device="cuda")
    g.manual_seed(zlib.crc32(f"{int(seed)}:{name}".encode()))
    return g


def _randn(shape, seed, name, std=1.0):
    return torch.randn(shape, generator=_gen(seed, name), device="cuda", dtype=torch.float32).mul_(std)


def _ids(shape, V, seed, name):
    return torch.randint(0, V, shape, generator=_gen(seed, name), device="cuda", dtype=torch.int32)


def _codes(N, K, seed, name, bits=8):
    """A seeded weight as affine group-64 codes: (codes u8 [N, K], scales, biases bf16 [N, K/64])."""
    levels = float(2 ** bits - 1)
    q = torch.empty((N, K), dtype=torch.uint8, device="cuda")
    s = torch.empty((N, K // 64), dtype=torch.bfloat16, device="cuda")
    b = torch.empty_like(s)
    g = _gen(seed, name)
    for n0 in range(0, N, 32768):
        n1 = min(N, n0 + 32768)
        w = torch.randn((n1 - n0, K // 64, 64), generator=g, device="cuda", dtype=torch.float32).mul_(0.02)
        lo, hi = w.amin(2), w.amax(2)
        s[n0:n1], b[n0:n1] = (hi - lo) / levels, lo
        w.sub_(b[n0:n1].float()[..., None]).div_(s[n0:n1].float()[..., None])
        q[n0:n1] = w.round_().clamp_(0, levels).view(n1 - n0, K).to(torch.uint8)
    return q, s, b


def _deq(c):
    q, s, b = c
    N, K = q.shape
    return (q.double().view(N, K // 64, 64) * s.double()[..., None] + b.double()[..., None]).view(N, K)


def _gains(n, seed, name, mean=1.0):
    return (mean * (1.0 + _randn((n,), seed, name, 0.1))).to(torch.bfloat16)


def _args(case):
    from mlx_dspark import synthetic

    a = synthetic.target_args(case["width"])
    a.num_hidden_layers = case["layers"]
    a.layer_types = tuple(a.layer_types[:case["layers"]])
    return a


def _layer_parts(a, seed, l, bits):
    """One layer's weights as codes, and its norm gains."""
    H, I, hd = a.hidden_size, a.intermediate_size, a.head_dim
    p = f"layer{l}."
    w = dict(qkv=_codes(a.n_qkv, H, seed, p + "qkv", bits),
             o=_codes(H, a.num_attention_heads * hd, seed, p + "o", bits),
             gate_up=_codes(2 * I, H, seed, p + "gate_up", bits), down=_codes(H, I, seed, p + "down", bits))
    n = dict(in_norm=_gains(H, seed, p + "in"), post_norm=_gains(H, seed, p + "post"),
             q_norm=_gains(hd, seed, p + "q", hd ** -0.25), k_norm=_gains(hd, seed, p + "k", hd ** -0.25))
    if a.sandwich_norms:
        n.update(attn_out_norm=_gains(H, seed, p + "ao"), ff_out_norm=_gains(H, seed, p + "fo"))
    return w, n


def _layers(a, seed, bits=8):
    from mlx_dspark.ops import W8Weight
    from mlx_dspark.qwen3 import LayerWeights

    out = []
    for l in range(a.num_hidden_layers):
        w, n = _layer_parts(a, seed, l, bits)
        out.append(LayerWeights(**{k: W8Weight.from_mlx(*c, paired=k == "gate_up", bits=bits) for k, c in w.items()},
                                **n))
    return out


def _embed_codes(a, seed):
    return _codes(a.vocab_size, a.hidden_size, seed, "embed")


def _head_codes(a, seed):
    return _embed_codes(a, seed) if a.tie_word_embeddings else _codes(a.vocab_size, a.hidden_size, seed, "head")


def _model(a, seed):
    from mlx_dspark.ops import W8Table, W8Weight
    from mlx_dspark.qwen3 import Qwen3W8

    return Qwen3W8(a, _layers(a, seed), W8Table(*_embed_codes(a, seed)), W8Weight.from_mlx(*_head_codes(a, seed)),
                   _gains(a.hidden_size, seed, "norm"))


def _drafter(case, seed):
    """A 4-bit DFlash drafter of the target's shape (the reference's default code width)."""
    from mlx_dspark.dflash_model import DFlashConfig, DFlashDraftModel
    from mlx_dspark.ops import W8Weight

    a = _args(case)
    cfg = DFlashConfig(hidden_size=a.hidden_size, num_hidden_layers=a.num_hidden_layers,
                       num_attention_heads=a.num_attention_heads, num_key_value_heads=a.num_key_value_heads,
                       head_dim=a.head_dim, intermediate_size=a.intermediate_size, vocab_size=a.vocab_size,
                       rms_norm_eps=a.rms_norm_eps, rope_theta=a.rope_theta,
                       max_position_embeddings=a.max_position_embeddings, block_size=case.get("W", 16),
                       target_layer_ids=tuple(range(DRAFT_TAPS)), num_target_layers=DRAFT_TAPS,
                       mask_token_id=a.vocab_size - 1)
    H = a.hidden_size
    fc = W8Weight.from_mlx(*_codes(H, DRAFT_TAPS * H, seed, "fc", 4), bits=4)
    return DFlashDraftModel(cfg, fc, _gains(H, seed, "hidden_norm"), _layers(a, seed, 4), _gains(H, seed, "norm"))


def _lengths(case):
    B = case["B"]
    lo, hi = case["ctx_lo"], case["ctx_hi"]
    return [int(round(lo * (hi / lo) ** (b / max(1, B - 1)))) for b in range(B)]


def _context(n_layers, nkv, hd, lengths, kv_bits, seed):
    """Cached keys and values of every row: per layer and row, (K, V) as bf16 [nkv, len, hd], or as
    (codes, words) with words = bf16 scale | bf16 bias << 16 per 64 dims."""
    def stored(name, n, std):
        x = _randn((nkv, n, hd), seed, name, std)
        if not kv_bits:
            return x.to(torch.bfloat16)
        g = x.view(nkv, n, hd // 64, 64)
        lo, hi = g.amin(3), g.amax(3)
        s, b = ((hi - lo) / 255.0).to(torch.bfloat16), lo.to(torch.bfloat16)
        q = ((g - b.float()[..., None]) / s.float()[..., None]).round_().clamp_(0, 255).to(torch.uint8)
        word = (s.view(torch.int16).int() & 0xFFFF) | (b.view(torch.int16).int() << 16)
        return q.view(nkv, n, hd), word

    # keys as normed and rotated ones are spread, values as projections of unit rows are
    return [[(stored(f"ctx{l}.{b}.k", n, hd ** -0.25), stored(f"ctx{l}.{b}.v", n, 1.0))
             for b, n in enumerate(lengths)] for l in range(n_layers)]


def _fill(cache, lengths, kv_bits, seed):
    """Put a context into a cache whose rows' pages are scattered over the pool, as after some use."""
    order = torch.randperm(cache.n_pages, generator=torch.Generator().manual_seed(seed & 0xFFFF)).tolist()
    for b in range(cache.B):
        cache.set_row_pages(b, order[b * cache.max_pages:(b + 1) * cache.max_pages])
    ctx = _context(cache.n_layers, cache.n_kv, cache.head_dim, lengths, kv_bits, seed)
    for l in range(cache.n_layers):
        k, v, ksb, vsb = cache.layer_args(l)
        for b, n in enumerate(lengths):
            np_ = -(-n // PAGE)
            pages = cache.block_table[b, :np_].long()
            for pool, sb, x in ((k, ksb, ctx[l][b][0]), (v, vsb, ctx[l][b][1])):
                for dst, src in ((pool, x[0]), (sb, x[1])) if kv_bits else ((pool, x),):
                    padded = torch.zeros((src.shape[0], np_ * PAGE, src.shape[2]), dtype=src.dtype, device="cuda")
                    padded[:, :n] = src
                    dst[pages] = padded.view(src.shape[0], np_, PAGE, -1).transpose(0, 1)
    cache.set_lengths(lengths)


def _captured(fn):
    """fn warmed up once and captured, as the engine's rounds capture theirs: a replay per pass."""
    fn()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = fn()
    return g, out


def _taps(case):
    return sorted({0, case["layers"] - 1})


def prepare(case, seed):
    kind = case["kind"]
    if kind == "forward":
        a = _args(case)
        model = _model(a, seed)
        lengths = _lengths(case)
        cache = model.make_cache(case["B"], max(lengths) + 64, case["kv_bits"] or None)
        _fill(cache, lengths, case["kv_bits"], seed)
        ids = _ids((case["B"], case["W"]), a.vocab_size, seed, "ids")
        logits = torch.empty((case["B"] * case["W"], a.vocab_size), dtype=torch.float32, device="cuda")
        graph, out = _captured(lambda: model.forward(ids, cache, _taps(case), advance=False, logits_out=logits))
        return dict(kind=kind, keep=(model, cache, ids), graph=graph, out=out)
    if kind == "prompt":
        a = _args(case)
        model = _model(a, seed)
        model.keep_dense_weights(case["L"] >= 256 and not a.sandwich_norms)
        cache = model.make_cache(1, case["L"] + 1, case["kv_bits"] or None)
        ids = _ids((1, case["L"]), a.vocab_size, seed, "ids")
        return dict(kind=kind, model=model, cache=cache, ids=ids, taps=_taps(case), kv=not case["kv_bits"])
    if kind == "draft":
        from types import SimpleNamespace

        from mlx_dspark.ops import W8Table, W8Weight

        a = _args(case)
        d = _drafter(case, seed)
        d.bind(SimpleNamespace(embed=W8Table(*_embed_codes(a, seed)), lm_head=W8Weight.from_mlx(*_head_codes(a, seed)),
                               args=a))
        cache = d.make_cache(case["ctx"] + 64)
        _fill(cache, [case["ctx"]], 0, seed)
        ids = _block_ids(case, a, seed)
        logits = torch.empty((case["W"] - 1, a.vocab_size), dtype=torch.float32, device="cuda")
        graph, out = _captured(lambda: d.block_logits(ids, cache, 1, out=logits))
        return dict(kind=kind, keep=(d, cache, ids), graph=graph, out=out)
    if kind == "context":
        d = _drafter(case, seed)
        return dict(kind=kind, drafter=d, cache=d.make_cache(case["L"]), hidden=_hidden(case, seed))
    if kind == "accept":
        p, q, draft = _accept_rows(case, seed)
        return dict(kind=kind, p=p, q=q, draft=draft, seed=seed, T=case["T"], top_p=case["top_p"],
                    top_k=case["top_k"], flags=torch.zeros((case["B"], case["L"]), dtype=torch.uint8, device="cuda"))
    if kind == "markov":
        from mlx_dspark.ops import W8Table, W8Weight

        base = _randn((case["B"], case["L"], case["V"]), seed, "base", 3.0)
        return dict(kind=kind, base=base, prev=_ids((case["B"],), case["V"], seed, "prev"),
                    w1=W8Table(*_codes(case["V"], 256, seed, "w1", 4)),
                    w2=W8Weight.from_mlx(*_codes(case["V"], 256, seed, "w2", 4), bits=8), seed=seed, T=case["T"],
                    top_p=case["top_p"], top_k=case["top_k"])
    logits, tokens = _logprob_rows(case, seed)
    return dict(kind=kind, logits=logits, tokens=tokens, top_k=case["top_k"])


def _block_ids(case, a, seed):
    ids = torch.full((1, case["W"]), a.vocab_size - 1, dtype=torch.int32, device="cuda")
    ids[:, :1] = _ids((1, 1), a.vocab_size - 1, seed, "anchor")
    return ids


def _hidden(case, seed):
    H = _args(case).hidden_size
    return _randn((case["L"], DRAFT_TAPS * H), seed, "hidden").to(torch.bfloat16)


def _accept_rows(case, seed):
    """Target rows that follow the draft rows (draft N(0, 9), target = draft + N(0, 1)), drafts drawn
    from the draft rows at the case's temperature."""
    B, L, V = case["B"], case["L"], case["V"]
    q = _randn((B, L, V), seed, "q", 3.0)
    p = torch.cat([q + _randn((B, L, V), seed, "pq"), _randn((B, 1, V), seed, "p", 3.0)], dim=1)
    u = torch.rand((B, L, V), generator=_gen(seed, "u"), device="cuda").clamp_(1e-30, 1 - 1e-7)
    draft = (q / case["T"] - torch.log(-torch.log(u))).argmax(2).to(torch.int32)
    return p, q, draft


def _logprob_rows(case, seed):
    logits = _randn((case["R"], case["V"]), seed, "logits", 3.0)
    return logits, logits.argmax(1).to(torch.int32)


def run(state):
    from mlx_dspark import ops

    kind = state["kind"]
    if "graph" in state:  # a decode, verify or draft round: the captured graph's own outputs
        state["graph"].replay()
        return state["out"]
    if kind == "prompt":
        cache = state["cache"]
        cache.trim_to(0)
        logits, fused = state["model"].prefill(state["ids"], cache, state["taps"])
        if not state["kv"]:  # 8-bit codes: read back by the same pass's attention
            return logits, fused
        return logits, fused, [c.keys for c in cache], [c.values for c in cache]
    if kind == "context":
        cache = state["cache"]
        cache.trim_to(0)
        state["drafter"].ingest(state["hidden"], cache)
        return [c.keys for c in cache], [c.values for c in cache], cache.seq_lens
    if kind == "accept":
        n, token = ops.accept_sample(state["p"], state["q"], state["draft"], state["T"], state["top_p"],
                                     state["top_k"], seed=state["seed"], offset=3, accept_out=state["flags"])
        return n, token, state["flags"]
    if kind == "markov":
        return ops.markov_block(state["base"], state["prev"], state["w1"], state["w2"], temperature=state["T"],
                                top_p=state["top_p"], top_k=state["top_k"], seed=state["seed"], offset=3)
    return ops.row_logprobs(state["logits"], state["tokens"], state["top_k"])


# ----------------------------------------------------------------------------- what a pass needs
def _linear(N, K, M, bits=8):
    return N * K * (bits / 8 + 1 / 16), 2.0 * M * N * K


def _layer_work(a, M, bits, keys, kv_bytes, windows):
    """Bytes and operations of every layer: weights once, each (row, layer)'s visible keys once,
    scores and values per query and key. keys: per row (context, new tokens, causal)."""
    H, I, nq, nkv, hd = a.hidden_size, a.intermediate_size, a.num_attention_heads, a.num_key_value_heads, a.head_dim
    byt = flo = 0.0
    for win in windows:
        for N, K in ((a.n_qkv, H), (H, nq * hd), (2 * I, H), (H, I)):
            x, y = _linear(N, K, M, bits)
            byt += x
            flo += y
        for n, w, causal in keys:
            read = min(n, win) if win else n
            pairs = sum(min(n + i + 1, win) if win else n + i + 1 for i in range(w)) if causal else w * (n + w)
            byt += 2 * nkv * hd * kv_bytes * (read + w)
            flo += 4.0 * pairs * nq * hd
    return byt, flo


def work(case):
    kind = case["kind"]
    if kind in ("forward", "prompt", "draft", "context"):
        a = _args(case)
        H, V, hd, nkv = a.hidden_size, a.vocab_size, a.head_dim, a.num_key_value_heads
        windows = [a.window(l) for l in range(a.num_hidden_layers)]
        kv_bytes = 1 + 4 / 64 if case.get("kv_bits") else 2
    if kind == "forward":
        M = case["B"] * case["W"]
        byt, flo = _layer_work(a, M, 8, [(n, case["W"], True) for n in _lengths(case)], kv_bytes, windows)
        x, y = _linear(V, H, M)
        return dict(bytes=byt + x + 4.0 * M * V + 2.0 * M * H * len(_taps(case)), flops=flo + y)
    if kind == "prompt":
        L = case["L"]
        byt, flo = _layer_work(a, L, 8, [(0, L, True)], kv_bytes, windows)
        x, y = _linear(V, H, 1)
        return dict(bytes=byt + x + 4.0 * V + 2.0 * L * H * len(_taps(case)), flops=flo + y)
    if kind == "draft":
        M = case["W"]
        byt, flo = _layer_work(a, M, 4, [(case["ctx"], M, False)], 2, [0] * a.num_hidden_layers)
        x, y = _linear(V, H, M - 1)
        return dict(bytes=byt + x + 4.0 * (M - 1) * V, flops=flo + y)
    if kind == "context":
        L = case["L"]
        byt, flo = _linear(H, DRAFT_TAPS * H, L, 4)
        for _ in range(a.num_hidden_layers):
            x, y = _linear(2 * nkv * hd, H, L, 4)
            byt += x + 4.0 * L * nkv * hd
            flo += y
        return dict(bytes=byt + 2.0 * L * DRAFT_TAPS * H, flops=flo)
    if kind == "accept":
        n = case["B"] * (2 * case["L"] + 1) * case["V"]
        return dict(bytes=4.0 * n, flops=20.0 * n)
    if kind == "markov":
        n = case["B"] * case["L"] * case["V"]
        return dict(bytes=8.0 * n + _linear(case["V"], 256, 1)[0], flops=2.0 * n * 256)
    return dict(bytes=4.0 * case["R"] * case["V"], flops=4.0 * case["R"] * case["V"])


def tolerance(case):
    """bf16 activations: a changed order of the float32 sums flips roundings of one bf16 step
    (2^-8), which the layers that follow carry on: against the 64-bit results the forward, prompt
    and draft cases are 0.008 to 0.014 off, the context 0.0037. Sampling returns whole numbers; the
    Markov rows are sums of bf16 terms rounded to bf16."""
    kind = case["kind"]
    if kind in ("forward", "prompt", "draft"):
        return dict(rel=0.03, max=0.4)
    if kind == "context":
        return dict(rel=0.014, max=0.2)
    if kind == "accept":
        return "exact"
    if kind == "markov":
        return dict(rel=1e-3, max=0.02, differ=0.0)
    return dict(rel=1e-5, max=1e-4, differ=0.0)


# ----------------------------------------------------------------------------- 64-bit results
def _rms(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * (1.0 if w is None else w.double())


def _rope(x, pos, theta):
    """x [n, heads, hd] rotated by halves at positions pos [n]."""
    hd = x.shape[-1]
    inv = (theta ** (-2.0 * torch.arange(hd // 2, device="cuda", dtype=torch.float64) / hd)).float().double()
    ang = pos.double()[:, None] * inv
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    x1, x2 = x[..., :hd // 2], x[..., hd // 2:]
    return torch.cat([x1 * c - x2 * s, x2 * c + x1 * s], dim=-1)


def _linear64(x, codes):
    out = torch.empty((x.shape[0], codes[0].shape[0]), dtype=torch.float64, device="cuda")
    for n0 in range(0, out.shape[1], 16384):
        out[:, n0:n0 + 16384] = x @ _deq(tuple(t[n0:n0 + 16384] for t in codes)).t()
    return out


def _stored64(x):
    if not isinstance(x, tuple):
        return x.double()
    q, word = x
    s = (word << 16).view(torch.float32).double()
    b = (word & -65536).view(torch.float32).double()
    nkv, n, hd = q.shape
    return (q.double().view(nkv, n, hd // 64, 64) * s[..., None] + b[..., None]).view(nkv, n, hd)


def _layer64(a, seed, l, h, rows, ctx, bits, causal):
    """h [M, H] after layer l (rows: (first, last, context length) of each batch row in M), and the
    new keys and values [M, nkv, hd]."""
    w, n = _layer_parts(a, seed, l, bits)
    nq, nkv, hd, eps = a.num_attention_heads, a.num_key_value_heads, a.head_dim, a.rms_norm_eps
    qkv = _linear64(_rms(h, n["in_norm"], eps), w["qkv"]).view(-1, nq + 2 * nkv, hd)
    theta = a.rope_local_base_freq if a.is_sliding(l) and a.rope_local_base_freq else a.rope_theta
    pos = torch.cat([torch.arange(c, c + m1 - m0, device="cuda") for m0, m1, c in rows])
    q = _rope(_rms(qkv[:, :nq], n["q_norm"], eps), pos, theta)
    k = _rope(_rms(qkv[:, nq:nq + nkv], n["k_norm"], eps), pos, theta)
    v = qkv[:, nq + nkv:]
    o = torch.empty((h.shape[0], nq, hd), dtype=torch.float64, device="cuda")
    win = a.window(l)
    for b, (m0, m1, c) in enumerate(rows):
        j = torch.arange(c + m1 - m0, device="cuda")[None]
        i = torch.arange(c, c + m1 - m0, device="cuda")[:, None]
        seen = (j <= i) if causal else torch.ones_like(j <= i)
        if win:
            seen = seen & (j > i - win)
        for g in range(nkv):
            kk, vv = k[m0:m1, g], v[m0:m1, g]
            if ctx is not None:
                kk = torch.cat([_stored64(ctx[l][b][0])[g], kk])
                vv = torch.cat([_stored64(ctx[l][b][1])[g], vv])
            for t in range(g * (nq // nkv), (g + 1) * (nq // nkv)):
                s = (q[m0:m1, t] @ kk.t() * a.attn_scale).masked_fill_(~seen, -math.inf)
                o[m0:m1, t] = torch.softmax(s, dim=1) @ vv
    y = _linear64(o.view(h.shape[0], -1), w["o"])
    h = h + (_rms(y, n["attn_out_norm"], eps) if a.sandwich_norms else y)
    gu = _linear64(_rms(h, n["post_norm"], eps), w["gate_up"])
    I = a.intermediate_size
    act = torch.nn.functional.silu(gu[:, :I]) if a.hidden_act == "silu" else \
        torch.nn.functional.gelu(gu[:, :I], approximate="tanh")
    y = _linear64(act * gu[:, I:], w["down"])
    return h + (_rms(y, n["ff_out_norm"], eps) if a.sandwich_norms else y), k, v


def _logits64(a, seed, h):
    y = _linear64(_rms(h, _gains(a.hidden_size, seed, "norm"), a.rms_norm_eps), _head_codes(a, seed))
    cap = a.final_logit_softcapping
    return torch.tanh(y / cap) * cap if cap else y


def _embed64(a, seed, ids):
    c = _embed_codes(a, seed)
    return _deq(tuple(t[ids.reshape(-1).long()] for t in c)) * a.embed_scale


def exact(case, seed):
    kind = case["kind"]
    if kind in ("forward", "prompt"):
        a = _args(case)
        if kind == "forward":
            B, W, lens = case["B"], case["W"], _lengths(case)
            ctx = _context(a.num_hidden_layers, a.num_key_value_heads, a.head_dim, lens, case["kv_bits"], seed)
        else:
            B, W, lens, ctx = 1, case["L"], [0], None
        rows = [(b * W, (b + 1) * W, n) for b, n in enumerate(lens)]
        h = _embed64(a, seed, _ids((B, W), a.vocab_size, seed, "ids"))
        taps, ks, vs = [], [], []
        for l in range(a.num_hidden_layers):
            h, k, v = _layer64(a, seed, l, h, rows, ctx, 8, True)
            ks.append(k)
            vs.append(v)
            if l in _taps(case):
                taps.append(h)
        fused = torch.cat(taps, dim=1).view(B, W, -1)
        if kind == "forward":
            return _logits64(a, seed, h).view(B, W, -1), fused
        logits = _logits64(a, seed, h[-1:]).view(1, 1, -1)
        if case["kv_bits"]:
            return logits, fused
        return logits, fused, _cache64(ks, case), _cache64(vs, case)
    if kind == "draft":
        a = _args(case)
        ctx = _context(a.num_hidden_layers, a.num_key_value_heads, a.head_dim, [case["ctx"]], 0, seed)
        h = _embed64(a, seed, _block_ids(case, a, seed))
        for l in range(a.num_hidden_layers):
            h, _, _ = _layer64(a, seed, l, h, [(0, case["W"], case["ctx"])], ctx, 4, False)
        return _logits64(a, seed, h[1:]).view(1, case["W"] - 1, -1)
    if kind == "context":
        return _context64(case, seed)
    if kind == "logprobs":
        logits, tokens = _logprob_rows(case, seed)
        lp = torch.log_softmax(logits.double(), dim=1)
        return lp.gather(1, tokens.long()[:, None])[:, 0], None, lp.topk(case["top_k"], dim=1).values
    return None


def _context64(case, seed):
    a = _args(case)
    H, nkv, hd, L = a.hidden_size, a.num_key_value_heads, a.head_dim, case["L"]
    fc = _codes(H, DRAFT_TAPS * H, seed, "fc", 4)
    x = _rms(_linear64(_hidden(case, seed).double(), fc), _gains(H, seed, "hidden_norm"), a.rms_norm_eps)
    ks, vs = [], []
    pos = torch.arange(L, device="cuda")
    for l in range(a.num_hidden_layers):
        w, n = _layer_parts(a, seed, l, 4)
        first = a.num_attention_heads * hd
        kv = _linear64(x, tuple(t[first:] for t in w["qkv"])).view(L, 2 * nkv, hd)
        ks.append(_rope(_rms(kv[:, :nkv], n["k_norm"], a.rms_norm_eps), pos, a.rope_theta))
        vs.append(kv[:, nkv:])
    return _cache64(ks, case), _cache64(vs, case), None


def _cache64(xs, case):
    """Per layer [n, nkv, hd] rows as the pages of the case's one-row cache hold them (zeros beyond)."""
    room = case["L"] + (16 if case["kind"] == "context" else 1)  # a drafter's cache keeps room for a block
    pages = -(-room // PAGE)
    out = []
    for x in xs:
        p = torch.zeros((pages * PAGE,) + tuple(x.shape[1:]), dtype=torch.float64, device="cuda")
        p[:x.shape[0]] = x
        out.append(p.view(pages, PAGE, *x.shape[1:]).transpose(1, 2).contiguous())
    return out
