"""GPU: the products of many rows (dsk_rows_prep, dsk_w8_rows) at the edges of every tile the planner
picks, and the many-row attention (dsk_attention_rows) at head_dim 128 and 256, against float64.

A product's error: each of its two sums (scaled code products, bias products) accumulates at most K
float32 terms, so K * 2^-24 of the sum of magnitudes, and the store rounds to bf16 (2^-8 of the
value, 2^-9 for the rounding and as much for a flip of the input's own rounding in the reference)."""

import pytest
import torch

pytestmark = pytest.mark.gpu

# (M, N, K): the plan each reaches (64-row blocks x column tiles, groups per step, K slices)
SHAPES = [
    (1, 48, 256),        # 1 x 1: an odd number of column tiles
    (65, 32, 256),       # 1 x 2, two slices (four groups), a second block of one row
    (70, 256, 512),      # 1 x 2, four slices
    (190, 4096, 256),    # 1 x 4, four slices
    (129, 4160, 512),    # 2 x 4, four slices
    (130, 8192, 768),    # 2 x 4, two slices
    (515, 16384, 256),   # 2 x 4, one slice (a 256-row tile would pad too much)
    (1024, 8192, 256),   # 4 x 4
    (203, 256, 8192 + 256),  # more groups than one step of the bias term
]


def _weight(N, K, bits, paired, dev):
    from mlx_dspark.ops import W8Weight
    g = torch.Generator(device=dev).manual_seed(N + K + bits)
    q, s, b = W8Weight.quantize_mlx(torch.randn(N, K, generator=g, device=dev) * 0.02, bits)
    qs = q.double().view(N, K // 64, 64) * s.double()[..., None]
    bb = b.double()[..., None].expand(N, K // 64, 64)
    return W8Weight.from_mlx(q, s, b, paired, bits), (qs + bb).reshape(N, K), (qs + bb.abs()).reshape(N, K)


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("bits", [8, 4])
def test_products_of_many_rows(dev, M, N, K, bits):
    from mlx_dspark.ops import DSK_EPI_GEGLU, DSK_EPI_RESIDUAL, DSK_EPI_SWIGLU, rows_prep, w8_rows
    print(f"rows M={M} N={N} K={K} bits={bits}", flush=True)
    g = torch.Generator(device=dev).manual_seed(M + bits)
    wide = (torch.randn(M, K + 64, generator=g, device=dev) * 3).to(torch.bfloat16)
    h = wide[:, :K]                                       # strided rows
    norm = (1 + 0.2 * torch.randn(K, generator=g, device=dev)).to(torch.bfloat16)
    eps = 1e-6
    W, w64, mag = _weight(N, K, bits, False, dev)
    x64 = (h.float() * norm.float()).to(torch.bfloat16).double()
    r = torch.rsqrt(h.double().square().mean(1, keepdim=True) + eps)
    ref, bound = (x64 @ w64.T) * r, K * 2.0 ** -24 * (x64.abs() @ mag.T) * r
    x = rows_prep(h, norm_w=norm, eps=eps, later=True)
    y = w8_rows(x, W)
    assert bool(((y.double() - ref).abs() <= bound + ref.abs() * 2.0 ** -8).all())
    # residual add, with a strided copy
    res = torch.randn(M, N, generator=g, device=dev).to(torch.bfloat16)
    hh, taps = res.clone(), torch.zeros((M, 2 * N), dtype=torch.bfloat16, device=dev)
    w8_rows(x, W, epi=DSK_EPI_RESIDUAL, h=hh, copy=taps[:, N:])
    want = res.double() + ref
    assert bool(((hh.double() - want).abs() <= bound + want.abs() * 2.0 ** -8).all())
    assert torch.equal(taps[:, N:], hh) and not bool(taps[:, :N].any())
    if N % 32:
        return
    Wp, w64, mag = _weight(N, K, bits, True, dev)
    ref, bound = (x64 @ w64.T) * r, K * 2.0 ** -24 * (x64.abs() @ mag.T) * r
    e_gate, e_up = (bound + 2.0 ** -8 * ref.abs()).split(N // 2, dim=1)   # each rounded to bf16
    gate, up = ref[:, :N // 2], ref[:, N // 2:]
    for epi, act in ((DSK_EPI_SWIGLU, torch.nn.functional.silu(gate)),
                     (DSK_EPI_GEGLU, torch.nn.functional.gelu(gate, approximate="tanh"))):
        y, want = w8_rows(x, Wp, epi=epi), act * up
        # three bf16 roundings (gate, up, act) of factors of at most slope 1.13, and the store's
        # element by element: the gate's error through the activation (slope at most 1.13) and its rounding,
        # times up, up's times the activation, and the store's rounding
        e_act = 1.13 * e_gate + 2.0 ** -8 * act.abs()
        assert bool(((y.double() - want).abs() <= act.abs() * e_up + e_act * (up.abs() + e_up)
                     + 2.0 ** -8 * want.abs()).all())


@pytest.mark.parametrize("M,K", [(1, 64), (3, 4096), (67, 4160), (130, 12288), (5, 24576)])
def test_prepared_rows(dev, M, K):
    """The residual add and norms against float64, the operand order, and the group sums' terms."""
    from mlx_dspark.ops import rows_prep
    g = torch.Generator(device=dev).manual_seed(M + K)
    rnd = lambda: (torch.randn(M, K, generator=g, device=dev) * 2).to(torch.bfloat16)
    w1, w2 = ((1 + 0.3 * torch.randn(K, generator=g, device=dev)).to(torch.bfloat16) for _ in range(2))
    h, y, copy, eps = rnd(), rnd(), torch.zeros((M, K), dtype=torch.bfloat16, device=dev), 1e-6
    h0 = h.clone()
    x = rows_prep(h, part=y, part_norm_w=w1, copy=copy, norm_w=w2, eps=eps)
    rms = lambda t: t * torch.rsqrt(t.square().mean(1, keepdim=True) + eps)
    h64 = h0.double() + rms(y.double()) * w1.double()
    assert bool(((h.double() - h64).abs() <= 2.0 ** -7 * (h64.abs() + rms(y.double()).abs() * w1.double().abs())).all())
    assert torch.equal(h, copy)
    Mp, G = (M + 15) // 16 * 16, K // 64
    rows = x.data.view(Mp // 16, G, 2, 4, 16, 8).permute(0, 4, 1, 3, 2, 5).reshape(Mp, K)[:M]
    x64 = rms(h.double()) * w2.double()
    assert bool(((rows.double() - x64).abs() <= x64.abs() * 2.0 ** -7 + 1e-6).all())
    Gp = (G + 63) // 64 * 64
    xt = x.xt.view(3, Mp // 16, Gp // 64, 2, 4, 16, 8).permute(0, 1, 5, 2, 4, 3, 6).reshape(3, Mp, Gp)[:, :M]
    sums = rows.double().view(M, G, 64).sum(2)
    mags = rows.double().abs().view(M, G, 64).sum(2)
    assert bool(((xt.double().sum(0)[:, :G] - sums).abs() <= mags * 2.0 ** -20).all())
    assert not bool(xt[:, :, G:].any())
    # without a norm the operand is the rows themselves
    plain = rows_prep(h)
    assert torch.equal(plain.data.view(Mp // 16, G, 2, 4, 16, 8).permute(0, 4, 1, 3, 2, 5).reshape(Mp, K)[:M], h)


def _check_many_rows(dev, hd, kv_bits, lens, W, nq, nkv, causal, window, two_terms=False):
    from mlx_dspark import ops
    from mlx_dspark.kv import PagedKVCache
    print(f"attention rows hd={hd} kv_bits={kv_bits} lens={lens} W={W} window={window}", flush=True)
    B = len(lens)
    cache = PagedKVCache(1, B, nkv, hd, max(lens) + W + 64, kv_bits=kv_bits, spare_pages=3)
    g = torch.Generator(device=dev).manual_seed(sum(lens) + W + hd)
    perm = torch.randperm(cache.n_pages, generator=torch.Generator().manual_seed(W))[: B * cache.max_pages]
    cache.block_table.copy_(perm.view(B, cache.max_pages).to(torch.int32))
    pools = []
    for pool, sb in ((cache.k[0], cache.k_sb[0]), (cache.v[0], cache.v_sb[0])):
        if kv_bits is None:
            pool.copy_(torch.randn(pool.shape, generator=g, device=dev))
            pools.append(pool.double())
            continue
        pool.copy_(torch.randint(0, 256, pool.shape, generator=g, device=dev))
        sc = (0.01 + 0.01 * torch.rand(sb.shape, generator=g, device=dev)).to(torch.bfloat16)
        bi = (-2.0 + torch.rand(sb.shape, generator=g, device=dev)).to(torch.bfloat16)
        sb.copy_((sc.view(torch.int16).int() & 0xFFFF) | (bi.view(torch.int16).int() << 16))
        v = pool.float().view(*pool.shape[:-1], hd // 64, 64) * sc.float()[..., None] + bi.float()[..., None]
        pools.append(v.view(pool.shape).to(torch.bfloat16).double())
    cache.set_lengths(lens)
    q = torch.randn(B * W, nq * hd, generator=g, device=dev).to(torch.bfloat16)
    outs = [f(q, B, W, nq, nkv, hd, hd ** -0.5, cache.seq_lens, cache.max_ctx, cache.block_table, cache.page,
              cache.kv_dtype, *cache.layer_args(0), causal=causal, window=window).double().view(B, W, nq, hd)
            for f in ([ops.attention_rows, ops.attention] if two_terms else [ops.attention_rows])]
    for b, L0 in enumerate(lens):
        n = L0 + W
        K, V = (p[cache.block_table[b].long()].transpose(1, 2).reshape(-1, nkv, hd)[:n] for p in pools)
        pos = torch.arange(L0, n, device=dev)[:, None]
        j = torch.arange(n, device=dev)[None, :]
        ok = j <= pos if causal else torch.ones((W, n), dtype=torch.bool, device=dev)
        if window:
            ok = ok & (j > pos - window)
        for t in range(nq):
            sc = (q.double().view(B, W, nq, hd)[b, :, t] @ K[:, t * nkv // nq].T) * hd ** -0.5
            ref = torch.softmax(sc.masked_fill(~ok, -float("inf")), -1) @ V[:, t * nkv // nq]
            for got in outs:
                assert float((got[b, :, t] - ref).abs().max()) <= 2.0 ** -7 * float(ref.abs().max())


@pytest.mark.parametrize("hd,kv_bits,lens,W,nq,nkv,causal,window", [
    (128, 8, [0], 203, 8, 2, True, 0),            # 64-row blocks
    (128, None, [5, 700], 1100, 64, 2, True, 0),  # 256-row blocks (G = 32)
    (128, None, [70], 65, 2, 2, True, 33),
    (256, None, [0], 1027, 4, 2, True, 0),
    (256, 8, [900, 3], 65, 8, 8, True, 130),      # windows that start inside a block
    (256, None, [40], 129, 4, 1, False, 0),
])
def test_many_row_attention(dev, hd, kv_bits, lens, W, nq, nkv, causal, window):
    """Against a float64 softmax over the stored keys: probabilities within 2^-26 and float32 sums
    leave the output's own bf16 rounding (2^-9) and the queries' and keys' products (float32) well
    inside 2^-7 of the largest output."""
    _check_many_rows(dev, hd, kv_bits, lens, W, nq, nkv, causal, window)


@pytest.mark.parametrize("kv_bits,lens,W,nq,nkv,causal,window", [
    (8, [100, 1000, 7], 700, 32, 8, True, 0),      # 256-row blocks: ragged rows, a partial last block
    (None, [100, 1000, 7], 700, 32, 8, True, 0),
    (8, [0], 2100, 64, 8, True, 333),              # windows that start inside a key block
    (None, [0], 2100, 64, 8, True, 333),
    (8, [50], 1100, 32, 8, False, 0),              # one 64-row block too many for two workgroups per CU
    (None, [0], 1300, 32, 8, True, 0),             # few cached positions: 64-row blocks past that
    (8, [900], 1024, 32, 8, True, 0),              # the last size of 64-row blocks, and one row more
    (8, [900], 1025, 32, 8, True, 0),
])
def test_many_row_attention_block_shapes(dev, kv_bits, lens, W, nq, nkv, causal, window):
    """Both block shapes of head_dim 128 on each side of their rule, with the probabilities as three bf16
    terms and as two (within 2^-17: the same bound)."""
    _check_many_rows(dev, 128, kv_bits, lens, W, nq, nkv, causal, window, two_terms=True)


@pytest.mark.parametrize("hd,W", [(128, 65), (128, 4200), (256, 65)])
def test_probabilities_carry_three_terms(dev, hd, W):
    """Values that cancel leave the probabilities' own error: five keys with weights of e^-1.2 to 1, the last
    two values chosen so that every output is below 2^-14 of the weighted magnitudes sum(p |v|) and its bf16
    store hides nothing above 2^-23 of them. Float32 probabilities (exp2 and its argument within 2^-22) and
    sums stay within 2^-21; two bf16 terms, each weight off by up to 2^-17, do not (dsk_attention, head_dim
    128). At 4200 rows the 256-row blocks run."""
    from mlx_dspark import ops
    from mlx_dspark.kv import PagedKVCache
    n = 8
    cache = PagedKVCache(1, 1, n, hd, W)
    g = torch.Generator(device=dev).manual_seed(hd + W)
    # keys 0-4 of head h: q . k = 8 a[h, j], exact in bf16; the others' weights vanish
    a = torch.zeros(n, 5)
    a[:, 1:] = -torch.rand(n, 4, generator=torch.Generator().manual_seed(hd)) * 1.2 * hd ** 0.5 / 8
    a = a.to(torch.bfloat16).to(dev)
    K = torch.zeros(n, cache.max_ctx, hd, dtype=torch.bfloat16, device=dev)
    K[:, :, 0] = -200.0
    K[:, :5, 0] = a
    p = torch.softmax(8 * a.double() * float(torch.tensor(hd ** -0.5)), 1)          # [n, 5]
    V = torch.zeros(n, cache.max_ctx, hd, dtype=torch.bfloat16, device=dev)
    V[:, :3] = torch.randn(n, 3, hd, generator=g, device=dev).to(torch.bfloat16)
    for j in (3, 4):
        V[:, j] = (-(p[:, :j, None] * V[:, :j].double()).sum(1) / p[:, j, None]).to(torch.bfloat16)
    for pool, x in ((cache.k[0], K), (cache.v[0], V)):
        pool.copy_(x.view(n, cache.max_pages, 64, hd).transpose(0, 1))
    q = torch.zeros(W, n, hd, dtype=torch.bfloat16, device=dev)
    q[:, :, 0] = 8.0
    ref = (p[..., None] * V[:, :5].double()).sum(1)
    size = (p[..., None] * V[:, :5].double().abs()).sum(1)
    assert bool((ref.abs() <= 2.0 ** -14 * size).all())
    args = (q.view(W, -1), 1, W, n, n, hd, hd ** -0.5, cache.seq_lens, cache.max_ctx, cache.block_table, cache.page,
            cache.kv_dtype, *cache.layer_args(0))
    err = lambda out: float(((out.double().view(W, n, hd) - ref).abs() / size).max())
    assert err(ops.attention_rows(*args, causal=False)) <= 2.0 ** -21
    if hd == 128:
        assert err(ops.attention(*args, causal=False)) > 2.0 ** -20


def test_prompt_longer_than_a_piece_equals_forward_passes(dev):
    """A Gemma-style prompt of one piece and a few rows more: the same cache, taps and logits as
    64-row forward passes, up to the rounding flips of other sums (2e-2 of the largest value)."""
    from mlx_dspark import synthetic
    from mlx_dspark.qwen3 import PREFILL_CHUNK
    model = synthetic.build_target("tiny-gemma", seed=41)
    n = PREFILL_CHUNK + 7
    prompt = torch.randint(0, model.args.vocab_size, (n,), generator=torch.Generator().manual_seed(1)).tolist()
    outs = []
    for chunk in (64, 63):           # 63: forward passes
        cache = model.make_cache(max_ctx=n + 64)
        seen = []
        logits, _ = model.prefill(prompt, cache, [0, 5], chunk=chunk, on_chunk=lambda f, pos: seen.append((pos, f)))
        torch.cuda.synchronize()
        assert cache.lengths[0] == n and int(cache.seq_lens[0]) == n
        assert [p for p, _ in seen] == list(range(0, n, PREFILL_CHUNK if chunk == 64 else 63))
        outs.append((logits, torch.cat([f for _, f in seen], dim=1), cache.k[5], cache.v[5]))
    for a, b in zip(*outs):
        assert float((a.float() - b.float()).abs().max()) <= 2e-2 * float(b.float().abs().max())


@pytest.mark.parametrize("name,n", [("tiny-gemma", 70), ("tiny-gemma", 200), ("tiny", 65), ("tiny", 130)])
def test_prompt_after_a_long_context_equals_forward_passes(dev, monkeypatch, name, n):
    """A second turn: few rows after many cached positions take the key-split attention (of the Gemma-style
    layers, the global one only). The taps and logits of 64-row forward passes, up to rounding flips."""
    from mlx_dspark import ops, synthetic
    model = synthetic.build_target(name, seed=45)
    a, cached = model.args, 6000
    prompt = torch.randint(0, a.vocab_size, (n,), generator=torch.Generator().manual_seed(3)).tolist()
    passes, real = [], ops.attention
    monkeypatch.setattr(ops, "attention", lambda q, B, W, *r, **k: (passes.append(W), real(q, B, W, *r, **k))[1])
    g = torch.Generator(device=dev).manual_seed(9)
    pools = [[torch.randn(p.shape, generator=g, device=dev).to(p.dtype) for p in pool]
             for pool in (lambda c: (c.k, c.v))(model.make_cache(max_ctx=cached + n))]
    outs = []
    for chunk in (64, 63):           # 63: forward passes
        cache = model.make_cache(max_ctx=cached + n)
        for pool, src in zip((cache.k, cache.v), pools):
            for p, x in zip(pool, src):
                p.copy_(x)
        cache.set_lengths([cached])
        passes.clear()
        logits, fused = model.prefill(prompt, cache, [0, a.num_hidden_layers - 1], chunk=chunk)
        if chunk == 64:
            split = a.num_hidden_layers if name == "tiny" else 1
            assert sorted(passes) == sorted([min(64, n - r) for r in range(0, n, 64)] * split)
        outs.append((logits, fused, cache.k[-1], cache.v[-1]))
    for x, y in zip(*outs):
        assert float((x.float() - y.float()).abs().max()) <= 2e-2 * float(y.float().abs().max())


def test_prompt_pieces_wider_than_a_forward_pass_are_refused(dev):
    """An explicit chunk of more than 64 rows, before any key is appended; a prompt that fits one pass is
    taken whatever the chunk."""
    from mlx_dspark import synthetic
    model = synthetic.build_target("tiny", seed=44)
    cache = model.make_cache(max_ctx=320)
    for chunk in (65, 128, 2048):
        with pytest.raises(ValueError, match="rows per batch row"):
            model.prefill(list(range(200)), cache, None, chunk=chunk)
    torch.cuda.synchronize()
    assert cache.lengths[0] == 0 and not any(bool(k.any()) for k in cache.k)
    model.prefill(list(range(50)), cache, None, chunk=128)
    assert cache.lengths[0] == 50


def test_prompt_into_a_very_long_cache_keeps_small_scratch(dev, monkeypatch):
    """A block table wider than the many-row attention takes: the split attention's scratch stays within
    a 64-row pass's, and the results are those of 64-row passes (rounding flips: 2e-2 of the largest)."""
    from mlx_dspark import _hip, ops, synthetic
    model = synthetic.build_target("tiny-gemma", seed=43)
    a, pages, n = model.args, ops.ROWS_MAX_PAGES + 1, 600
    prompt = torch.randint(0, a.vocab_size, (n,), generator=torch.Generator().manual_seed(2)).tolist()
    reserve, asked = ops.Workspace.reserve, []
    monkeypatch.setattr(ops.Workspace, "reserve",
                        lambda self, kind, b: (asked.append(b) if kind == "attn" else None, reserve(self, kind, b))[1])
    outs = []
    for chunk in (64, 63):           # 63: forward passes
        cache = model.make_cache(max_ctx=pages * 64)
        assert cache.block_table.shape[1] == pages
        logits, fused = model.prefill(prompt, cache, [0, 5], chunk=chunk)
        outs.append((logits, fused))
    assert max(asked) <= _hip.lib.dsk_attn_ws_bytes(1, 64, a.num_attention_heads, a.head_dim, pages * 64)
    for x, y in zip(*outs):
        assert float((x.float() - y.float()).abs().max()) <= 2e-2 * float(y.float().abs().max())


@pytest.mark.parametrize("hd,nq,nkv,kv_bits,v_norm,B,W", [
    (128, 4, 2, None, False, 1, 203), (128, 0, 3, 8, False, 2, 70), (128, 5, 1, 8, True, 1, 128),
    (256, 4, 2, 8, False, 1, 131), (256, 2, 1, None, True, 3, 50), (512, 3, 1, 8, True, 1, 130),
])
def test_append_of_many_rows_equals_the_general_form(dev, hd, nq, nkv, kv_bits, v_norm, B, W):
    """A workgroup per row (bf16 projections of many rows) against a wave per head, which the
    same projection given as one f32 slice takes: only the order of the norm's float32 sums differs, so
    a value may differ by one bf16 step (2^-7 of it) and a code by that step in units of its scale. Odd
    head counts, rows past the block table (dropped) and uneven lengths."""
    from mlx_dspark import ops
    from mlx_dspark.kv import PagedKVCache
    print(f"append hd={hd} nq={nq} nkv={nkv} kv_bits={kv_bits} v_norm={v_norm} B={B} W={W}", flush=True)
    g = torch.Generator(device=dev).manual_seed(hd + W)
    M, N = B * W, (nq + 2 * nkv) * hd
    qkv = (torch.randn(M, N, generator=g, device=dev) * 2).to(torch.bfloat16)
    gains = [(1 + 0.2 * torch.randn(hd, generator=g, device=dev)).to(torch.bfloat16) for _ in range(3)]
    inv = ops.rope_inv_freq(hd, 1e6, dev)
    outs = []
    for x in (qkv, qkv.float()[None]):
        cache = PagedKVCache(1, B, nkv, hd, 192, kv_bits=kv_bits)
        cache.set_lengths([(37 * b + 5) % 100 for b in range(B)])
        q = ops.qkv_rope_append(x.contiguous(), B, W, nq, nkv, hd, gains[0], gains[1], 1e-6, inv, cache.seq_lens,
                                cache.block_table, cache.page, cache.kv_dtype, *cache.layer_args(0),
                                v_norm=gains[2] if v_norm else None)
        kv = []
        for pool, sb in ((cache.k[0], cache.k_sb[0]), (cache.v[0], cache.v_sb[0])):
            if kv_bits:
                s, b = ((sb << 16).view(torch.float32)[..., None], (sb & -65536).view(torch.float32)[..., None])
                kv.append((pool.float().view(*sb.shape, 64) * s + b).view(pool.shape))
                kv.append(s.expand(*sb.shape, 64).reshape(pool.shape))
            else:
                kv += [pool.float(), torch.zeros_like(pool, dtype=torch.float32)]
        outs.append((q, kv))
    (qa, ka), (qb, kb) = outs
    if nq:
        assert bool(((qa.float() - qb.float()).abs() <= 2.0 ** -7 * qb.float().abs() + 2.0 ** -7).all())
        assert float((qa != qb).float().mean()) < 0.01
    for i in (0, 2):
        step = ka[i + 1].abs() + 2.0 ** -7 * kb[i].abs().amax(-1, keepdim=True)
        assert bool(((ka[i] - kb[i]).abs() <= step).all())
        assert float((ka[i] != kb[i]).float().mean()) < 0.02


@pytest.mark.parametrize("hd,nq,nkv,kv_bits,B,W", [
    (128, 32, 8, 8, 1, 4096), (128, 5, 1, None, 2, 515), (128, 0, 3, 8, 3, 200), (128, 0, 2, None, 1, 800),
    (128, 2, 1, 8, 1, 2048), (256, 16, 8, None, 1, 2048), (256, 2, 1, 8, 4, 131), (512, 3, 1, 8, 1, 700),
])
def test_append_of_many_rows_has_the_general_forms_bits(dev, hd, nq, nkv, kv_bits, B, W):
    """The norm's float32 sums are taken in the order of the wave-per-head form: the same queries, keys,
    values and scales, bit for bit (another order flips a few of a million roundings). Four heads and more,
    odd head counts, uneven lengths, rows past the block table."""
    from mlx_dspark import ops
    from mlx_dspark.kv import PagedKVCache
    print(f"append bits hd={hd} nq={nq} nkv={nkv} kv_bits={kv_bits} B={B} W={W}", flush=True)
    g = torch.Generator(device=dev).manual_seed(hd + W)
    qkv = (torch.randn(B * W, (nq + 2 * nkv) * hd, generator=g, device=dev) * 2).to(torch.bfloat16)
    gains = [(1 + 0.2 * torch.randn(hd, generator=g, device=dev)).to(torch.bfloat16) for _ in range(3)]
    inv = ops.rope_inv_freq(hd, 1e6, dev)
    outs = []
    for x in (qkv, qkv.float()[None]):
        cache = PagedKVCache(1, B, nkv, hd, W, kv_bits=kv_bits)
        cache.set_lengths([37 * b + 5 for b in range(B)])
        q = ops.qkv_rope_append(x.contiguous(), B, W, nq, nkv, hd, gains[0], gains[1], 1e-6, inv, cache.seq_lens,
                                cache.block_table, cache.page, cache.kv_dtype, *cache.layer_args(0), v_norm=gains[2])
        q = torch.zeros(0) if q is None else q
        outs.append([q] + [t for t in cache.layer_args(0) if t is not None])
    assert all(torch.equal(a, b) for a, b in zip(*outs))


@pytest.mark.parametrize("n,H", [(1, 64), (3, 1024), (130, 4096)])
def test_embed_in_whole_pieces_equals_the_general_form(dev, n, H):
    """16 codes per thread (aligned rows and outputs) against one element per thread (an output row
    stride that is no multiple of 8), bit for bit, with ids out of range."""
    from mlx_dspark.ops import W8Table, W8Weight, w8_embed
    g = torch.Generator(device=dev).manual_seed(n + H)
    t = W8Table(*W8Weight.quantize_mlx(torch.randn(50, H, generator=g, device=dev)))
    ids = torch.randint(0, 50, (n,), generator=g, device=dev, dtype=torch.int32)
    ids[-1] = 77
    odd = torch.zeros((n, H + 3), dtype=torch.bfloat16, device=dev)[:, :H]
    for scale in (1.0, 62.0):
        assert torch.equal(w8_embed(ids, t, scale), w8_embed(ids, t, scale, out=odd))
