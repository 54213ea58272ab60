"""Prompt batches (styx_amd/csrc/prompt.hip): styx_moe_generate runs every
prompt token but the last in batches on the matrix cores.  The K/V rows it
leaves and the logits after it are compared with the same tokens forwarded
one by one (the path the other engine tests hold to the oracle), and the
logits with the oracle itself.

How exact the rows are is a test of its own, against 64-bit arithmetic of the
same model: no further off than the token-by-token path's.

Tolerance of the other tests: every value is an f32 sum of at most 2048 products, whose order
differs between the two paths (forward error about sqrt(n) 2^-24 = 2.7e-6 of
the result's norm for random signs, and the same again through a second
layer), so 1e-5 relative L2."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import model_hparams, oracle_from_model, rel_l2
from oracle import oracle as O

pytestmark = pytest.mark.gpu

TOL = 1e-5
Q8_0, Q4_K, Q5_K, Q6_K = 8, 12, 13, 14


@pytest.fixture(scope="module")
def gpu():
    from styx_amd import Gpu
    g = Gpu(0)
    yield g
    g.close()


def cfg(**kw):
    from styx_amd import SynthConfig
    base = dict(n_layers=2, n_embd=512, n_heads=4, n_kv_heads=2, head_dim=128, n_expert=32,
                n_expert_used=4, n_ff_exp=256, n_vocab=1024, exp_type=(Q4_K, Q5_K, Q6_K), seed=21)
    return SynthConfig(**{**base, **kw})


def check(gpu, c, n_prompt, oracle=True, n_ctx=None, **opts):
    """Prompt of n_prompt tokens through generate against token by token."""
    from styx_amd import MoeModel
    n_ctx = n_ctx or n_prompt + 8
    prompt = np.random.default_rng(n_prompt + c.seed).integers(0, c.n_vocab, n_prompt).astype(np.uint32)
    a, b = MoeModel.synth(gpu, c, n_ctx=n_ctx, **opts), MoeModel.synth(gpu, c, n_ctx=n_ctx, **opts)
    toks, _, _ = a.generate(prompt, 2)
    want = None
    for t in prompt:
        want = b.forward_token(int(t))
    from styx_amd.model import argmax_last
    assert toks[0] == argmax_last(want)
    for layer in range(c.n_layers):
        for x, y in zip(a.read_kv(layer, 0, n_prompt), b.read_kv(layer, 0, n_prompt)):
            assert rel_l2(x, y) < TOL, layer
            rows = np.linalg.norm(x - y, axis=1) / np.linalg.norm(y, axis=1)
            assert rows.max() < TOL, (layer, int(rows.argmax()))
    la = a.forward_token(int(toks[1]))
    b.forward_token(int(toks[0]))
    lb = b.forward_token(int(toks[1]))
    assert rel_l2(la, lb) < TOL
    if oracle:
        orc = oracle_from_model(b, n_ctx)
        for pos, t in enumerate([*prompt.tolist(), *toks.tolist()]):
            ol, _, _, margins = orc.forward(pos, int(t))
        assert rel_l2(la, ol) < 1e-4
        clear = np.asarray(margins) > 1e-4  # (layers that route without a doubt)
        assert np.array_equal(a.last_expert_ids()[clear], b.last_expert_ids()[clear])
    a.close()
    b.close()


def tensors64(m):
    out = {}
    for name in m.tensor_names():
        t, dims, data = m.export_tensor(name)
        a = data.view(np.float32) if t == 0 else O.dequant(t, data, int(np.prod(dims)))
        out[name] = a.astype(np.float64).reshape(dims[::-1])
    return out


def kv64(m, toks):
    """The first two layers' (K, V) rows of toks at positions 0.. in 64 bits,
    and each token's routing margin (k-th against k+1-th logit)."""
    hp, W, T = m.hp, tensors64(m), len(toks)
    nh, nkv, hd, k, half = hp.n_heads, hp.n_kv_heads, hp.head_dim, hp.n_expert_used, hp.head_dim // 2
    eps = float(np.float32(hp.rms_eps))
    norm = lambda x, w: x / np.sqrt((x * x).mean(-1, keepdims=True) + eps) * (1 if w is None else w)
    silu = lambda v: v / (1 + np.exp(-v))
    ang = np.arange(T)[:, None] * float(np.float32(hp.rope_base)) ** (-2.0 * np.arange(half) / hd)
    c, s = np.cos(ang)[:, None, :], np.sin(ang)[:, None, :]
    rope = lambda x: np.concatenate([x[..., :half] * c - x[..., half:] * s,
                                     x[..., :half] * s + x[..., half:] * c], -1)
    x = W["token_embd.weight"][toks]
    rows = []
    for l in range(2):
        w = lambda n: W.get(f"blk.{l}.{n}.weight")
        h = norm(x, w("attn_norm"))
        q, kk, v = ((h @ w(n).T).reshape(T, -1, hd) for n in ("attn_q", "attn_k", "attn_v"))
        if w("attn_q_norm") is not None:
            q = norm(q, w("attn_q_norm"))
        if w("attn_k_norm") is not None:
            kk = norm(kk, w("attn_k_norm"))
        q, kk = rope(q), rope(kk)
        rows.append((kk.reshape(T, -1), v.reshape(T, -1)))
        if l == 1:
            return rows, margin
        o = np.empty((T, nh, hd))
        for i in range(nh):
            sc = q[:, i] @ kk[:, i * nkv // nh].T / np.sqrt(hd)
            sc[np.triu_indices(T, 1)] = -np.inf
            p = np.exp(sc - sc.max(1, keepdims=True))
            o[:, i] = p / p.sum(1, keepdims=True) @ v[:, i * nkv // nh]
        x = x + o.reshape(T, -1) @ w("attn_output").T
        h = norm(x, w("ffn_norm"))
        lg = h @ w("ffn_gate_inp").T
        order = np.argsort(-lg, axis=1, kind="stable")
        top = np.take_along_axis(lg, order, 1)
        margin = top[:, k - 1] - top[:, k]
        p = np.exp(top[:, :k] - top[:, :1])
        p /= p.sum(1, keepdims=True)
        for e in range(hp.n_expert):
            t, sl = np.nonzero(order[:, :k] == e)
            g, u = h[t] @ w("ffn_gate_exps")[e].T, h[t] @ w("ffn_up_exps")[e].T
            x[t] += p[t, sl][:, None] * ((silu(g) * u) @ w("ffn_down_exps")[e].T)


BIG = dict(n_embd=1024, n_heads=32, n_kv_heads=4, n_expert=16, n_expert_used=8)


# each type's dense products in their few-token, four-wave and eight-wave (or
# two-row-tile) forms, and each type in each expert role with enough tokens
# for the latter; 800 and 1312 rows end inside a workgroup's 128; 8192
# columns are 32 steps of a workgroup
@pytest.mark.parametrize("kw,n", [
    *[(dict(attn_type=t), n) for t in (Q8_0, Q4_K, Q5_K, Q6_K) for n in (20, 70)],
    *[(dict(n_embd=8192, attn_type=t), 60) for t in (Q8_0, Q4_K, Q6_K)],
    *[(dict(BIG, attn_type=t, exp_type=e, n_ff_exp=f), 261) for t, e, f in (
        (Q8_0, (Q4_K, Q5_K, Q8_0), 800), (Q4_K, (Q6_K, Q4_K, Q8_0), 800), (Q5_K, (Q8_0, Q8_0, Q8_0), 1312),
        (Q6_K, (Q5_K, Q6_K, Q4_K), 768), (Q8_0, (Q5_K, Q4_K, Q5_K), 768), (Q8_0, (Q6_K, Q6_K, Q6_K), 768))],
])
def test_rows_as_exact_as_token_by_token(gpu, kw, n):
    """K/V rows against 64 bits: relative L2 at most 1.05 times that of the
    tokens forwarded one by one (the two differ only in roundings, so their
    ratio over 1e5 values moves by about 1%), and no bias: the mean error
    towards larger values within half an f32 rounding (2^-25)."""
    from styx_amd import MoeModel
    c = cfg(**kw)
    as_exact(*(MoeModel.synth(gpu, c, n_ctx=n + 8) for _ in range(2)), n)


def test_rows_with_an_outlier_as_exact(gpu, tmp_path):
    """One activation of a row 8192 times the others, and no weight on it or
    on its block of 32: the others keep 23 bits, each off by up to 2^-23 more
    than token by token, where a block of 32 has a scale of its own."""
    from styx_amd import MoeModel
    m = MoeModel.synth(gpu, cfg(), n_ctx=8)
    tensors = {n: m.export_tensor(n) for n in m.tensor_names()}
    tensors["blk.0.attn_norm.weight"][2].view(np.float32)[5] = 8192
    for n in ("attn_q", "attn_k", "attn_v"):
        blocks = tensors[f"blk.0.{n}.weight"][2].reshape(-1, 512 // 32, 34)
        blocks[:, 0, 2:] = 0
    path = write_model(tmp_path, m, tensors)
    m.close()
    as_exact(*(MoeModel.load(gpu, path, n_ctx=48) for _ in range(2)), 40, 2.0 ** -23 / 3 ** 0.5)


def write_model(tmp_path, m, tensors):
    from styx_amd import gguf_io
    path = tmp_path / "m.gguf"
    gguf_io.write(path, gguf_io.model_metadata(model_hparams(m)), [(n, t, d, b) for n, (t, d, b) in tensors.items()])
    return str(path)


def as_exact(a, b, n, more=0.0):
    toks = np.random.default_rng(n).integers(0, a.hp.n_vocab, n + 1).astype(np.uint32)
    a.generate(toks, 1)
    for t in toks:
        b.forward_token(int(t), False)
    ref, margin = kv64(b, toks[:n])
    for layer in (0, 1):
        sel = margin > 1e-4 if layer else slice(None)  # (tokens routed without a doubt)
        for x, y, r in zip(a.read_kv(layer, 0, n), b.read_kv(layer, 0, n), ref[layer]):
            x, y, r = (v.reshape(n, -1)[sel].astype(np.float64) for v in (x, y, r))
            assert rel_l2(x, r) <= np.hypot(1.05 * rel_l2(y, r), more), (layer, rel_l2(x, r), rel_l2(y, r))
            assert abs((np.sign(r) * (x - r)).mean()) <= 2.0 ** -25 * np.abs(r).mean(), layer
    a.close()
    b.close()


# batches around the tile sizes (16 and 32 tokens; the last prompt token is
# not in the batch), the shortest, and one past a second tile
@pytest.mark.parametrize("n", [5, 17, 18, 33, 34, 66])
def test_batch_lengths(gpu, n):
    check(gpu, cfg(), n)


@pytest.mark.parametrize("kw", [
    dict(exp_type=(Q8_0, Q8_0, Q8_0), n_ff_exp=96),            # rows of 3 q8_0 blocks
    dict(exp_type=(Q8_0, Q8_0, Q8_0), n_ff_exp=1312, n_embd=256),  # 41 blocks: a ragged last step
    dict(exp_type=(Q6_K, Q4_K, Q5_K), attn_type=Q6_K, embd_type=Q4_K, head_type=Q6_K),
    dict(exp_type=(Q5_K, Q6_K, Q4_K), attn_type=Q4_K, n_ff_exp=768, n_expert=16, n_expert_used=10),
    dict(n_heads=6, n_kv_heads=2, head_dim=64, n_embd=768),  # 3 heads per kv head, 12-block rows
    dict(attn_type=Q5_K),
    dict(n_heads=16, n_kv_heads=1, head_dim=64, n_embd=1024),                 # 16 heads per kv head
    dict(n_heads=2, n_kv_heads=2, head_dim=256),
    dict(n_ff_shexp=256), dict(n_ff_shexp=96, exp_type=(Q8_0, Q8_0, Q8_0)),   # shared expert
    dict(router_zipf_s=1.1),                                                  # router bias
    dict(embd_type=0), dict(embd_type=1),                                     # f32, f16 embeddings
])
def test_types_and_shapes(gpu, kw):
    check(gpu, cfg(**kw), 40)


def test_several_batches_and_pages(gpu):
    """700 tokens: two batches, K/V rows over two pages of 512."""
    check(gpu, cfg(n_embd=256, n_ff_exp=256, n_expert=16), 700, oracle=False)


@pytest.mark.parametrize("budget,arena", [(0, True), (1, False)])
def test_host_experts(gpu, budget, arena):
    """Experts in pinned host memory: every slab that the batch meets passes
    through its 64 MiB staging buffer."""
    check(gpu, cfg(), 40, expert_budget_mb=budget, arena=arena)


@pytest.mark.parametrize("kw", [
    # about 54 experts met, 40 slabs of 1.7 MB to the buffer: the others are read in place
    dict(n_embd=2048, n_ff_exp=768, n_expert=64, n_expert_used=8, exp_type=(Q8_0, Q8_0, Q8_0)),
    # slabs of 36 MB, one to the buffer, and of 71 MB, none
    dict(n_embd=8192, n_ff_exp=8192, n_expert=16, n_expert_used=2, exp_type=(Q4_K, Q4_K, Q8_0)),
])
def test_host_experts_past_the_staging_buffer(gpu, kw):
    from styx_amd import MoeModel
    m = MoeModel.synth(gpu, cfg(**kw), n_ctx=64, expert_budget_mb=0)
    toks = np.random.default_rng(2).integers(0, 1024, 41).astype(np.uint32)
    m.generate(toks, 1)
    batch = m.read_kv(1, 0, 40)
    m.reset()
    met = set()
    for t in toks:
        m.forward_token(int(t), False)
        met |= set(m.last_expert_ids()[0].tolist())
    assert len(met) > (64 << 20) // (kw["n_embd"] * kw["n_ff_exp"] // 32 * 34)
    for x, y in zip(batch, m.read_kv(1, 0, 40)):
        assert (np.linalg.norm(x - y, axis=1) < TOL * np.linalg.norm(y, axis=1)).all()
    m.close()


# 16 tokens a row tile, 2 tokens a row tile, keys in several chunks
@pytest.mark.parametrize("nh,nkv,past", [(4, 4, 0), (16, 2, 0), (4, 4, 900)])
def test_token_without_finite_values(gpu, tmp_path, nh, nkv, past):
    """A token whose embedding row is not finite: the rows of the tokens
    before it are what they are token by token, its own is not finite."""
    from styx_amd import MoeModel
    c = cfg(n_heads=nh, n_kv_heads=nkv, embd_type=1, seed=31)
    m = MoeModel.synth(gpu, c, n_ctx=32)
    tensors = {n: m.export_tensor(n) for n in m.tensor_names()}
    tensors["token_embd.weight"][2].view(np.uint16).reshape(c.n_vocab, c.n_embd)[7, 5] = 0x7C00  # inf
    path = write_model(tmp_path, m, tensors)
    m.close()
    toks = np.arange(100, 123, dtype=np.uint32)
    toks[12] = 7
    a, b = (MoeModel.load(gpu, path, n_ctx=past + 32) for _ in range(2))
    if past:
        a.fill_kv(past)
        b.fill_kv(past)
    a.generate(toks, 1)
    for t in toks:
        b.forward_token(int(t), False)
    for x, y in zip(a.read_kv(1, past, 22), b.read_kv(1, past, 22)):
        assert np.isfinite(y[:12]).all() and rel_l2(x[:12], y[:12]) < TOL
        assert not np.isfinite(x[12]).any() and not np.isfinite(y[12]).any()
    a.close()
    b.close()


def test_prompt_after_prompt(gpu):
    """A second prompt continues the context of the first."""
    from styx_amd import MoeModel
    c = cfg(seed=5)
    a, b = MoeModel.synth(gpu, c, n_ctx=96), MoeModel.synth(gpu, c, n_ctx=96)
    rng = np.random.default_rng(1)
    fed = []
    for n in (20, 37):
        p = rng.integers(0, c.n_vocab, n).astype(np.uint32)
        toks, _, _ = a.generate(p, 1)
        fed += p.tolist()
    for t in fed:
        want = b.forward_token(t)
    from styx_amd.model import argmax_last
    assert toks[0] == argmax_last(want)
    for x, y in zip(a.read_kv(1, 0, len(fed)), b.read_kv(1, 0, len(fed))):
        assert rel_l2(x, y) < TOL
    a.close()
    b.close()


# keys at the edge of the split (256), token tiles that end before the last
# chunk begins (2040 + 17 tokens), several chunks per workgroup pass
@pytest.mark.parametrize("hd,nh,nkv", [(64, 8, 8), (128, 32, 4), (256, 6, 2)])
@pytest.mark.parametrize("past,n", [(251, 6), (252, 6), (2040, 18), (4000, 5), (5000, 41)])
def test_short_prompt_on_a_long_context(gpu, hd, nh, nkv, past, n):
    from styx_amd import MoeModel
    c = cfg(n_heads=nh, n_kv_heads=nkv, head_dim=hd, n_embd=256, n_expert=16)
    toks = np.random.default_rng(past + n).integers(0, c.n_vocab, n).astype(np.uint32)
    a, b = (MoeModel.synth(gpu, c, n_ctx=past + n + 8) for _ in range(2))
    a.fill_kv(past)
    b.fill_kv(past)
    out, _, _ = a.generate(toks, 1)
    for t in toks:
        want = b.forward_token(int(t))
    from styx_amd.model import argmax_last
    assert out[0] == argmax_last(want)
    for x, y in zip(a.read_kv(1, past, n), b.read_kv(1, past, n)):
        rows = np.linalg.norm(x - y, axis=1) / np.linalg.norm(y, axis=1)
        assert rows.max() < TOL
    a.close()
    b.close()


def test_short_prompt_on_a_long_context_is_no_slower_than_its_tokens(gpu):
    """Five tokens (the shortest batch) on 32000 keys, medians of seven: well
    under half the time of the tokens one by one; with each row tile's keys
    walked by one workgroup it was 1.5 times."""
    import time
    from styx_amd import MoeModel
    n = 5
    m = MoeModel.synth(gpu, cfg(n_heads=32, n_kv_heads=4), n_ctx=32100)
    toks = np.arange(n, dtype=np.uint32)
    batch, single = [], []
    for _ in range(7):
        m.fill_kv(32000)
        t0 = time.perf_counter()
        m.generate(toks, 1)
        batch.append(time.perf_counter() - t0)
        m.fill_kv(32000)
        t0 = time.perf_counter()
        for t in toks:
            m.forward_token(int(t), False)
        single.append(time.perf_counter() - t0)
    m.close()
    print(f"{n} tokens: {1e6 * np.median(batch):.0f} us, one by one {1e6 * np.median(single):.0f} us")
    assert np.median(batch) < np.median(single)


def test_token_out_of_range_mid_prompt(gpu):
    """The tokens before it are forwarded, then the call fails, as it does
    token by token."""
    from styx_amd import MoeModel, StyxError
    c = cfg(seed=8)
    a, b = MoeModel.synth(gpu, c, n_ctx=32), MoeModel.synth(gpu, c, n_ctx=32)
    good = [3, 9, 27, 81, 243, 729, 11]
    with pytest.raises(StyxError, match="out of range"):
        a.generate(np.array(good + [c.n_vocab, 5], np.uint32), 1)
    for t in good:
        b.forward_token(t)
    la, lb = a.forward_token(7), b.forward_token(7)
    assert rel_l2(la, lb) < TOL
    a.close()
    b.close()
