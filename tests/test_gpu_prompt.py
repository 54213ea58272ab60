"""Prompt batches (styx_amd/csrc/prompt.hip): styx_moe_generate runs every
prompt token but the last in batches on the matrix cores.  The K/V rows it
leaves and the logits after it are compared with the same tokens forwarded
one by one (the path the other engine tests hold to the oracle), and the
logits with the oracle itself.

Tolerance: every value is an f32 sum of at most 2048 products, whose order
differs between the two paths (forward error about sqrt(n) 2^-24 = 2.7e-6 of
the result's norm for random signs, and the same again through a second
layer), so 1e-5 relative L2."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import oracle_from_model, rel_l2

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
    assert (a.last_expert_ids().shape == b.last_expert_ids().shape)
    la = a.forward_token(int(toks[1]))
    b.forward_token(int(toks[0]))
    lb = b.forward_token(int(toks[1]))
    assert rel_l2(la, lb) < TOL
    if oracle:
        orc = oracle_from_model(b, n_ctx)
        for pos, t in enumerate([*prompt.tolist(), *toks.tolist()]):
            ol, *_ = orc.forward(pos, int(t))
        assert rel_l2(la, ol) < 1e-4
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
])
def test_types_and_shapes(gpu, kw):
    check(gpu, cfg(**kw), 40)


def test_several_batches_and_pages(gpu):
    """700 tokens: two batches, K/V rows over two pages of 512."""
    check(gpu, cfg(n_embd=256, n_ff_exp=256, n_expert=16), 700, oracle=False)


@pytest.mark.parametrize("budget,arena", [(0, True), (1, False)])
def test_host_experts(gpu, budget, arena):
    """Experts in pinned host memory, read in place by the batch."""
    check(gpu, cfg(), 40, expert_budget_mb=budget, arena=arena)


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
