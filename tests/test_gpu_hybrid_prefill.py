"""A prompt through the hybrid decoder's row kernels against the same tokens
through its decode step, one at a time: logits of the prompt's end and of the
steps that follow.  Both sum in f32 in orders of their own (the step's residual
in 2^-32 fixed point); the bar is a tenth of the decoder's own bar against the
oracle (2e-4 of the largest logit)."""
import numpy as np
import pytest

import oracle as O
from perf import cases
from synapse_amd import hip

pytestmark = pytest.mark.gpu
TOL = 2e-5

BASE = dict(hidden=256, n_layers=4, vocab=640, n_heads=4, n_kv_heads=2, head_dim=64, inner=256,
            conv_kernel=3, inter=512, eps=1e-5, rope_theta=1e6, layer_kinds=[0, 1, 0, 1])
CASES = {
    "mixed": BASE,
    "conv_bias_taps4": dict(BASE, conv_kernel=4, conv_bias=1, layer_kinds=[0, 0, 1, 0]),
    "gqa_hd128": dict(BASE, n_layers=2, n_heads=2, n_kv_heads=1, head_dim=128,
                      layer_kinds=[1, 1]),
    "conv_only_wide": dict(BASE, n_layers=2, hidden=512, inner=768, inter=1280,
                           layer_kinds=[0, 0]),
}


@pytest.fixture(scope="module", autouse=True)
def gpu():
    hip.init(0)


def _rel(a, b):
    # (a zero row through conv layers alone gives zero logits)
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-20))


# the smallest prompt of the row kernels, one and two 32-row tiles and their
# neighbours, an odd and an even length (the conv state's halves)
@pytest.mark.parametrize("name", sorted(CASES))
def test_prompt_rows_match_the_token_loop(name):
    cfg = dict(CASES[name], max_seq=160)
    g = hip.HybridLM(cfg)
    g.init_synthetic(std=0.06)
    assert g.fused_active
    ids = O.token_ids(140, 0x5EED0000 + 0xFFFF, cfg["vocab"])
    ids[2] = cfg["vocab"] + 9  # an id outside the vocabulary is a zero row
    for n in (1, 2, 3, 4, 5, 31, 32, 33, 64, 65, 130):
        g.reset()
        for t in ids[:n]:
            want = g.decode_one(int(t))
        after_w = [g.decode_one(int(t)) for t in ids[n:n + 4]]
        g.reset()
        got = g.prefill(ids[:n])
        after = [g.decode_one(int(t)) for t in ids[n:n + 4]]
        worst = max(_rel(a, b) for a, b in zip([got] + after, [want] + after_w))
        print("case", name, "n", n, "worst", worst, flush=True)
        assert worst <= TOL, (n, worst)
        # a second prompt into the filled cache goes token by token
        if n == 5:
            g.reset()
            for t in ids[:9]:
                want = g.decode_one(int(t))
            g.reset()
            g.prefill(ids[:5])
            assert _rel(g.prefill(ids[5:9]), want) <= TOL
    g.close()


def test_generate_after_a_prompt_and_full_cache():
    cfg = dict(BASE, max_seq=48)
    g = hip.HybridLM(cfg)
    g.init_synthetic(std=0.06)
    ids = O.token_ids(33, 0x5EED0000 + 0xFFFF, cfg["vocab"])
    toks, margins = g.generate(ids, 8)
    g.reset()
    lg = g.prefill(ids)
    for t, mg in zip(toks, margins):
        top = np.sort(lg)[-2:]
        if top[1] - top[0] < 1e-3:
            break
        assert int(np.argmax(lg)) == int(t)
        assert abs(float(mg) - float(top[1] - top[0])) < 1e-3
        lg = g.decode_one(int(t))
    # a prompt longer than the cache fails as the token loop does
    g.reset()
    with pytest.raises(hip.SynapseError):
        g.prefill(O.token_ids(49, 1, cfg["vocab"]))
    g.close()


# the row products round nothing before their f32 sums and have no sum to cancel (the step takes
# 8 sum(x) off every block): their logits are less than half as far from float64 as the step's
@pytest.mark.parametrize("prompt", [9, 64])
def test_prompt_rows_error_against_float64(prompt):
    case = dict(kind="lm", model="hybrid", layers=4, vocab=32000, prompt=prompt, steps=0)
    state = cases.prepare(case, 1)
    lm, ids = state["lm"], state["ids"]
    want = cases.exact(case, 1)[0]
    rows = lm.prefill(ids)
    lm.reset()
    for t in ids:
        step = lm.decode_one(int(t))
    err = [float(np.linalg.norm(v - want) / np.linalg.norm(want)) for v in (rows, step)]
    print("prompt", prompt, "rows", err[0], "step", err[1], flush=True)
    assert err[0] <= 0.5 * err[1], err
    lm.close()


# the rows kernels' most tokens at once, then the rest of the prompt token by token
def test_prompt_past_the_rows_limit():
    cfg = dict(BASE, n_layers=2, layer_kinds=[0, 1], max_seq=2070)
    g = hip.HybridLM(cfg)
    g.init_synthetic(std=0.06)
    ids = O.token_ids(2052, 0x5EED0000 + 0xFFFF, cfg["vocab"])
    loop = [g.decode_one(int(t)) for t in ids]
    for n in (2047, 2048, 2049, 2051):
        g.reset()
        got = g.prefill(ids[:n])
        assert g.pos == n
        after = g.decode_one(int(ids[n]))
        worst = max(_rel(got, loop[n - 1]), _rel(after, loop[n]))
        print("n", n, "worst", worst, flush=True)
        assert worst <= TOL, (n, worst)
    for n in (2048, 2049):
        g.reset()
        toks, margins = g.generate(ids[:n], 1)
        top = np.sort(loop[n - 1])[-2:]
        assert top[1] - top[0] < 1e-3 or int(toks[0]) == int(np.argmax(loop[n - 1]))
        assert abs(float(margins[0]) - float(top[1] - top[0])) < 1e-3
    g.close()


# weights whose block scales reach 2^13 (standard deviation 3e4): the step's sums saturate, and a
# prompt follows it, token by token
def test_wide_block_scales_follow_the_step():
    cfg = dict(BASE, n_layers=2, layer_kinds=[0, 1], max_seq=40)
    g = hip.HybridLM(cfg)
    g.init_synthetic(std=3e4)
    ids = O.token_ids(12, 0x5EED0000 + 0xFFFF, cfg["vocab"])
    for t in ids:
        want = g.decode_one(int(t))
    g.reset()
    got = g.prefill(ids)
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
    g.close()
