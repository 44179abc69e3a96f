"""Prefill attention on the matrix cores: bits of the INT8 decoder against
the oracle over head widths and prompt lengths around 16-row blocks, partial
8x8 micro-tiles (rows and columns the reference computes without fused
multiply-add), the 256-position segments of the softmax and the longest prompt
whose scores fit LDS; rows appended at each start within a group of four
positions; and the tolerance form against the decode step's attention."""
import numpy as np
import pytest

import oracle as O
from synapse_amd import hip
from tests.test_gpu_speculative import KCFG, LLAMA_FMTS, _bits, _ids, _pair, build_pair

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    hip.init(0)


def _cfg(hd, max_seq):
    return dict(hidden=64, n_layers=2, n_heads=4, n_kv_heads=2, head_dim=hd, inter=64, vocab=128,
                max_seq=max_seq)


@pytest.mark.parametrize("hd", [16, 32, 64, 128])
def test_exact_bits_around_the_tiles(hd):
    cfg = _cfg(hd, 320)
    o, g = _pair(cfg, 0.25)
    for n in (1, 2, 7, 8, 9, 15, 16, 17, 23, 24, 25, 31, 32, 33, 40, 47, 49, 55, 57, 64, 79, 255,
              256, 257, 283, 303):
        print("hd", hd, "n", n, flush=True)
        ids = _ids(cfg, n)
        np.testing.assert_array_equal(_bits(g.prefill(ids)), _bits(o.prefill(ids)), err_msg=str(n))
        if n <= 57:  # appended rows attend among themselves, after n cached ones
            a = _ids(cfg, 27, n)
            np.testing.assert_array_equal(_bits(g.prefill_append(a)), _bits(o.prefill_append(a)),
                                          err_msg=f"append after {n}")
            t = int(ids[0])  # and the caches' rows are read back by a step
            np.testing.assert_array_equal(_bits(g.forward_one(t)), _bits(o.forward_one(t)))
    o.close()
    g.close()


# the longest prompt of the matrix-core kernel (rows of 1988 scores: 1985 tokens) and the
# per-row kernel from there on
@pytest.mark.parametrize("n", [1000, 1985, 1986])
def test_exact_bits_at_the_lds_limit(n):
    cfg = dict(_cfg(32, 2000), n_layers=1, n_heads=2, n_kv_heads=1)
    o, g = _pair(cfg, 0.25)
    ids = _ids(cfg, n)
    np.testing.assert_array_equal(_bits(g.prefill(ids)), _bits(o.prefill(ids)))
    o.close()
    g.close()


def test_tolerance_form_is_the_same_at_every_start():
    o, g = build_pair(KCFG, LLAMA_FMTS)
    for n in (5, 16, 21, 40):
        a = _ids(KCFG, n, 9)
        want = _bits(g.prefill(a))
        for c in range(1, 10):
            g.prefill(_ids(KCFG, c))
            np.testing.assert_array_equal(_bits(g.prefill_append(a)), want, err_msg=f"{n} at {c}")
    o.close()
    g.close()


# both sum in f32 in orders of their own; a tenth of the decoder's bar
# against the oracle (2e-4 of the largest logit)
@pytest.mark.parametrize("hd", [16, 32, 64, 128])
def test_tolerance_form_matches_the_step(hd):
    cfg = dict(hidden=256, n_layers=2, vocab=640, n_heads=4, n_kv_heads=2, head_dim=hd, inner=256,
               conv_kernel=3, inter=512, eps=1e-5, rope_theta=1e6, layer_kinds=[1, 1],
               max_seq=300)
    g = hip.HybridLM(cfg)
    g.init_synthetic(std=0.06)
    ids = O.token_ids(290, 0x5EED0000 + 0xFFFF, cfg["vocab"])
    want = [g.decode_one(int(t)) for t in ids]
    for n in (3, 15, 16, 17, 33, 64, 129, 257, 290):
        g.reset()
        got = g.prefill(ids[:n])
        err = float(np.abs(got - want[n - 1]).max() / np.abs(want[n - 1]).max())
        print("hd", hd, "n", n, err, flush=True)
        assert err <= 2e-5, (n, err)
    g.close()
