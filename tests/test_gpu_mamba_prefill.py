"""A prompt through the Mamba decoder's row kernels against the same tokens
through its decode step, one at a time: the same bits (every value is the
step's float operations in its order), and the same state for the steps that
follow."""
import numpy as np
import pytest

import oracle as O
from synapse_amd import hip

pytestmark = pytest.mark.gpu

TINY = dict(d_model=64, d_inner=128, d_state=16, d_conv=4, dt_rank=8, n_layers=2, vocab=256)
RAGGED = dict(d_model=72, d_inner=136, d_state=16, d_conv=3, dt_rank=12, n_layers=3, vocab=301)
WIDE = dict(d_model=1024, d_inner=2048, d_state=16, d_conv=4, dt_rank=64, n_layers=2, vocab=512)
# a block of 512 tokens fills 256 tiles of 128 x 128 in in_proj
BROAD = dict(d_model=256, d_inner=4096, d_state=16, d_conv=4, dt_rank=32, n_layers=1, vocab=256)
# shapes the row kernels do not take: the token loop serves the prompt
SHORT_STATE = dict(TINY, d_state=8)


@pytest.fixture(scope="module", autouse=True)
def gpu():
    hip.init(0)


def _bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


# around the row kernels' edges: their smallest prompt, 16 and 17 rows (GEMV
# and GEMM), a block of 32 scanned tokens, the 64-row tile, a whole block of
# 512 tokens and one more
@pytest.mark.parametrize("cfg,lengths", [(TINY, (2, 3, 4, 5, 16, 17, 33, 65, 512, 513)),
                                         (RAGGED, (3, 16, 31, 32, 130)),
                                         (WIDE, (8, 64, 70)), (BROAD, (512,)),
                                         (SHORT_STATE, (5, 20))],
                         ids=["tiny", "ragged", "wide", "broad", "short_state"])
@pytest.mark.parametrize("xdt", [False, True], ids=["ref", "int8xdt"])
@pytest.mark.parametrize("fused", [True, False], ids=["fused", "unfused"])
def test_prompt_rows_equal_the_token_loop(cfg, lengths, xdt, fused):
    if xdt and fused and (cfg["d_state"], cfg["d_conv"]) != (16, 4):
        pytest.skip("the fused INT8 x/dt step takes d_state 16 and four taps only")
    g = hip.QuantizedMamba(dict(cfg, max_tokens=max(lengths) + 8), int8_xdt=xdt)
    g.init_synthetic(std=0.1)
    g.set_options(fused=fused, graph=True)
    ids = O.token_ids(max(lengths) + 3, 0x5EED0000 + 0xFFFF, cfg["vocab"])
    ids[1] = cfg["vocab"] + 5  # an id outside the vocabulary is a zero row
    for n in lengths:
        print("case", cfg, "int8_xdt", xdt, "fused", fused, "n", n, flush=True)
        want = g.prefill(ids[:1])
        for t in ids[1:n]:
            want = g.decode_one(int(t))
        after_w = [g.decode_one(int(t)) for t in ids[n:n + 3]]
        got = g.prefill(ids[:n])
        after = [g.decode_one(int(t)) for t in ids[n:n + 3]]
        np.testing.assert_array_equal(_bits(got), _bits(want), err_msg=f"n={n}")
        for a, b in zip(after, after_w):
            np.testing.assert_array_equal(_bits(a), _bits(b), err_msg=f"after n={n}")
    g.close()
