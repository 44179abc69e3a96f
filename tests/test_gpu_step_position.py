"""Single decode steps between the other calls of a decoder: the position a
step is run at (known to the host from the call before, or read back after a
call that ends elsewhere) against the oracle's cache length and logits, and
for the recurrent decoders against the same tokens in one prompt."""
import numpy as np
import pytest

import oracle as O
from synapse_amd import hip
from tests.test_gpu_hybrid_prefill import BASE as HYBRID
from tests.test_gpu_mamba_prefill import TINY as MAMBA
from tests.test_gpu_speculative import KCFG, LLAMA_FMTS, MID, _bits, _cos, _ids, _pair, build_pair

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    hip.init(0)


# every call that moves the position, each followed by single steps
def _script(draft):
    yield "prefill", 9
    yield "one", 3
    yield "append", 4
    yield "one", 2
    yield "truncate", 6
    yield "one", 2
    yield "truncate", 90  # longer than the cache: no change
    yield "one", 1
    yield "speculative", 12
    yield "one", 2
    if draft:
        yield "draft", 2
        yield "one", 2
    yield "generate", 5
    yield "one", 2
    yield "prefill", 1
    yield "one", 2


@pytest.mark.parametrize("graph", [True, False])
@pytest.mark.parametrize("kind", ["int8", "kquant"])
def test_steps_between_other_calls_track_the_oracle(kind, graph):
    cfg = MID if kind == "int8" else KCFG
    o, g = _pair(MID, 0.15) if kind == "int8" else build_pair(KCFG, LLAMA_FMTS)
    g.set_options(graph=graph)

    def same(a, b, what):
        if kind == "int8":
            np.testing.assert_array_equal(_bits(a), _bits(b), err_msg=str(what))
        else:
            assert _cos(a, b) >= 0.9999, (what, _cos(a, b))

    for i, (op, n) in enumerate(_script(kind == "kquant")):
        ids = _ids(cfg, 16, i)
        if op == "prefill":
            same(g.prefill(ids[:n]), o.prefill(ids[:n]), (i, op))
        elif op == "append":
            same(g.prefill_append(ids[:n]), o.prefill_append(ids[:n]), (i, op))
        elif op == "truncate":
            o.truncate(n), g.truncate(n)
        elif op == "draft":
            for t in ids[:n]:
                same(g.forward_one_draft(int(t), 2), o.forward_one_draft(int(t), 2), (i, op))
        elif op == "speculative":
            o.generate_speculative(ids[:5], n, 2), g.generate_speculative(ids[:5], n, 2)
            # near ties may end the K-quant rounds at other lengths
            o.truncate(6), g.truncate(6)
        elif op == "generate":
            o.generate(ids[:5], n), g.generate(ids[:5], n)
            o.truncate(5), g.truncate(5)
        else:
            for t in ids[:n]:
                same(g.forward_one(int(t)), o.forward_one(int(t)), (i, op))
        assert g.cache_len() == o.cache_len(), (i, op)
    o.close()
    g.close()


@pytest.mark.parametrize("fused", [True, False])
def test_mamba_steps_between_other_calls(fused):
    g = hip.QuantizedMamba(dict(MAMBA, max_tokens=64))
    g.init_synthetic(std=0.1)
    g.set_options(fused=fused, graph=True)
    ids = O.token_ids(24, 0x5EED0000 + 0xFFFF, MAMBA["vocab"])
    want = [_bits(g.prefill(ids[:n])) for n in (3, 4, 5, 12, 13)]
    g.prefill(ids[:2])
    for n in (2, 3, 4):
        assert (_bits(g.decode_one(int(ids[n]))) == want[n - 2]).all(), n
    g.generate(ids[:7], 6)
    g.decode_timed(3)
    g.prefill(ids[:11])
    for n in (11, 12):
        assert (_bits(g.decode_one(int(ids[n]))) == want[n - 8]).all(), n
    g.prefill(ids[:1])
    for _ in range(62):  # the step limit is still where it was
        g.decode_one(1)
    with pytest.raises(hip.SynapseError):
        for _ in range(4):
            g.decode_one(1)
    g.close()


@pytest.mark.parametrize("fused", [True, False])
def test_hybrid_steps_between_other_calls(fused):
    g = hip.HybridLM(dict(HYBRID, max_seq=40))
    g.init_synthetic(std=0.06)
    g.set_options(fused=fused, graph=True)
    ids = O.token_ids(24, 0x5EED0000 + 0xFFFF, HYBRID["vocab"])
    for _ in range(2):
        g.reset()
        assert g.pos == 0
        got = [g.decode_one(int(t)) for t in ids[:2]]
        g.prefill(ids[2:6])
        got += [g.decode_one(int(t)) for t in ids[6:8]]
        assert g.pos == 8
        g.generate(ids[8:13], 4)
        assert g.pos == 16
        g.decode_timed(3)
        g.decode_one(int(ids[0]))
        assert g.pos == 20
        g.reset()
        got.append(g.prefill(ids[:7]))
        got.append(g.decode_one(int(ids[7])))
        assert g.pos == 8
        # the same tokens one at a time
        for a, b in ((got[2], got[4]), (got[3], got[5])):
            assert np.abs(a - b).max() <= 2e-5 * np.abs(b).max()
    for _ in range(32):
        g.decode_one(1)
    with pytest.raises(hip.SynapseError):
        g.decode_one(1)
    g.close()
