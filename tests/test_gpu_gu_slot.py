"""The experts' gate/up on the matrix cores (k_gu_slot, 64 tokens and up)
against the oracle's block at the edges of its slots.  The kernel keeps the
oracle's bits, and a difference in them would move a quant of the intermediate
by a step (about 1e-3 of the output's RMS); down sums its 16 to 32 block
products a row in 32 bits in an order of its own: 32 * 2^-24 = 2e-6 of a term,
so 1e-5 of the RMS is the bound."""
import numpy as np
import pytest

from biv_amd import synth

pytestmark = pytest.mark.gpu

Q8_0, Q4K, Q6K = synth.Q8_0, synth.Q4K, synth.Q6K


@pytest.fixture(scope="module")
def engine():
    from biv_amd import hip
    e = hip.HipEngine(0)
    yield e
    e.close()


# tokens per expert: k = n_expert routes every token to every expert, so the
# slots hold 16, ..., 16 and a remainder of T % 16 pairs
@pytest.mark.parametrize("types", [(Q8_0, Q8_0, Q8_0), (Q4K, Q4K, Q6K)])
@pytest.mark.parametrize("n_embd,n_ff", [(512, 512), (1024, 512), (2048, 1024)])
def test_slot_remainders(orc, engine, types, n_embd, n_ff):
    layer = synth.make_layer(31, n_embd=n_embd, n_expert=2, k=2, n_ff=n_ff, n_ff_sh=n_ff, types=types)
    moe = engine.moe(layer)
    for T in (64, 65, 68, 69, 72, 73, 79):
        print(f"case {types} {n_embd} x {n_ff} T={T}", flush=True)
        h = synth.make_tokens(3000 + T, T, n_embd=n_embd)
        ref = orc.moe(layer, h, threads=8)
        got = moe.ffn(h)
        rms = float(np.sqrt(np.mean(ref.astype(np.float64) ** 2)))
        assert np.abs(ref.astype(np.float64) - got).max() <= 1e-5 * rms
        assert np.array_equal(got.view(np.uint32), moe.ffn(h).view(np.uint32))
