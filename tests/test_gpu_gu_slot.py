"""The experts' gate/up on the matrix cores (k_gu_slot, 64 tokens and up)
against the oracle's block at the edges of its slots.  With a Q4_K down, which
stays on the chain kernels at these sizes, every operation of the block is the
oracle's and in its order, so the bound is equality.  The downs that sum their
16 to 32 block products a row on the matrix cores in an order of their own
(Q8_0, Q6_K) are held to 32 * 2^-24 = 2e-6 of a term: 1e-5 of the output's
RMS, which a gate/up rounding that moves a quant of the intermediate by a step
(about 1e-3) exceeds and a smaller one does not."""
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
SHAPES = [(512, 512), (1024, 512), (2048, 1024)]
TOKENS = (64, 65, 68, 69, 72, 73, 79)


@pytest.mark.parametrize("types", [(Q8_0, Q8_0, Q4K), (Q4K, Q4K, Q4K)])
@pytest.mark.parametrize("n_embd,n_ff", SHAPES)
def test_slot_bits(orc, engine, types, n_embd, n_ff):
    """Rows of zeros and of large and tiny values beside ordinary ones, the
    last row of a slot among them."""
    layer = synth.make_layer(32, n_embd=n_embd, n_expert=2, k=2, n_ff=n_ff, n_ff_sh=n_ff, types=types)
    moe = engine.moe(layer)
    for T in TOKENS:
        print(f"case bits {types} {n_embd} x {n_ff} T={T}", flush=True)
        h = synth.make_tokens(3100 + T, T, n_embd=n_embd)
        h[1] = 0.0
        h[2] *= np.float32(1e4)
        h[T - 2] *= np.float32(1e-3)
        h[T - 1] *= np.float32(1e-12)
        ref = orc.moe(layer, h, threads=8)
        got = moe.ffn(h)
        same = ref.view(np.uint32) == got.view(np.uint32)
        assert np.all(same), f"{np.mean(~same):.2e} of the outputs differ"


@pytest.mark.parametrize("types", [(Q8_0, Q8_0, Q8_0), (Q4K, Q4K, Q6K)])
@pytest.mark.parametrize("n_embd,n_ff", SHAPES)
def test_slot_remainders(orc, engine, types, n_embd, n_ff):
    layer = synth.make_layer(31, n_embd=n_embd, n_expert=2, k=2, n_ff=n_ff, n_ff_sh=n_ff, types=types)
    moe = engine.moe(layer)
    for T in TOKENS:
        print(f"case {types} {n_embd} x {n_ff} T={T}", flush=True)
        h = synth.make_tokens(3000 + T, T, n_embd=n_embd)
        ref = orc.moe(layer, h, threads=8)
        got = moe.ffn(h)
        rms = float(np.sqrt(np.mean(ref.astype(np.float64) ** 2)))
        assert np.abs(ref.astype(np.float64) - got).max() <= 1e-5 * rms
        assert np.array_equal(got.view(np.uint32), moe.ffn(h).view(np.uint32))
