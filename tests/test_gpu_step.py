"""biv_hip_moe_ffn_step, x += moe(rms_norm(x)), against the oracle at every
width: on both sides of the router launch's switches at 16/17 and 64/65 tokens,
and with the f16 quants of 64 tokens and up, to 256, where the pre-pass takes
over.
Every sum runs in the reference's order (from 64 tokens with a Q4_K down, which
stays on the chain kernels), so the bound is equality."""
import numpy as np
import pytest

from biv_amd import synth

pytestmark = pytest.mark.gpu

Q8_0, Q4K, Q6K, BF16 = synth.Q8_0, synth.Q4K, synth.Q6K, synth.BF16
EPS = 1e-6


@pytest.fixture(scope="module")
def engine():
    from biv_amd import hip
    e = hip.HipEngine(0)
    yield e
    e.close()


def inputs(n_embd, T):
    rng = np.random.default_rng(400 + T)
    w = (1.0 + 0.05 * rng.standard_normal(n_embd)).astype(np.float32)
    x = np.float32(3.0) * synth.make_tokens(500 + T, T, n_embd=n_embd, offsets=T > 1)
    return x, w


def step(engine, moe, x, w, shift=0):
    """The step with the norm weights `shift` floats into their buffer."""
    xd, nd = engine.malloc(x.nbytes), engine.malloc(w.nbytes + 16)
    try:
        engine.h2d(xd, x)
        engine.h2d(nd + 4 * shift, w)
        moe.ffn_step_device(xd, nd + 4 * shift, EPS, x.shape[0])
        return engine.d2h(np.empty_like(x), xd)
    finally:
        engine.free(xd)
        engine.free(nd)


@pytest.mark.parametrize("n_embd", [512, 1024, 2048])
def test_norm_alignment(engine, n_embd):
    """The norm weights at any float's address give the bits that they give
    at an aligned one."""
    moe = engine.moe(synth.make_layer(41, n_embd=n_embd, n_expert=8, k=2, n_ff=512, n_ff_sh=512))
    for T in (1, 5, 16, 17):
        x, w = inputs(n_embd, T)
        ref = step(engine, moe, x, w)
        for shift in (1, 2, 3):
            print(f"case norm_alignment {n_embd} T={T} shift={shift}", flush=True)
            assert np.array_equal(ref.view(np.uint32), step(engine, moe, x, w, shift).view(np.uint32))


def against_oracle(orc, engine, layer, n_embd, tokens):
    moe = engine.moe(layer)
    for T in tokens:
        print(f"case step {n_embd} T={T}", flush=True)
        x, w = inputs(n_embd, T)
        ref = x + orc.moe(layer, orc.rms_norm(x, w, EPS), threads=8)
        got = step(engine, moe, x, w)
        assert np.array_equal(ref.view(np.uint32), got.view(np.uint32)), np.mean(ref != got)


# 20 experts (and the gate row): the last row groups of a router launch are partial
@pytest.mark.parametrize("n_embd", [512, 1024, 2048])
@pytest.mark.parametrize("types", [(Q8_0, Q8_0, Q8_0), (Q4K, Q4K, Q6K), (BF16, BF16, BF16)])
@pytest.mark.parametrize("shared", [True, False])
def test_step_few_tokens(orc, engine, n_embd, types, shared):
    layer = synth.make_layer(42, n_embd=n_embd, n_expert=20, k=4, types=types, shared=shared)
    against_oracle(orc, engine, layer, n_embd, (1, 2, 3, 4, 6, 15, 16, 17, 33, 63))


# Q6_K gate/up, which stays on the chain kernels: no f16 quants
@pytest.mark.parametrize("n_embd", [512, 1024, 2048])
def test_step_chains(orc, engine, n_embd):
    layer = synth.make_layer(44, n_embd=n_embd, n_expert=20, k=4, types=(Q6K, Q6K, Q4K))
    against_oracle(orc, engine, layer, n_embd, (64, 65, 255, 256))


@pytest.mark.parametrize("n_embd", [512, 1024, 2048])
@pytest.mark.parametrize("types", [(Q8_0, Q8_0, Q4K), (Q4K, Q4K, Q4K)])
def test_step_f16_quants(orc, engine, n_embd, types):
    layer = synth.make_layer(43, n_embd=n_embd, n_expert=20, k=4, types=types)
    against_oracle(orc, engine, layer, n_embd, (64, 65, 255, 256))
