"""The matrix-core kernel of the dense FFN (k_exact) against the oracle's
dense_ffn: every output carries the oracle's bits, at the edges of its tiles
(16, 32 and 64 input rows a workgroup, a last workgroup that holds fewer),
for every quantised type, from one chunk pair of a row up.  Its operations
and their order are the reference's, so the bound is equality."""
import numpy as np
import pytest

from biv_amd import synth

pytestmark = pytest.mark.gpu

Q8_0, Q4K, Q6K, BF16 = synth.Q8_0, synth.Q4K, synth.Q6K, synth.BF16


@pytest.fixture(scope="module")
def engine():
    from biv_amd import hip
    e = hip.HipEngine(0)
    yield e
    e.close()


def run(orc, engine, types, n_embd, n_ff, tokens, edit=None):
    layer = synth.make_dense(21, n_embd=n_embd, n_ff=n_ff, types=types)
    d = engine.dense(layer)
    g, u, dn = layer.gate, layer.up, layer.down
    for T in tokens:
        print(f"case {types} {n_embd} x {n_ff} T={T}", flush=True)
        h = synth.make_tokens(1000 + T, T, n_embd=n_embd)
        if edit:
            edit(h)
        ref = orc.dense_ffn(g.ty, g.data, u.ty, u.data, dn.ty, dn.data, n_embd, n_ff, h, threads=8)
        got = d.ffn(h)
        same = ref.view(np.uint32) == got.view(np.uint32)
        assert np.all(same | (np.isnan(ref) & np.isnan(got))), f"{np.mean(~same):.2e} of the outputs differ"
        x = synth.make_tokens(2000 + T, T, n_embd=n_embd)
        add = d.ffn(h, out=x.copy(), add=True)
        assert np.array_equal(add, x + ref, equal_nan=True)


# 16-row tiles (and the smallest rows, where Q8_0 takes the matvecs)
@pytest.mark.parametrize("types,n_embd,n_ff,tokens", [
    ((Q8_0, Q8_0, Q8_0), 2048, 2560, (15, 16)),
    ((Q4K, Q4K, Q6K), 1536, 2560, (7, 16)),
    ((Q6K, Q6K, Q4K), 512, 512, (7, 15, 16)),
    ((Q4K, Q4K, BF16), 512, 1024, (9,)),
    ((BF16, BF16, Q6K), 1024, 512, (9,)),
])
def test_exact_16(orc, engine, types, n_embd, n_ff, tokens):
    run(orc, engine, types, n_embd, n_ff, tokens)


@pytest.mark.parametrize("types,n_embd,n_ff,tokens", [
    ((Q8_0, Q8_0, Q8_0), 2048, 2560, (17, 32, 33, 48, 65)),
    ((Q8_0, Q8_0, Q8_0), 512, 2048, (73, 129)),
    ((Q4K, Q4K, Q6K), 1536, 2560, (17, 32, 33, 64)),
    ((Q6K, Q6K, Q4K), 512, 512, (17, 33, 50)),
])
def test_exact_32(orc, engine, types, n_embd, n_ff, tokens):
    run(orc, engine, types, n_embd, n_ff, tokens)


# enough output rows for 64-row tiles: the last of 36 (three tiles), 64, 8 and 32 rows
@pytest.mark.parametrize("types", [(Q8_0, Q8_0, Q8_0), (Q4K, Q4K, Q6K), (Q6K, Q6K, Q4K)])
@pytest.mark.parametrize("n_embd,n_ff,tokens", [(512, 16384, (100, 128, 200, 224)), (16384, 512, (100, 128))])
def test_exact_64(orc, engine, types, n_embd, n_ff, tokens):
    run(orc, engine, types, n_embd, n_ff, tokens)


# The edges of the rule that takes a half of the layer here (a matrix-core half
# beside a matvec one among them): the first token counts of Q4_K, and with
# 5120 rows on one side every tile of Q8_0's and Q6_K's gate/up and down from
# the first counts on
@pytest.mark.parametrize("types,n_embd,n_ff,tokens", [
    ((Q4K, Q4K, Q4K), 1024, 1536, (3, 4, 5, 6, 15, 17, 33)),
    ((Q8_0, Q8_0, Q8_0), 512, 5120, (5, 6, 7, 15, 17, 33, 49)),
    ((Q8_0, Q8_0, Q8_0), 5120, 1536, (14, 15, 16, 17, 32, 33, 49)),
    ((Q6K, Q6K, Q6K), 512, 5120, (5, 6, 16, 17, 33, 49)),
    ((Q6K, Q6K, Q6K), 5120, 1536, (7, 8, 16, 17, 33, 49)),
])
def test_exact_edges(orc, engine, types, n_embd, n_ff, tokens):
    run(orc, engine, types, n_embd, n_ff, tokens)


@pytest.mark.parametrize("types,T", [((Q8_0, Q8_0, Q8_0), 40), ((Q4K, Q4K, Q6K), 20)])
def test_exact_special_rows(orc, engine, types, T):
    """Rows of zeros, of huge and tiny values, and with an infinity or a NaN,
    beside ordinary ones.  (Q4_K's mins read the block sums, and the oracle
    sums a NaN's quant as C converts it, undefined, where Rust's `as` gives 0:
    no NaN there.)"""
    def edit(h):
        h[1] = 0.0
        h[2] *= np.float32(1e30)
        h[3] *= np.float32(1e-30)
        h[4, 5] = np.inf
        if types[0] == Q8_0:
            h[5, 7] = np.nan
    with np.errstate(all="ignore"):
        run(orc, engine, types, 2048, 1536, (T,), edit)


def test_scratch_limit(orc):
    """Where the f16 quants no longer fit the device and int8 ones do, the
    layer runs in the matvecs: the same bits, and nothing is left behind by the
    refused allocations; where neither fits, an error, after which smaller
    calls work."""
    from biv_amd import hip
    E = ff = 512
    T = 100_000
    f16 = T * (10 * E + 6 * ff + (E + ff) // 4)  # bytes of scratch
    int8 = f16 - T * (E + ff)
    layer = synth.make_dense(23, n_embd=E, n_ff=ff, types=(Q4K, Q4K, Q4K))
    h = synth.make_tokens(5, T, n_embd=E)
    outs = {}
    for room in (None, (f16 + int8) // 2, int8 // 2):
        with hip.HipEngine(0) as e, hip.HipEngine(0) as filler:
            d = e.dense(layer)
            hd, od = e.malloc(h.nbytes), e.malloc(h.nbytes)
            e.h2d(hd, h)
            d.forward_device(hd, 1, od)  # (code is loaded before the room is taken)
            e.sync()
            held = []
            if room:
                hole, size = filler.malloc(room), 8 << 30
                while size >= 8 << 20:
                    try:
                        held.append(filler.malloc(size))
                    except hip.HipError as err:
                        assert err.code == -4
                        size >>= 1
                filler.free(hole)
            print(f"case scratch_limit room={room} fills={len(held)}", flush=True)
            try:
                if room and room < int8:
                    with pytest.raises(hip.HipError) as err:
                        d.forward_device(hd, T, od)
                    assert err.value.code == -4
                    d.forward_device(hd, 40, od)
                else:
                    d.forward_device(hd, T, od)
                e.sync()
                outs[room] = e.d2h(np.empty_like(h), od)
            finally:
                for p in held:
                    filler.free(p)
                e.free(hd)
                e.free(od)
    full, mid, small = outs.values()
    assert np.array_equal(full.view(np.uint32), mid.view(np.uint32))
    assert np.array_equal(full[:40].view(np.uint32), small[:40].view(np.uint32))
    rows = [0, 1, 7, 8, T // 2, T - 1]
    g, u, dn = layer.gate, layer.up, layer.down
    ref = orc.dense_ffn(g.ty, g.data, u.ty, u.data, dn.ty, dn.data, E, ff, h[rows], threads=8)
    assert np.array_equal(ref.view(np.uint32), full[rows].view(np.uint32))
