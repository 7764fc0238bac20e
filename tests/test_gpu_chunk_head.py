"""The chunk's output head at the edges of its 16-token and 64-row tiles:
every position's logits against the oracle's token path, bit for bit, with
an infinity, a NaN and subnormals in the embedding rows of some tokens."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CFG = dict(n_layer=1, n_ff=256, n_rot=64, eps=1e-5, rope_base=500000.0)


@pytest.mark.parametrize("n_embd", [128, 640])
@pytest.mark.parametrize("n_vocab,n", [(1, 2), (4, 15), (127, 16), (129, 17), (130, 33), (257, 2), (300, 48)])
def test_every_logit(amd, orc, dev, n_embd, n_vocab, n):
    print("[case] head", n_embd, n_vocab, n, flush=True)
    model = amd.synth_model(dict(CFG, n_embd=n_embd, n_vocab=n_vocab, n_head=n_embd // 64, n_head_kv=n_embd // 128), 7)
    e = model["tok_embd"].reshape(n_vocab, n_embd)
    e[n_vocab // 2, 1::7] = 0x0203                        # subnormals
    e[n_vocab - 1, 5] = 0x8001
    if n_vocab > 100:
        e[3, 9], e[70, 100] = 0x7C00, 0x7E01              # infinity, NaN: rows of no token below
    rng = np.random.default_rng(n_vocab + n)
    toks = rng.integers(100 if n_vocab > 100 else 0, n_vocab, n).astype(np.int32)
    g, o = amd.DeviceDecoder(dev, model, n + 1), orc.Decoder(model, n + 1)
    got = g.forward_chunk(toks, 0)
    want = np.stack([o.forward(int(t), i) for i, t in enumerate(toks)])
    g.close()
    o.close()
    nan = np.isnan(want)
    np.testing.assert_array_equal(np.isnan(got), nan)
    np.testing.assert_array_equal(got.view(np.uint32)[~nan], want.view(np.uint32)[~nan])


@pytest.mark.parametrize("norm", [2e-38, 1e-36])
def test_subnormal_products(amd, orc, dev, norm):
    """Normalised rows so small that the products with the embedding are
    subnormal f32, all of them and every sum, or some of them: a matrix
    instruction that flushed its inputs, products or sums would give other bits."""
    n_vocab, n = 130, 33
    model = amd.synth_model(dict(CFG, n_embd=640, n_vocab=n_vocab, n_head=10, n_head_kv=5), 8)
    model["output_norm"][:] = norm * np.linspace(0.5, 1.5, 640)
    e = model["tok_embd"].view(np.float16)
    e[:] = e / np.float16(1024)
    toks = np.random.default_rng(5).integers(0, n_vocab, n).astype(np.int32)
    g, o = amd.DeviceDecoder(dev, model, n), orc.Decoder(model, n)
    got = g.forward_chunk(toks, 0)
    want = np.stack([o.forward(int(t), i) for i, t in enumerate(toks)])
    g.close()
    o.close()
    low = np.abs(want) < 2.0 ** -126
    assert np.count_nonzero(want) > 0.9 * want.size and (low.all() if norm == 2e-38 else low.any())
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
