"""The chunk's attention kernels where their tiles and row forms meet: head
widths on and off 16 dimensions, token counts on and off 16, prefixes that
put rows on both sides of 512, 1024 and 2048 positions. Every logit against
the oracle's token path, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _model(amd, n_embd, n_head, n_head_kv, n_rot, seed):
    return amd.synth_model(dict(n_layer=1, n_embd=n_embd, n_ff=256, n_head=n_head, n_head_kv=n_head_kv, n_rot=n_rot,
                                n_vocab=300, eps=1e-5, rope_base=500000.0), seed)


def _compare(got, want):
    nan = np.isnan(want)
    np.testing.assert_array_equal(np.isnan(got), nan)
    np.testing.assert_array_equal(got.view(np.uint32)[~nan], want.view(np.uint32)[~nan])


@pytest.mark.parametrize("n_embd,n_head,n_head_kv,n_rot", [(128, 16, 4, 8), (384, 16, 8, 16), (640, 16, 4, 40),
                                                           (384, 6, 2, 64), (512, 4, 1, 128)])
@pytest.mark.parametrize("n", [17, 129, 150])
def test_head_widths(amd, orc, dev, n_embd, n_head, n_head_kv, n_rot, n):
    """Head widths of 8, 24, 40, 64 and 128; one token's embedding holds a NaN,
    which reaches its own and later positions and no earlier one."""
    print("[case] widths", n_embd, n_head, n, flush=True)
    model = _model(amd, n_embd, n_head, n_head_kv, n_rot, 31)
    toks = np.random.default_rng(n).integers(1, 299, n).astype(np.int32)
    model["tok_embd"].reshape(300, n_embd)[299, 3] = 0x7E00
    toks[n - 5] = 299
    g, o = amd.DeviceDecoder(dev, model, n), orc.Decoder(model, n)
    got = g.forward_chunk(toks, 0)
    want = np.stack([o.forward(int(t), i) for i, t in enumerate(toks)])
    g.close()
    o.close()
    _compare(got[:n - 5], want[:n - 5])               # (the NaN row's own logits are NaN throughout)
    assert np.isnan(got[n - 5:]).all() and np.isnan(want[n - 5:]).all() and np.isfinite(got[:n - 5, :299]).all()


@pytest.mark.parametrize("base,n,n_ctx", [(380, 140, 520), (505, 130, 640), (1000, 133, 1135), (1990, 129, 2119),
                                          (2048, 145, 2200), (3000, 99, 3100), (4000, 120, 4125)])
def test_row_lengths(amd, orc, dev, base, n, n_ctx):
    print("[case] rows", base, n, flush=True)
    model = _model(amd, 128, 2, 1, 64, 32)
    toks = np.random.default_rng(base).integers(0, 300, n).astype(np.int32)
    rng = np.random.default_rng(base + 1)
    k, v = (rng.standard_normal((1, 1, base, 64)).astype(np.float32) for _ in range(2))
    g, o = amd.DeviceDecoder(dev, model, n_ctx), orc.Decoder(model, n_ctx)
    ok, ov = o.caches()
    ok[:, :, :base], ov[:, :, :base] = k, v
    g.kv_load(k, v, base)
    got = g.forward_chunk(toks, base)
    want = np.stack([o.forward(int(t), base + i) for i, t in enumerate(toks)])
    g.close()
    o.close()
    _compare(got, want)


@pytest.mark.parametrize("n", [33, 150])
def test_subnormal_values(amd, orc, dev, n):
    """Values so small that every p * v, and every sum of them, is a subnormal
    f32; the norm behind the attention, the quantiser and the output projection's
    scale bring them back to the residual's size, so a matrix instruction that
    flushed them would change the logits.
    (The scores have no such test: a product below 2^-126 moves no score, and so no
    exp, by anything that rounding keeps.)"""
    base, hd, e = 300, 64, 256
    model = _model(amd, e, 4, 2, 64, 33)
    layer = model["layers"][0]
    rows = 2 * hd
    at = rows * e // 4
    layer["wv"][at:at + 4] = np.frombuffer(np.float32(1e-40).tobytes(), np.uint8)      # the tensors' scales
    layer["wo"][e * e // 4:e * e // 4 + 4] = np.frombuffer(np.float32(1e32).tobytes(), np.uint8)
    layer["attn_sub_norm"][:] *= np.float32(1e4)
    toks = np.random.default_rng(n).integers(0, 300, n).astype(np.int32)
    rng = np.random.default_rng(n + 1)
    k, v = (rng.standard_normal((1, 2, base, hd)).astype(np.float32) for _ in range(2))
    v = (v.astype(np.float64) * 2e-39).astype(np.float32)
    g, o = amd.DeviceDecoder(dev, model, base + n), orc.Decoder(model, base + n)
    ok, ov = o.caches()
    ok[:, :, :base], ov[:, :, :base] = k, v
    g.kv_load(k, v, base)
    got = g.forward_chunk(toks, base)
    want = np.stack([o.forward(int(t), base + i) for i, t in enumerate(toks)])
    flushed = orc.Decoder(model, base + n)               # no values at all: other logits
    fk, _ = flushed.caches()
    fk[:, :, :base] = k
    assert not np.array_equal(flushed.forward(int(toks[0]), base), want[0])
    for d in (g, o, flushed):
        d.close()
    _compare(got, want)
