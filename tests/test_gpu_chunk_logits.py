"""Chunks whose logits are large enough to reach the host in pinned pieces by
several threads: every row against the oracle's, bit for bit, at sizes on and
off the piece, into fresh memory each time, from two contexts in turn; and into
memory that is pinned already, which takes one copy."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CFG = dict(n_layer=1, n_embd=128, n_ff=256, n_head=2, n_head_kv=1, n_rot=64, eps=1e-5, rope_base=500000.0)


@pytest.mark.parametrize("n_vocab,n", [(32768, 64), (32769, 65), (30011, 100), (128256, 17)])
def test_large_logits(amd, orc, dev, n_vocab, n):
    print("[case] logits", n_vocab, n, flush=True)
    model = amd.synth_model(dict(CFG, n_vocab=n_vocab), 5)
    toks = np.random.default_rng(n).integers(0, n_vocab, n).astype(np.int32)
    o = orc.Decoder(model, n)
    want = np.stack([o.forward(int(t), i) for i, t in enumerate(toks)])
    o.close()
    gs = [amd.DeviceDecoder(dev, model, n) for _ in range(2)]
    got = [gs[0].forward_chunk(toks, 0), None]
    for g in gs:
        g.reset()
    np.testing.assert_array_equal(got[0].view(np.uint32), want.view(np.uint32))
    # one context after the other on this thread, the copies' buffers kept
    for i, g in enumerate(gs):
        got[i] = g.forward_chunk(toks, 0)
        np.testing.assert_array_equal(got[i].view(np.uint32), want.view(np.uint32))
        g.close()


def _hip():
    """The HIP runtime that the library is linked to, as loaded."""
    with open("/proc/self/maps") as f:
        return ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))


def test_large_logits_into_pinned_memory(amd, orc, dev):
    n_vocab, n = 32769, 65
    model = amd.synth_model(dict(CFG, n_vocab=n_vocab), 6)
    toks = np.random.default_rng(n).integers(0, n_vocab, n).astype(np.int32)
    o, g = orc.Decoder(model, n), amd.DeviceDecoder(dev, model, n)
    want = np.stack([o.forward(int(t), i) for i, t in enumerate(toks)])
    o.close()
    hip, pin, off = _hip(), ctypes.c_void_p(), 4100
    assert hip.hipHostMalloc(ctypes.byref(pin), ctypes.c_size_t(want.nbytes + off), 0) == 0
    try:
        assert amd.lib().sllm_gfx950_forward_chunk(g.m, g.c, amd.ptr(toks), n, 0, ctypes.c_void_p(pin.value + off)) == 0
        got = np.ctypeslib.as_array(ctypes.cast(pin.value + off, ctypes.POINTER(ctypes.c_uint32)), want.shape)
        np.testing.assert_array_equal(got, want.view(np.uint32))
    finally:
        g.close()
        assert hip.hipHostFree(pin) == 0
