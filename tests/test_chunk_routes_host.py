"""Which kernel forms silu(gate) * up of a chunk, on the CPU: the library's C
sources against the host-memory HIP stand-in, which records the launches. The
gate + up GEMM forms it itself on the 32 x 128 tile where the tile that the
GEMM alone would take has more workgroups than the 256 CUs, or where the FFN is
at least twice as wide as the model."""
from ctypes import byref, c_void_p

import numpy as np
import pytest

from test_failure_injection import P, _err, fake  # noqa: F401


@pytest.mark.parametrize("n_embd, n_ff, fused", [
    (256, 512, {2: True, 16: True, 64: True, 100: True}),
    (512, 512, {2: False, 16: False, 64: False, 100: False}),
    # 204 and 272 workgroups of 16 x 64, 204 of 32 x 64, 136 of 32 x 128 (picked by itself)
    (1280, 2176, {16: False, 48: False, 49: True, 64: True, 65: False, 100: True}),
    (512, 896, {64: False, 256: False}),
    (384, 768, {16: False})])                                            # K % 256 != 0: no such tile
def test_gate_up_kernel(amd, fake, n_embd, n_ff, fused):  # noqa: F811
    L = fake
    L.sllm_gfx950_close()
    L.fakehip_clear()
    assert L.sllm_gfx950_open(0) == 0
    model = amd.synth_model(dict(n_layer=1, n_embd=n_embd, n_ff=n_ff, n_head=n_embd // 64, n_head_kv=n_embd // 128,
                                 n_rot=64, n_vocab=100, eps=1e-5, rope_base=10000.0), 3)
    desc, keep = amd.model_desc(model)
    m, c = c_void_p(), c_void_p()
    assert L.sllm_gfx950_model_upload(byref(desc), byref(m)) == 0, _err(L)
    assert L.sllm_gfx950_ctx_new(m, 256, byref(c)) == 0, _err(L)
    tokens = np.zeros(256, np.int32)
    for n, want in fused.items():
        assert L.sllm_gfx950_ctx_reset(c) == 0
        L.fakehip_clear()
        assert L.sllm_gfx950_forward_chunk(m, c, P(tokens), n, 0, None) == 0, _err(L)
        assert any("_glu:" in e for e in L.fakehip_launches().decode().split()) == want, n
    L.sllm_gfx950_ctx_free(c)
    L.sllm_gfx950_model_free(m)
    del keep
