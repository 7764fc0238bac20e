"""Large results on their way to pageable host memory, on the CPU: the
library's C sources against the host-memory HIP stand-in. The copy goes
through pinned pieces and several threads; a failing call reaches the caller
as a status and leaves the copy usable; without pinned memory the plain copy
runs; closing the library gives everything back."""
from ctypes import byref, c_void_p

import numpy as np

from test_failure_injection import HIP_INVALID_VALUE, HIP_OUT_OF_MEMORY, P, _err, fake  # noqa: F401

VOCAB, N = 65536, 37                     # 9.7 MB of logits: two pieces and a remainder


def test_staged_copy_statuses_and_release(amd, fake):  # noqa: F811
    L = fake
    L.sllm_gfx950_close()
    L.fakehip_clear()
    before = L.fakehip_live()
    assert L.sllm_gfx950_open(0) == 0
    model = amd.synth_model(dict(n_layer=1, n_embd=128, n_ff=128, n_head=2, n_head_kv=1, n_rot=64, n_vocab=VOCAB,
                                 eps=1e-5, rope_base=10000.0), 3)
    desc, keep = amd.model_desc(model)
    m, c = c_void_p(), c_void_p()
    assert L.sllm_gfx950_model_upload(byref(desc), byref(m)) == 0, _err(L)
    assert L.sllm_gfx950_ctx_new(m, N, byref(c)) == 0, _err(L)
    tokens = np.arange(N, dtype=np.int32)
    logits = np.empty(N * VOCAB, np.float32)

    def chunk():
        assert L.sllm_gfx950_ctx_reset(c) == 0
        logits.fill(7.0)
        return L.sllm_gfx950_forward_chunk(m, c, P(tokens), N, 0, P(logits))

    # no pinned memory: the plain copy
    L.fakehip_fail(b"hipHostMalloc", HIP_OUT_OF_MEMORY, 0)
    assert chunk() == 0 and L.fakehip_fired() and not logits.any()      # (the stand-in's kernels write nothing)
    L.fakehip_clear()
    assert chunk() == 0 and not logits.any()                            # staged
    live = L.fakehip_live()
    for call in (b"hipEventSynchronize", b"hipEventRecord"):
        for skip in (0, 2):
            assert L.sllm_gfx950_ctx_reset(c) == 0
            L.fakehip_fail(call, HIP_INVALID_VALUE, skip)
            assert chunk() == -61 and L.fakehip_fired(), (call, skip)
            L.fakehip_clear()
            assert chunk() == 0 and not logits.any()
            assert L.fakehip_live() == live
    L.sllm_gfx950_ctx_free(c)
    L.sllm_gfx950_model_free(m)
    L.sllm_gfx950_close()
    assert L.fakehip_live() == before
    del keep
