"""Large results on their way to host memory, on the CPU: the library's C
sources against the host-memory HIP stand-in. To pageable memory the copy goes
through pinned pieces and several threads; a failing call reaches the caller
as a status and leaves the copy usable; without pinned memory the plain copy
runs, and to memory that is pinned already; closing the library gives everything
back."""
from ctypes import POINTER, byref, c_float, c_size_t, c_void_p, cast

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
    # pinned by the caller: one plain copy, no event and no piece
    pin = c_void_p()
    assert L.hipHostMalloc(byref(pin), c_size_t(4 * N * VOCAB), 0) == 0
    for at in (0, 4096):
        rows = N if at == 0 else N - 1
        held = np.ctypeslib.as_array(cast(pin.value + at, POINTER(c_float)), (rows * VOCAB,))
        held.fill(7.0)
        assert L.sllm_gfx950_ctx_reset(c) == 0
        L.fakehip_fail(b"hipEventRecord", HIP_INVALID_VALUE, 0)
        assert L.sllm_gfx950_forward_chunk(m, c, P(tokens), rows, 0, pin.value + at) == 0, _err(L)
        assert not L.fakehip_fired() and not held.any()
        L.fakehip_clear()
    del held
    assert L.hipHostFree(pin) == 0
    # a runtime that cannot say what the memory is: staged, as pageable
    L.fakehip_fail(b"hipPointerGetAttributes", HIP_INVALID_VALUE, 0)
    assert chunk() == 0 and L.fakehip_fired() and not logits.any()
    L.fakehip_clear()
    L.sllm_gfx950_ctx_free(c)
    L.sllm_gfx950_model_free(m)
    L.sllm_gfx950_close()
    assert L.fakehip_live() == before
    del keep
