"""Batched GEMM with K % 256 == 128 (a half last super-step) in every shape
the host picks by itself, at the edges of its tiles: int8 rows and outputs
against the oracle, dots against an integer matrix product. One block only
(K = 128), an even and an odd number of super-steps per K group, rows and
tokens on and off the tiles; the last token row and the last weight row end
their buffers."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [(m, n_rows, n) for m in (1, 16, 17, 64) for n_rows, n in ((1, 128), (65, 384), (200, 1408), (1000, 2688))]
CASES += [(64, 12290, 640), (65, 65, 128), (100, 1000, 1408), (256, 8192, 384), (257, 130, 6784), (300, 12290, 640),
          (300, 12290, 128), (513, 700, 896)]


@pytest.mark.parametrize("m,n_rows,n", CASES)
def test_half_super_step(amd, orc, dev, m, n_rows, n):
    print("[case] tail", m, n_rows, n, flush=True)
    seed = amd.synth_seed(13, n_rows & 0xFFFF, n & 0xFFFF, m)
    w = amd.synth_i2s(seed, n_rows, n)
    x = amd.synth_normal(seed ^ 5, m * n).reshape(m, n)
    q_o, s_o, t_o = orc.quant_act_rows(x)
    d_o = (q_o.astype(np.float32) @ amd.synth_codes(seed, n_rows, n).astype(np.float32).T).astype(np.int32)   # < 2^24: exact
    w_scale = np.frombuffer(w[n_rows * n // 4:n_rows * n // 4 + 4].tobytes(), np.float32)[0]
    y_o = (d_o - t_o[:, None]).astype(np.float32) * (w_scale / s_o)[:, None]
    bw, bx, bq, ba = dev.put(w), dev.put(x), dev.alloc(m * n), dev.alloc(8 * m)
    by, bd = dev.alloc(4 * m * n_rows), dev.alloc(4 * m * n_rows)
    dev.linear_batch(bw.vp, n_rows, n, bx.vp, m, bq.vp, ba.vp, by.vp, bd.vp)
    dev.sync()
    np.testing.assert_array_equal(bq.download(np.int8, m * n).reshape(m, n), q_o)
    np.testing.assert_array_equal(bd.download(np.int32, m * n_rows).reshape(m, n_rows), d_o)
    np.testing.assert_array_equal(by.download(np.uint32, m * n_rows), y_o.astype(np.float32).view(np.uint32).ravel())
    for b in (bw, bx, bq, ba, by, bd):
        b.free()
