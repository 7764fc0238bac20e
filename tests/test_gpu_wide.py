"""GPU parity of the wide GEMV kernel (7168 < K <= 16384) at the edges of its
chunk counts and row groups, fused and from a quantised row, alone and in
plans beside the slab and streaming kernels: every output bit the oracle's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [7296, 8192, 8320, 12288, 12416, 14336, 16384, 16512])
@pytest.mark.parametrize("n_rows", [1, 15, 17, 4099])
def test_wide_linear_matches_oracle(amd, orc, dev, n_rows, n):
    print("[case] wide", n_rows, n, flush=True)
    w = amd.synth_i2s(amd.synth_seed(11, n_rows & 0xFFFF, n & 0xFFFF, 1), n_rows, n)
    x = amd.synth_normal(n_rows * 31 + n, n)
    y_o, q_o, d_o, s_o, t_o = orc.linear(w, n_rows, n, x, orc.DOT_V3)
    bw, bx, bq, ba = dev.put(w), dev.put(x), dev.alloc(n), dev.alloc(8)
    by, bd = dev.alloc(4 * n_rows), dev.alloc(4 * n_rows)
    for outputs in ((bq.vp, ba.vp), (None, None)):
        by.upload(np.full(n_rows, -7, np.float32))
        dev.linear(bw.vp, n_rows, n, bx.vp, *outputs, by.vp)
        dev.sync()
        np.testing.assert_array_equal(by.download(np.uint32, n_rows), y_o.view(np.uint32))
    np.testing.assert_array_equal(bq.download(np.int8, n), q_o)
    a = ba.download(np.uint8, 8).view(np.dtype([("scale", "<f4"), ("sum", "<i4")]))[0]
    assert a["scale"] == s_o and a["sum"] == t_o
    dev.gemv(bw.vp, n_rows, n, bq.vp, bd.vp)
    dev.gemv_epilogue(bw.vp, n_rows, n, bq.vp, ba.vp, by.vp)
    dev.sync()
    np.testing.assert_array_equal(bd.download(np.int32, n_rows), d_o)
    np.testing.assert_array_equal(by.download(np.uint32, n_rows), y_o.view(np.uint32))
    for b in (bw, bx, bq, ba, by, bd):
        b.free()


@pytest.mark.parametrize("slab_kib", [0, 32])
def test_plan_of_every_kernel(amd, orc, dev, slab_kib):
    """Slab, wide and streaming jobs in one plan, run twice."""
    shapes = [(300, 2560), (1029, 8192), (33, 20480), (4096, 14336), (16, 7296), (129, 6912), (2500, 16384)]
    bufs, jobs, want = [], [], []
    for i, (n_rows, n) in enumerate(shapes):
        w = amd.synth_i2s(amd.synth_seed(12, i, 0, 0), n_rows, n)
        x = amd.synth_normal(100 + i, n)
        want.append(orc.linear(w, n_rows, n, x, orc.DOT_V3))
        b = [dev.put(w), dev.put(x), dev.alloc(4 * n_rows), dev.alloc(n), dev.alloc(8)]
        bufs.append(b)
        q, act = (b[3].ptr, b[4].ptr) if i % 2 else (None, None)
        jobs.append(amd.GemvJob(b[0].ptr, n_rows, n, b[1].ptr, q, act, b[2].ptr, None))
    dev.set_tuning(slab_kib=slab_kib)
    try:
        plan = dev.plan(jobs)
        for _ in range(2):
            dev.plan_run(plan)
        dev.sync()
        dev.plan_destroy(plan)
    finally:
        dev.set_tuning()
    for i, ((n_rows, n), b, (y, q, _, _, _)) in enumerate(zip(shapes, bufs, want)):
        np.testing.assert_array_equal(b[2].download(np.uint32, n_rows), y.view(np.uint32), err_msg=f"job {i}")
        if i % 2:
            np.testing.assert_array_equal(b[3].download(np.int8, n), q, err_msg=f"job {i}")
        for v in b:
            v.free()


def test_outputs_over_inputs_are_ordered(amd, orc, dev):
    """out over its own x, and a job that takes the row another one publishes:
    what the quantiser launch and the streaming kernel make of them."""
    n_rows, n = 4099, 8192
    w = amd.synth_i2s(amd.synth_seed(13, 0, 0, 0), n_rows, n)
    x = amd.synth_normal(77, n)
    y_o, q_o, _, _, _ = orc.linear(w, n_rows, n, x, orc.DOT_V3)
    bw, bx, bq, ba, b1, b2 = dev.put(w), dev.put(x), dev.alloc(n), dev.alloc(8), dev.alloc(4 * n_rows), dev.alloc(4 * n_rows)
    try:
        dev.gemv_batch([amd.GemvJob(bw.ptr, n_rows, n, None, bq.ptr, ba.ptr, b2.ptr, None),
                        amd.GemvJob(bw.ptr, n_rows, n, bx.ptr, bq.ptr, ba.ptr, b1.ptr, None)])
        dev.linear(bw.vp, n_rows, n, bx.vp, None, None, bx.vp)
        dev.sync()
        np.testing.assert_array_equal(bq.download(np.int8, n), q_o)
        for b in (b1, b2, bx):
            np.testing.assert_array_equal(b.download(np.uint32, n_rows), y_o.view(np.uint32))
    finally:
        for b in (bw, bx, bq, ba, b1, b2):
            b.free()


def test_job_without_rows_publishes_its_row(amd, orc, dev):
    n = 8192
    w = amd.synth_i2s(amd.synth_seed(14, 0, 0, 0), 16, n)
    x = amd.synth_normal(78, n)
    _, q_o, _, s_o, t_o = orc.linear(w, 16, n, x, orc.DOT_V3)
    bufs = bw, bx, bq, ba, by = dev.put(w), dev.put(x), dev.put(np.full(n, 99, np.int8)), dev.alloc(8), dev.alloc(64)
    dev.gemv_batch([amd.GemvJob(bw.ptr, 0, n, bx.ptr, bq.ptr, ba.ptr, by.ptr, None)])
    np.testing.assert_array_equal(bq.download(np.int8, n), q_o)
    a = ba.download(np.uint8, 8).view(np.dtype([("scale", "<f4"), ("sum", "<i4")]))[0]
    assert a["scale"] == s_o and a["sum"] == t_o
    for b in bufs:
        b.free()
