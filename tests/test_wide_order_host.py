"""Which kernels a GEMV of 7168 < K <= 16384 takes, on the CPU: the library's C
sources against the host-memory HIP stand-in (256 CUs), which records the
launches. The wide kernel is the better one while its workgroups are all
resident: at most one a CU, of about equal slabs, up to 136 MiB in all.
Where a call's jobs read what others (or they themselves) write, the wide
kernel's workgroups would read beside the writes; such a call keeps the
quantiser launch and the streaming kernel, which order them."""
from ctypes import byref, c_void_p

import numpy as np
import pytest

from test_failure_injection import _err, fake  # noqa: F401

K, N = 8192, 300
WIDE, SLAB, STREAM = "sllm_k_gemv_wide", "sllm_k_gemv_slab", "sllm_k_gemv_stream_l8"


CU, MAX_BYTES = 256, 256 * 544 * 1024


class Mem:
    """16-byte aligned stretches of one host array (the stand-in's device memory)."""

    def __init__(self):
        self.a = np.zeros(1 << 20, np.uint8)
        self.base = (self.a.ctypes.data + 255) & ~255

    def at(self, off):
        assert 0 <= off < (1 << 20) - 256
        return self.base + off


@pytest.fixture
def lib(fake):  # noqa: F811
    fake.sllm_gfx950_close()
    fake.fakehip_clear()
    assert fake.sllm_gfx950_open(0) == 0
    yield fake
    fake.fakehip_clear()


def _launches(L, call):
    L.fakehip_clear()
    assert call() == 0, _err(L)
    return [e.split(":")[0] for e in L.fakehip_launches().decode().split()]


def _wide_grid(L):
    """Workgroups of the last call's wide launch."""
    g = [int(e.split(":")[1]) for e in L.fakehip_launches().decode().split() if e.startswith(WIDE)]
    assert len(g) == 1
    return g[0]


def _batches(amd, L, jobs):
    """The same jobs as a batch, without allocations and as a plan."""
    arr = (amd.GemvJob * len(jobs))(*jobs)

    def plan():
        p = c_void_p()
        st = L.sllm_gfx950_plan_create(arr, len(jobs), byref(p))
        if st == 0:
            st = L.sllm_gfx950_plan_run(p)
            L.sllm_gfx950_plan_destroy(p)
        return st
    runs = [_launches(L, lambda: L.sllm_gfx950_gemv_batch(arr, len(jobs))),
            _launches(L, lambda: L.sllm_gfx950_gemv_batch_noalloc(arr, len(jobs))), _launches(L, plan)]
    assert runs[0] == runs[1] == runs[2]
    return runs[0]


# bytes of out ahead of x's end (or, negative, past it): apart, then overlapping by one value or wholly
@pytest.mark.parametrize("ahead, meets", [(0, False), (-16, False), (16, True), (4 * K, True), (4 * K + 4 * N - 16, True),
                                          (4 * K + 4 * N, False)])
def test_out_beside_and_over_x(amd, lib, ahead, meets):
    m = Mem()
    x, out = 65536, 65536 + 4 * K - ahead
    call = lambda: lib.sllm_gfx950_linear(m.at(400000), N, K, m.at(x), None, None, m.at(out))  # noqa: E731
    want = ["sllm_k_quant_act", STREAM] if meets else [WIDE]
    assert _launches(lib, call) == want
    job = amd.GemvJob(m.at(400000), N, K, m.at(x), None, None, None, m.at(out))     # raw dots
    assert _batches(amd, lib, [job]) == (["sllm_k_quant_list", STREAM] if meets else [WIDE])


def test_published_row_over_x(amd, lib):
    m = Mem()
    for q, act in ((65536, 0), (0, 65536 + 4 * K - 16)):
        call = lambda: lib.sllm_gfx950_linear(m.at(400000), N, K, m.at(65536), m.at(q), m.at(act), m.at(200000))  # noqa: E731,B023
        assert _launches(lib, call) == ["sllm_k_quant_act", STREAM]


def test_out_over_the_quantised_row(lib):
    m = Mem()
    for out, want in ((0, STREAM), (K, STREAM), (K + 16, WIDE)):            # q, act, behind both
        call = lambda: lib.sllm_gfx950_gemv_epilogue(m.at(400000), N, K, m.at(0), m.at(K), m.at(out))  # noqa: E731,B023
        assert _launches(lib, call) == [want]


def test_jobs_that_depend_on_each_other(amd, lib):
    m = Mem()
    w, x, q, act, o1, o2 = (m.at(v) for v in (400000, 0, 65536, 131072, 200000, 300000))
    publish = amd.GemvJob(w, N, K, x, q, act, o1, None)
    alone = amd.GemvJob(w, N, K, x, None, None, o2, None)
    takes = amd.GemvJob(w, N, K, None, q, act, o2, None)
    slab = amd.GemvJob(w, N, 2560, m.at(350000), None, None, o2, None)
    slab_takes = amd.GemvJob(w, N, 2560, None, q, act, o2, None)
    slab_over_x = amd.GemvJob(w, N, 2560, m.at(350000), None, None, x + 4 * 100, None)
    ordered = ["sllm_k_quant_list"]
    # no dependence: one row published by two jobs, one x for several
    assert _batches(amd, lib, [publish, alone]) == [WIDE]
    assert _batches(amd, lib, [publish, publish]) == [WIDE]
    assert _batches(amd, lib, [slab, publish]) == [SLAB, WIDE]
    # one job takes the row that another publishes
    for jobs in ([publish, takes], [takes, publish]):
        assert _batches(amd, lib, jobs) == ordered + [STREAM]
    # the slab launch runs ahead of the wide one
    assert _batches(amd, lib, [slab_takes, publish]) == ordered + [SLAB, STREAM]
    assert _batches(amd, lib, [publish, slab_over_x]) == ordered + [SLAB, STREAM]
    # one job's out over another's x
    assert _batches(amd, lib, [amd.GemvJob(w, N, K, x, None, None, o1, None),
                               amd.GemvJob(w, N, K, o1, None, None, o2, None)]) == ordered + [STREAM]


def test_job_without_rows_publishes_its_row(amd, lib):
    """No rows, but q / act to write: the quantiser launch writes them (the
    wide kernel would leave before it does)."""
    m = Mem()
    w, x, q, act, out = (m.at(v) for v in (400000, 0, 65536, 131072, 200000))
    assert _batches(amd, lib, [amd.GemvJob(w, 0, K, x, q, act, out, None)]) == ["sllm_k_quant_list"]
    assert _batches(amd, lib, [amd.GemvJob(w, 0, K, x, q, act, out, None),
                               amd.GemvJob(w, N, K, x, None, None, out, None)]) == ["sllm_k_quant_list", WIDE]


@pytest.mark.parametrize("k", [7296, 8192, 12416, 16384])
def test_single_tensor_sizes(amd, lib, k):
    """Up to 136 MiB; nothing is read here, so the weights' extent does not matter."""
    m = Mem()
    last = MAX_BYTES // (k // 4)
    for rows, want in ((1, [WIDE]), (last, [WIDE]), (last + 1, ["sllm_k_quant_act", STREAM])):
        call = lambda: lib.sllm_gfx950_linear(m.at(400000), rows, k, m.at(0), None, None, 1 << 40)  # noqa: E731,B023
        assert _launches(lib, call) == want
        if want == [WIDE]:
            assert _wide_grid(lib) <= CU


@pytest.mark.parametrize("shapes, wide", [
    ([(1, 8192)] * 256, True), ([(1, 8192)] * 257, False), ([(6510, 8192)] * 6, True), ([(300, 7296)] * 16, True),
    ([(4096, 14336), (1029, 8192), (16, 7296), (2500, 16384)], True), ([(300, 7296)] * 128, True),
    ([(314, 8192)] * 171, True), ([(385, 8192)] * 171, False), ([(17408, 16384)] * 2, True), ([(17409, 16384)] * 2, False),
    ([(20000, 8192)] + [(16, 8192)] * 200, False), ([(0, 8192)] * 300 + [(5, 8192)], True)])
def test_batches_are_resident_together(amd, lib, shapes, wide):
    m = Mem()
    jobs = [amd.GemvJob(m.at(400000), n, k, m.at(0), None, None, 1 << 40, None) for n, k in shapes]
    arr = (amd.GemvJob * len(jobs))(*jobs)
    got = _launches(lib, lambda: lib.sllm_gfx950_gemv_batch(arr, len(jobs)))
    assert [g for g in got if g != "sllm_k_quant_list"] == [WIDE if wide else STREAM]
    if wide:
        assert _wide_grid(lib) <= CU
    # from quantised rows the streaming kernel needs no launch ahead of it
    jobs = [amd.GemvJob(m.at(400000), n, k, None, m.at(0), None, None, 1 << 40) for n, k in shapes]
    arr = (amd.GemvJob * len(jobs))(*jobs)
    if shapes == [(314, 8192)] * 171:
        wide = False
    assert _launches(lib, lambda: lib.sllm_gfx950_gemv_batch(arr, len(jobs))) == [WIDE if wide else STREAM]


def test_static_array_takes_what_needs_no_rows(amd, lib):
    """300 rows of 8192 quantised values do not fit the static array; the wide
    kernel quantises in place. Where the order needs the rows, it is refused."""
    m = Mem()
    jobs = [amd.GemvJob(m.at(400000), 16, K, m.at(256 * i), None, None, (1 << 40) + 64 * i, None) for i in range(300)]
    arr = (amd.GemvJob * 300)(*jobs)
    assert _launches(lib, lambda: lib.sllm_gfx950_gemv_batch_noalloc(arr, 300)) == [WIDE]
    assert _launches(lib, lambda: lib.sllm_gfx950_gemv_batch(arr, 300)) == ["sllm_k_quant_list", STREAM]
    arr[7].out = m.at(512)
    assert lib.sllm_gfx950_gemv_batch_noalloc(arr, 300) == -36 and "the array holds" in _err(lib)
    assert _launches(lib, lambda: lib.sllm_gfx950_gemv_batch_noalloc(arr, 20)) == ["sllm_k_quant_list", STREAM]
