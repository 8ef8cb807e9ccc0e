"""The timed choices of a dense GEMM and of gate|up (csrc/hb_select.cpp) over
a HIP runtime on host memory, whose launches write 1.0 into their output's
first element: what a choice leaves in the caller's buffers."""
import numpy as np
import pytest

import host_gpu

M, K, N = 256, 512, 256


@pytest.fixture(scope="module")
def hb(tmp_path_factory):
    mp = pytest.MonkeyPatch()
    mp.setenv("HB_CACHE_DIR", "")
    yield host_gpu.load(tmp_path_factory.mktemp("host"))
    mp.undo()


def test_choice_restores_its_output(hb):
    """Y (Out::Residual: every timed run adds into it) and state[3] after a
    choice, and gate|up's h, are what they were."""
    g = hb.Gpu(0)
    try:
        st = g.alloc_with(np.array([7, 8, 9, M], np.uint32))
        w, x, gu = g.alloc(2 * N * K * 2), g.alloc(M * K * 2), g.alloc(M * 2 * N * 2)
        y0 = np.arange(M * N, dtype=np.uint16)
        y, h = g.alloc_with(y0), g.alloc_with(y0)
        with hb.Engine(g, "") as e:
            e.gemm(K, N, hb.Out.Residual, hb.r(st), hb.r(w), hb.r(x), hb.r(y), M)
            e.gate_up(K, N, hb.r(st), hb.r(w), hb.r(x), hb.r(gu), hb.r(h), M)
            assert "[autotune] gemm %dx%d Residual, %d rows" % (K, N, M) in e.log() and "224 rows" in e.log()
        assert np.array_equal(g.download(y, np.uint16, M * N), y0)
        assert np.array_equal(g.download(h, np.uint16, M * N), y0)
        assert g.download(st, np.uint32, 4)[3] == M
    finally:
        g.close()


def test_output_that_cannot_be_read_stays(hb):
    """A choice that could not read Y before its runs fails and writes none
    of it."""
    g = hb.Gpu(0)
    try:
        st = g.alloc_with(np.array([7, 8, 9, M], np.uint32))
        w, x = g.alloc(N * K * 2), g.alloc(M * K * 2)
        y0 = np.arange(1, M * N + 1, dtype=np.uint16)
        y = g.alloc_with(y0)
        with hb.Engine(g, "") as e:
            hb.lib.fake_fail_reads(1)
            with pytest.raises(hb.HerbertError):
                e.gemm(K, N, hb.Out.Residual, hb.r(st), hb.r(w), hb.r(x), hb.r(y), M)
        hb.lib.fake_fail_reads(0)
        assert np.array_equal(g.download(y, np.uint16, M * N), y0)
    finally:
        g.close()
