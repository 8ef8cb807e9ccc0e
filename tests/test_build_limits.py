"""Descriptors at the edges of what a workgroup holds, compiled for gfx950
without a GPU (hb_kernel_precompile): what the library accepts compiles, and
what it refuses it names."""
import ctypes

import pytest

import herbert_hip as hb


def precompile(d, monkeypatch):
    monkeypatch.setenv("HB_CACHE_DIR", "")
    hb.check(hb.lib.hb_kernel_precompile(ctypes.byref(d)))


@pytest.mark.parametrize("bm,bn,wm,wn", [(256, 288, 4, 3), (256, 320, 4, 2), (512, 256, 8, 2)])
def test_fused_swiglu_tiles_past_the_lds_epilogue(monkeypatch, bm, bn, wm, wn):
    """Dense fused tiles whose staged output is below and above 160 KiB of
    LDS: above it the gate and up sums pair in registers."""
    precompile(hb.gemm_mma_swiglu(256, 512, bm=bm, bn=bn, bk=32, wm=wm, wn=wn, mfma=16, dbuf=1, lds_dma=1), monkeypatch)


def test_fused_swiglu_tiles_that_pair_nowhere(monkeypatch):
    """Past that size an odd count of W fragments per wave and the ping-pong
    schedule, which pairs in LDS only, are refused by name."""
    with pytest.raises(hb.HerbertError, match="even count"):
        precompile(hb.gemm_mma_swiglu(256, 512, bm=512, bn=240, bk=32, wm=8, wn=1, mfma=16, lds_dma=1), monkeypatch)
    with pytest.raises(hb.HerbertError, match="output tile, beyond 160 KiB"):
        precompile(hb.gemm_mma_swiglu(256, 512, bm=256, bn=320, bk=32, wm=4, wn=2, mfma=16, dbuf=3, lds_dma=1, sched=1),
                   monkeypatch)


@pytest.mark.parametrize("d", [81664, 81920, 262144])
def test_rmsnorm_rows_past_lds(monkeypatch, d):
    """Rows that LDS holds, and longer ones, which it does not."""
    precompile(hb.rmsnorm(d, 1e-6, True), monkeypatch)
