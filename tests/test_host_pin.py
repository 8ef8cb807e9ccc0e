"""hb_engine_pin / hb_engine_picks (csrc/hb_select.cpp) over a HIP runtime on
host memory: which text a choice by rows may be read from."""
import numpy as np
import pytest

import host_gpu

TILE = dict(bm=128, bn=128, bk=64, wm=2, wn=2, mfma=16, dbuf=1, lds_dma=1, order=1)
M, K, N = 128, 1024, 512


@pytest.fixture(scope="module")
def hb(tmp_path_factory):
    mp = pytest.MonkeyPatch()
    mp.setenv("HB_CACHE_DIR", "")
    yield host_gpu.load(tmp_path_factory.mktemp("host"))
    mp.undo()


@pytest.fixture()
def g(hb):
    g = hb.Gpu(0)
    yield g
    g.close()


def text(hb, g, d):
    return "%s\t%s" % (g.kernel_name(g.pipeline(d)), " ".join(str(getattr(d, f)) for f in hb._DESC_FIELDS))


def gemm_line(hb, g, base, *by_rows, key="%dx%d Bf16, %d rows" % (K, N, M)):
    line = "gemm\t%s\t%s" % (key, text(hb, g, base))
    for rows, d in by_rows:
        line += "\t%s\t%s" % (rows, text(hb, g, d))
    return line + "\n"


@pytest.mark.parametrize("key,rows,ok", [("%dx%d Bf16, 128 rows" % (K, N), 128, True),
                                         ("%dx%d Bf16, 128 rows" % (K, N), 129, False),
                                         ("%dx%d Bf16, 128 rows" % (K, N), 4294967295, False),
                                         ("%dx%d Bf16" % (K, N), 96, False)])
def test_rows_within_the_choices_own(hb, g, key, rows, ok):
    """A range past the rows the choice was made at (they size the split-K
    workspace), or a choice that names none, is refused."""
    split = hb.gemm_mma(K, N, 0, **dict(TILE, ksplit=2))
    line = gemm_line(hb, g, hb.gemm_mma(K, N, 0, **TILE), (rows, split), key=key)
    with hb.Engine(g, "") as e:
        if ok:
            e.pin(line)
            assert "\t%d\t" % rows in e.picks()
        else:
            with pytest.raises(hb.HerbertError, match="rows %d" % rows):
                e.pin(line)


def swiglu_line(hb, g, base, *by_rows):
    line = "gate_up\t%dx%d, %d rows\t%s\t-\t-" % (K, 2 * N, M, text(hb, g, base))
    for rows, d in by_rows:
        line += "\t%d\t%s" % (rows, text(hb, g, d))
    return line + "\n"


def test_text_of_every_dense_kind_reads_back(hb, g):
    """A timed choice's candidates are tiles, split or not, and the direct
    forms; with a caller's also the VALU form: any of them may be chosen at
    any rows, and the text of such a choice pins and prints unchanged."""
    kinds = [hb.gemm_mma(K, N, 0, **TILE), hb.gemm_mma(K, N, 0, **dict(TILE, ksplit=2)),
             hb.gemm_mm2d(K, N, 0, 32, 16).replace(mfma=16), hb.gemm_simt(K, N, 0).replace(bm=64, bn=64)]
    for base in kinds:
        line = gemm_line(hb, g, base, *[(32 * (i + 1), d) for i, d in enumerate(kinds) if d is not base])
        with hb.Engine(g, "") as e:
            e.pin(line)
            assert e.picks() == line
    fused = hb.gemm_mma_swiglu(K, N, **TILE)
    line = swiglu_line(hb, g, fused, (64, hb.gemm_mma_swiglu(K, N, **dict(TILE, bm=64))))
    with hb.Engine(g, "") as e:
        e.pin(line)
        assert e.picks() == line


def test_text_of_other_kernels_is_refused(hb, g):
    """A kernel that reads other operands: grouped rows (the list and the tile
    table, which a dense launch has not), another shape or output, a fused
    SwiGLU for a GEMM and the reverse."""
    grouped = dict(TILE, rows_of=hb.Rows.Scatter, top_k=8, experts=64, tiles=80, rows_max=M)
    dense = hb.gemm_mma(K, N, 0, **TILE)
    fused = hb.gemm_mma_swiglu(K, N, **TILE)
    for base, other in [(dense, hb.Desc(kind=hb.Kind.GEMM, k=K, n=N, out=0, **grouped)), (dense, hb.gemm_mma(K, N + 64, 0, **TILE)),
                        (dense, hb.gemm_mma(K // 2, N, 0, **TILE)), (dense, hb.gemm_mma(K, N, hb.Out.F32, **TILE)),
                        (dense, fused), (hb.Desc(kind=hb.Kind.GEMM, k=K, n=N, out=0, **grouped), dense)]:
        with hb.Engine(g, "") as e, pytest.raises(hb.HerbertError, match="is no kernel of this choice"):
            e.pin(gemm_line(hb, g, base, (64, other)))
    for base, other in [(fused, dense), (fused, hb.gemm_mma_swiglu(K, N, **dict(grouped, rows_of=hb.Rows.Gather)))]:
        with hb.Engine(g, "") as e, pytest.raises(hb.HerbertError, match="is no kernel of this choice"):
            e.pin(swiglu_line(hb, g, base, (64, other)))


@pytest.mark.parametrize("rows", ["", "x", "99999999999999999999999"])
def test_experts_line_without_tile_rows_is_refused(hb, g, rows):
    """An experts line whose tile rows are no number is an error like any
    other line's."""
    line = "experts\tkey\t%s\t" % rows + "\t".join(["-", "-"] * 4) + "\n"
    with hb.Engine(g, "") as e, pytest.raises(hb.HerbertError, match="line 1: rows"):
        e.pin(line)
