"""NaN and infinite inputs through every epilogue: the vector stores round by
v_cvt_pk_bf16_f32, which quiets a NaN and keeps its upper bits, the contract
by integer arithmetic (src/core/bf16.rs:13-23), which adds to them.  The two
agree on the NaNs that bf16 operands lead to (quiet, low 16 bits zero), so
each output has the bits of the integer form."""
import numpy as np
import pytest

import herbert_hip as hb
import hb_oracle as orc

pytestmark = pytest.mark.gpu

# quiet, signalling and payload NaNs of both signs, the infinities
SPECIAL = np.array([0x7FC0, 0xFFC0, 0x7FC1, 0x7F81, 0xFF81, 0x7FBF, 0x7FFF, 0xFFFF, 0x7F80, 0xFF80, 0xFFA5], np.uint16)
TILE = dict(bm=128, bn=128, bk=64, wm=2, wn=2, mfma=16, dbuf=1, lds_dma=1, order=1)
FORMS = {
    "lds": TILE, "registers": dict(TILE, lds_dma=0), "mfma32": dict(TILE, mfma=32), "split": dict(TILE, ksplit=2),
    "pp": dict(bm=256, bn=128, bk=32, wm=4, wn=2, mfma=16, dbuf=2, lds_dma=1, order=1, sched=1),
}


def integer_form(bits):
    """The contract's rounding on f32 bit patterns."""
    return ((bits + 0x7FFF + ((bits >> 16) & 1)) >> 16).astype(np.uint16)


def is_nan(h):
    return (h & 0x7FFF) > 0x7F80


@pytest.mark.parametrize("n", [256, 132])  # whole 16-byte output chunks, and not
@pytest.mark.parametrize("form", sorted(FORMS))
def test_gemm_nan_outputs(gpu, form, n):
    """Bf16 has the integer form's bits of the same kernel's F32 output, and
    its NaNs where the oracle has them; Residual keeps a NaN of y alone,
    quieted, and takes the sum's where that is one."""
    m, k = 96, 256
    x, w = hb.normal_bf16(1, 1.0, (m, k)), hb.normal_bf16(2, 0.02, (n, k))
    y0 = hb.normal_bf16(3, 1.0, (m, n))
    for i, s in enumerate(SPECIAL):
        x[2 * i, 37 * i % k] = w[3 * i + 1, 11 * i + 5] = s
        y0[30 + i] = s
    x[70, 3], x[70, 9] = 0x7F80, 0xFF80  # inf - inf
    w[:, 3] = w[:, 9] = 0x3C00
    bufs = [gpu.alloc_with(a) for a in (np.array([0, 0, 0, m], np.uint32), w, x)] + [gpu.alloc(m * n * 4)]
    st, W, X, Y = (hb.r(b) for b in bufs)
    got = {}
    try:
        for out in hb.Out.F32, hb.Out.Bf16, hb.Out.Residual:
            if out == hb.Out.Residual:
                gpu.upload(bufs[3], y0)
            gpu.launch(gpu.pipeline(hb.gemm_mma(k, n, out, **FORMS[form])), [st, W, X, Y, st, st], m)
            got[out] = gpu.download(bufs[3], np.uint32 if out == hb.Out.F32 else np.uint16, m * n).reshape(m, n)
    finally:
        for b in bufs:
            gpu.free(b)
    want = integer_form(got[hb.Out.F32])
    assert np.array_equal(is_nan(want), is_nan(orc.gemm(x, w))) and is_nan(want).any()
    assert np.array_equal(got[hb.Out.Bf16], want)
    res, y_nan, s_nan = got[hb.Out.Residual], is_nan(y0), is_nan(want)
    assert np.array_equal(res[y_nan & ~s_nan], (y0 | 0x0040)[y_nan & ~s_nan])
    assert np.array_equal(res[s_nan & ~y_nan], (want | 0x0040)[s_nan & ~y_nan])
    assert np.array_equal(is_nan(res), is_nan(orc.gemm(x, w, orc.OUT_RESIDUAL, y0)))


def test_row_kernels_nan_outputs(gpu):
    """RMSNorm, combine and moe_out give the oracle's bits with one NaN or
    infinity a row, and combine with two that meet as inf - inf."""
    d, rows, top_k = 512, 32, 4
    x, w = hb.normal_bf16(5, 2.0, (rows, d)), hb.normal_bf16(6, 0.1, (d,))
    y = hb.normal_bf16(9, 1.0, (rows * top_k, d))
    xn, ex, sh, xx = (hb.normal_bf16(s, 1.0, (rows, d)) for s in (14, 10, 11, 12))
    gate = hb.normal_bf16(13, 0.05, (d,))
    for i, s in enumerate(SPECIAL):
        x[i, 3 * i] = y[3 * i, 2 * i] = y[3 * i + 1, 2 * i + 1] = ex[i, 1] = sh[i, 2] = xx[i, 3] = xn[15 + i, 4] = s
        w[50 + i] = s if i % 2 else w[50 + i]
    y[40, 5], y[41, 5] = 0x7F80, 0xFF80
    x[:len(SPECIAL), 50:61] = 0x3F80
    route = np.zeros((rows, 2 * top_k), np.uint32)
    route[:, :top_k], route[:, top_k:] = np.arange(top_k), 0x3E800000

    def run(desc, arrays, out, n):
        bufs = [gpu.alloc_with(a) for a in arrays]
        try:
            gpu.launch(gpu.pipeline(desc), [hb.r(b) for b in bufs], n)
            return gpu.download(bufs[out], np.uint16, rows * d).reshape(rows, d)
        finally:
            for b in bufs:
                gpu.free(b)

    nowhere = np.zeros((rows, d), np.uint16)
    clean = np.array([i for i in range(rows) if i >= len(SPECIAL)])
    for p1 in (False, True):
        got, want = run(hb.rmsnorm(d, 1e-6, p1), [x, w, nowhere], 2, rows), orc.rmsnorm_rows(x, w, 1e-6, p1, 0)
        # where a row's NaN meets a weight's, which of the two is kept is not fixed
        both = np.zeros((rows, d), bool)
        both[:len(SPECIAL), 50:61] = True
        assert np.array_equal(got[~both], want[~both]) and np.array_equal(is_nan(got), is_nan(want))
        assert np.array_equal(got[clean], want[clean])
    got = run(hb.Desc(kind=hb.Kind.COMBINE, n=d, top_k=top_k), [y, route, nowhere], 2, rows)
    assert np.array_equal(got, orc.combine(y, route, top_k, d))
    got = run(hb.moe_out(d), [xn, gate, ex, sh, xx], 4, rows)
    assert np.array_equal(got, orc.moe_out(xn, gate, ex, sh, xx))
