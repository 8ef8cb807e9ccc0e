"""The split-K workspace of a context (csrc/hb_runtime.cpp) where memory runs
out, on a HIP runtime over host memory: what the host allocates and which
kernels it launches with which pointers."""
import numpy as np
import pytest

import host_gpu

SPLIT = dict(bm=128, bn=128, bk=64, wm=2, wn=2, mfma=16, dbuf=1, lds_dma=1, order=1, ksplit=2)
NONE = 2**64 - 1
M, K, N = 512, 768, 8192   # a split kernel's slabs over M rows: 32 MiB
MB = 1 << 20


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    mp = pytest.MonkeyPatch()
    mp.setenv("HB_CACHE_DIR", "")
    yield host_gpu.load(tmp_path_factory.mktemp("host"))
    mp.undo()


class Rig:
    """A context with the operands of an M x K x N GEMM."""

    def __init__(self, hb):
        self.hb, self.lib = hb, hb.lib
        hb.lib.fake_limit(NONE)
        self.g = hb.Gpu(0)
        g = self.g
        self.st = g.alloc_with(np.array([0, 0, 0, M], np.uint32))
        self.bind = [hb.r(b) for b in (self.st, g.alloc(N * K * 2), g.alloc(M * K * 2), g.alloc(M * N * 2), self.st, self.st)]
        self.split, self.plain = hb.gemm_mma(K, N, 0, **SPLIT), hb.gemm_mma(K, N, 0, **dict(SPLIT, ksplit=0))
        self.ks, self.kp = g.pipeline(self.split), g.pipeline(self.plain)
        self.slab = N * 4 * 2  # bytes of both parts' slabs, a row

    def room(self, bytes_):
        """Memory for `bytes_` more."""
        self.lib.fake_limit(self.lib.fake_in_use() + bytes_)

    def launches(self, rows, kern):
        self.lib.fake_forget()
        self.g.launch(kern, self.bind, rows)
        return self.last()

    def last(self):
        return [self.lib.fake_launch_name(i).decode() for i in range(self.lib.fake_launches())]

    def slabs(self, i=0):
        """Bytes from launch i's slab pointer to the end of its allocation."""
        return self.lib.fake_launch_span(i, 3)


@pytest.fixture()
def rig(host):
    r = Rig(host)
    yield r
    r.lib.fake_limit(NONE)
    r.g.close()


def test_failed_growth_keeps_the_workspace(rig):
    """A launch whose slabs find no memory is refused; the workspace of
    earlier launches stays, and they run as before without allocating."""
    rig.launches(128, rig.ks)
    held = rig.lib.fake_in_use()
    rig.room(4 * MB)
    with pytest.raises(rig.hb.HerbertError, match="out of memory"):
        rig.g.launch(rig.ks, rig.bind, M)
    assert rig.lib.fake_in_use() == held
    rig.room(0)
    assert len(rig.launches(128, rig.ks)) == 2 and rig.slabs() >= 128 * rig.slab


def test_growth_that_fits_in_the_old_ones_place(rig):
    """Memory for the new workspace only once the old one is given back."""
    rig.launches(256, rig.ks)
    rig.room(M * rig.slab - 256 * rig.slab)
    assert len(rig.launches(M, rig.ks)) == 2 and rig.slabs() >= M * rig.slab


def text(rig, d):
    return "%s\t%s" % (rig.g.kernel_name(rig.g.pipeline(d)), " ".join(str(getattr(d, f)) for f in rig.hb._DESC_FIELDS))


def choice(rig, base, *by_rows, rows=M):
    """The handle of a pinned choice: `base`, and (rows, desc) below it."""
    line = "gemm\t%dx%d Bf16, %d rows\t%s" % (K, N, rows, text(rig, base))
    for at, d in by_rows:
        line += "\t%d\t%s" % (at, text(rig, d))
    with rig.hb.Engine(rig.g, "") as e:
        e.pin(line + "\n")
        return e.gemm(K, N, 0, *rig.bind[:4], rows)


def test_sequence_whose_later_op_finds_no_memory(rig):
    """A split kernel, then a choice whose growth fails: the choice falls back
    to its own kernel and the first op keeps slabs of the size it needs."""
    kern = choice(rig, rig.plain, (300, rig.split))
    ops = [rig.hb.Op(rig.ks, rig.bind, 128), rig.hb.Op(kern, rig.bind, 300)]
    rig.launches(128, rig.ks)
    rig.room(0)
    rig.lib.fake_forget()
    rig.g.time_ops(ops, 1)
    assert rig.last() == [rig.g.kernel_name(rig.ks), "gemm_splitk_%d_bf16_s2" % N, rig.g.kernel_name(rig.kp)]
    assert rig.slabs() >= 128 * rig.slab


@pytest.mark.parametrize("entry", ["time_ops", "graph"])
def test_sequence_that_lost_the_workspace_is_refused(rig, entry):
    """Where the growth for a later op leaves no workspace at all, the whole
    sequence is refused before anything is launched."""
    kern = choice(rig, rig.plain, (300, rig.split))
    ops = [rig.hb.Op(rig.ks, rig.bind, 128), rig.hb.Op(kern, rig.bind, 300)]
    rig.launches(128, rig.ks)
    rig.lib.fake_forget()
    rig.lib.fake_limit(0)
    with pytest.raises(rig.hb.HerbertError, match="workspace"):
        getattr(rig.g, entry)(ops)
    assert rig.last() == []


@pytest.mark.parametrize("swap", [False, True])
def test_first_launch_sizes_every_row_count(rig, swap):
    """Whichever of a choice's kernels splits K, its own or that of fewer
    rows: after a first launch at few rows and a graph, every row count up to
    the choice's runs the kernel chosen for it."""
    base, few = (rig.split, rig.plain) if swap else (rig.plain, rig.split)
    kern = choice(rig, base, (300, few))
    rig.launches(10, kern)
    gr = rig.g.graph([rig.hb.Op(rig.kp, rig.bind, M)])
    try:
        for rows, d in ((10, few), (300, few), (301, base), (M, base)):
            assert rig.launches(rows, kern)[0] == rig.g.kernel_name(rig.g.pipeline(d)), rows
            if d is rig.split:
                assert rig.slabs() >= rows * rig.slab
    finally:
        gr.free()


def test_refused_growth_is_not_tried_at_every_launch(rig):
    """A choice whose growth found no memory runs its own kernel without
    asking again, until memory is given back."""
    kern = choice(rig, rig.plain, (300, rig.split))
    spare = rig.g.alloc(32 * MB)
    rig.room(4 * MB)
    assert rig.launches(300, kern) == [rig.g.kernel_name(rig.kp)]
    tries = rig.lib.fake_malloc_tries()
    for _ in range(3):
        assert rig.launches(300, kern) == [rig.g.kernel_name(rig.kp)]
    rig.g.time_ops([rig.hb.Op(kern, rig.bind, 300)], 2)
    assert rig.lib.fake_malloc_tries() == tries
    rig.g.free(spare)
    assert rig.launches(300, kern)[0] == rig.g.kernel_name(rig.ks) and rig.slabs() >= 300 * rig.slab
