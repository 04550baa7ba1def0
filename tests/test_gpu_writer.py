"""The GPU cache writers (kvb_write_paged) against the host writers: scatter_to_paged for f32/f16
and quantize_to_paged_i8 for int8 (the reference's src/reference.hpp:60-68 and
src/reference.cpp:32-51, whose host restatements are pinned bit for bit against the reference's
own code in the oracle tests). Every byte of the pool and every scale must come out as the host
writes them: live rows written, everything else left as it was."""
import ctypes

import numpy as np
import pytest

from conftest import progress

pytestmark = pytest.mark.gpu


def _bytes(a):
    return np.ascontiguousarray(a).view(np.uint8)


def _elems(a):
    """The array as unsigned integers of its element size (bitwise, NaNs included)."""
    a = np.ascontiguousarray(a)
    return a.view({1: np.uint8, 2: np.uint16, 4: np.uint32}[a.dtype.itemsize])


def check_writer(kvb, w, page, seed, pool_factor):
    want = kvb.PagedCache(w, page, seed, pool_factor=pool_factor, poison=True)
    plain = kvb.PagedCache(w, page, seed, pool_factor=pool_factor, poison=False)
    table = kvb.Buffer.from_array(want.table)
    lens = kvb.Buffer.from_array(w.lens)
    total = 0.0
    for src, pool_want, pool_plain, sc_want, sc_plain in (
            (w.k, want.k, plain.k, want.k_scale, plain.k_scale),
            (w.v, want.v, plain.v, want.v_scale, plain.v_scale)):
        # the pool before the write: the host result, with every live element (equal in the poisoned
        # and the plain pool) overwritten
        before = _elems(pool_want).copy()
        live = before == _elems(pool_plain)
        before[live] = 0x5A5A5A5A & np.iinfo(before.dtype).max
        contig = kvb.Buffer.from_array(src)
        paged = kvb.Buffer.from_array(before)
        scales = None
        if sc_want is not None:
            sc_before = _elems(sc_want).copy()
            sc_before[sc_before == _elems(sc_plain)] = 0x5A5A5A5A
            scales = kvb.Buffer.from_array(sc_before)
        total += kvb.write_paged(w, want, contig, paged, table, lens, scales)
        got = paged.download(before.dtype, before.size)
        bad = np.flatnonzero(got != _elems(pool_want).ravel())
        assert bad.size == 0, f"{bad.size} pool elements differ, first at {bad[:4]} (live: {live.ravel()[bad[:4]]})"
        if scales is not None:
            got_s = scales.download(np.uint32, sc_before.size)
            assert np.array_equal(got_s, _elems(sc_want).ravel()), "scales"
            scales.free()
        contig.free()
        paged.free()
    table.free()
    lens.free()
    return total, want


@pytest.mark.parametrize("kv", ["f32", "f16", "i8"])
@pytest.mark.parametrize("page", [1, 3, 16, 64])
def test_writer_matches_host_bytes(gpu, kv, page):
    kvb = gpu
    lens = [0, 1, 15, 16, 17, 63, 64, 65, 129, 300, 2, 0]
    w = kvb.Workload(kvb.Shape(len(lens), 8, 2, 64), kv, lens, seed=41, varied=(kv == "i8"))
    check_writer(kvb, w, page, page * 5 + 1, 2.0)


# One page around each limit of the quantiser's forms (a wave per block up to 2048 values, a workgroup
# with 8 and 16 registers up to 8192 and 16384, two passes past that) and pages that straddle the copy's
# 16 KB runs, with lengths around the runs' and the blocks' ends.
@pytest.mark.parametrize("kv,dim,page", [("i8", 64, 32), ("i8", 64, 33), ("i8", 128, 16), ("i8", 128, 17), ("i8", 128, 64),
                                         ("i8", 128, 65), ("i8", 128, 128), ("i8", 128, 129), ("f16", 128, 7),
                                         ("f16", 64, 100), ("f32", 128, 31), ("f32", 64, 200)])
def test_writer_form_limits(gpu, kv, dim, page):
    kvb = gpu
    lens = [page, 0, page + 1, 4 * page - 1, 31, 32, 33, 63, 65, 127, 128, 129, 257]
    w = kvb.Workload(kvb.Shape(len(lens), 4, 2, dim), kv, lens, seed=page, varied=(kv == "i8"))
    if kv == "i8":  # ties of the quantiser (scale 1/8), a zero block, and rows whose division is inexact
        w.k[0, 0] = ((np.arange(w.k[0, 0].size) % 253 - 126) / 16.0).reshape(w.k[0, 0].shape)
        w.k[0, 0, 0, 0] = 127 / 8.0
        w.k[0, 1] = 0.0
    check_writer(kvb, w, page, page + 3, 1.5)


@pytest.mark.parametrize("kv", ["f16", "i8"])
def test_writer_c5_shape(gpu, kv):
    """BASELINE c5's ragged batch (page 64, 3x pool, N(0,1)): the GPU-written pool and scales are the
    host's, byte for byte."""
    kvb = gpu
    lens = kvb.c5_lengths()
    w = kvb.Workload(kvb.Shape(len(lens), 32, 8, 128), kv, lens, seed=16384, q_amp=1.0, dist="normal", threads=16)
    ms, _ = check_writer(kvb, w, 64, 16384 * 131 + 64, 3.0)
    progress(f"[writer] c5 {kv}: K+V written in {ms * 1e3:.1f} us "
             f"({w.min_bytes() / (ms * 1e-3) / 1e9:.0f} GB/s of cache bytes)")


def test_writer_refusals_leave_the_pool(gpu):
    kvb = gpu
    w = kvb.Workload(kvb.Shape(2, 8, 2, 64), "i8", [32, 40], seed=3)
    c = kvb.PagedCache(w, 16, 1, poison=False)
    contig = kvb.Buffer.from_array(w.k)
    paged = kvb.Buffer(c.k.nbytes)
    paged.fill(0x33)
    table, lens = kvb.Buffer.from_array(c.table), kvb.Buffer.from_array(w.lens)
    with pytest.raises(kvb.KvbInvalidArgument):
        kvb.write_paged(w, c, contig, paged, table, lens, None)  # int8 without scales
    assert (paged.download(np.uint8, c.k.nbytes) == 0x33).all()
    for b in (contig, paged, table, lens):
        b.free()


# Both sides of the lines between the quantiser's forms that the number of blocks draws (a wave per block
# from 1024 blocks on, at the 256 CUs of an MI355X), and sequences that end long before their page does.
@pytest.mark.parametrize("dim,page,batch,length", [(128, 16, 31, 256), (128, 16, 32, 256), (64, 32, 33, 511),
                                                   (128, 1000, 2, 100), (64, 1000, 3, 300), (128, 200, 2, 230), (128, 140, 2, 129)])
@pytest.mark.parametrize("max_len", [0, 700])
def test_writer_block_counts(gpu, dim, page, batch, length, max_len):
    kvb = gpu
    lens = [length] * (batch - 1) + [length - 3]
    w = kvb.Workload(kvb.Shape(batch, 4, 2, dim), "i8", lens, seed=page + batch, varied=True)
    if max_len:  # a cache whose rows go on past the longest sequence
        pad = [(0, 0), (0, 0), (0, max_len - length), (0, 0)]
        w = kvb.Workload.from_arrays("i8", lens, w.q, np.pad(w.k, pad), np.pad(w.v, pad))
    check_writer(kvb, w, page, page + 3, 1.2)


@pytest.mark.parametrize("kv,batch", [("f16", 15), ("f16", 16), ("i8", 12), ("i8", 13)])
def test_writer_full_size_streams(gpu, kv, batch):
    """Calls either side of 128 MiB read and written, past which the rows are read with the streaming policy."""
    kvb = gpu
    per = 2048 * 8 * 128 * (4 if kv == "f16" else 5)
    assert (batch * per >= 128 << 20) == ((kv, batch) in (("f16", 16), ("i8", 13)))
    w = kvb.Workload(kvb.Shape(batch, 8, 8, 128), kv, [2048] * batch, seed=batch)
    check_writer(kvb, w, 64, batch, 1.0)
