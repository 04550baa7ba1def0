"""The three-pass baseline at the edges of its layout: lengths around a 128-token chunk and many
chunks, groups below, at and past the 8 heads of one sweep, both head dims and storage types, against
the oracle's fp64 attention; rows past a sequence's end must not reach it, whatever they hold."""
import ctypes

import numpy as np
import pytest

from conftest import progress

pytestmark = pytest.mark.gpu

# heads, KV heads, head_dim, lengths
CASES = [
    (4, 4, 128, [1, 127, 128, 129]),
    (6, 2, 64, [0, 63, 256, 257]),
    (16, 2, 128, [385, 2]),
    (9, 1, 64, [130, 16]),          # 8 heads, then one
    (24, 2, 128, [500]),            # 8 and 4
    (8, 2, 64, [17 * 128 + 5, 3]),  # past the 16 chunks one round trip of the last pass loads
]


@pytest.mark.parametrize("kv", ["f32", "f16"])
@pytest.mark.parametrize("heads,kv_heads,dim,lens", CASES)
def test_naive_edges(gpu, oracle, kv, heads, kv_heads, dim, lens):
    kvb = gpu
    w = kvb.Workload(kvb.Shape(len(lens), heads, kv_heads, dim), kv, lens, seed=sum(lens) + heads)
    want = oracle.attention(w.shape, w.lens, w.max_len, w.q, w.k, w.v)
    for b, n in enumerate(lens):  # the rows past the end: not read as data
        w.k[b, :, n:] = np.nan
        w.v[b, :, n:] = np.nan
    bufs = [kvb.Buffer.from_array(x) for x in (w.q, w.k, w.v, w.lens)]
    out = kvb.Buffer(w.out_floats() * 4)
    out.fill(0xFF)
    kvb.run_naive(w, out, *bufs)
    got = out.download(np.float32, w.q.shape)
    # |v| < 1 and the weights sum to 1: the fp32 error of a score of |s| <= 3 sqrt(D) is below
    # 2^-24 * 4 * 34 = 8e-6 and moves the output by at most twice that; the sums add 1e-6
    err = oracle.max_abs_diff(got, want)
    assert err <= 2e-5, err
    progress(f"[naive] {heads}/{kv_heads} D{dim} {kv} lens {lens}: max err {err:.3g}")


@pytest.mark.parametrize("kv", ["f32", "f16"])
@pytest.mark.parametrize("dim,heads,kv_heads", [(64, 4, 2), (128, 9, 1)])
def test_naive_takes_elements_at_any_offset(gpu, oracle, kv, dim, heads, kv_heads):
    """q and V are read as elements: a program may pass any slice of a larger buffer (K's rows are read in
    16-byte words, as they always were)."""
    kvb = gpu
    lens = [129, 40]
    w = kvb.Workload(kvb.Shape(2, heads, kv_heads, dim), kv, lens, seed=dim + heads)
    want = oracle.attention(w.shape, w.lens, w.max_len, w.q, w.k, w.v)

    def shifted(a):
        pad = np.zeros(a.size + 1, a.dtype)
        pad[1:] = a.ravel()
        return kvb.Buffer.from_array(pad), a.dtype.itemsize

    (q, q_off), (v, v_off) = shifted(w.q), shifted(w.v)
    k, lens_buf, out = kvb.Buffer.from_array(w.k), kvb.Buffer.from_array(w.lens), kvb.Buffer(w.out_floats() * 4)
    a = kvb.NaiveArgsC()
    a.batch, a.num_heads, a.num_kv_heads, a.head_dim = 2, heads, kv_heads, dim
    a.kv_type, a.max_len = w.kv_type, w.max_len
    a.q, a.k, a.v, a.seq_lens, a.out = q.ptr + q_off, k.ptr, v.ptr + v_off, lens_buf.ptr, out.ptr
    a.host_seq_lens = w.lens.ctypes.data
    ms = ctypes.c_double()
    kvb.check(kvb.hip.kvb_run_naive(ctypes.byref(a), ctypes.byref(ms)), "run_naive")
    err = oracle.max_abs_diff(out.download(np.float32, w.q.shape), want)
    assert err <= 2e-5, err  # (as above)
