"""Steps whose partition the caller leaves to the library (part_tokens 0): every sequence is cut evenly,
into fewer and larger partitions than kvb_auto_part_tokens gives. Against the oracle, at the edges of the
cut (a token either side of a partition, one token, empty, many partitions, batches past the ragged
order's limit); the fused step, the two-kernel step, a captured graph and the static-scratch step agree
bit for bit, and a workspace of the caller's still gets the nominal partition's slots."""
import ctypes

import numpy as np
import pytest

import parity_battery as pb
from conftest import progress

pytestmark = pytest.mark.gpu

# (H, Hkv, D), lengths, page
CASES = [
    ((8, 2, 64), [128, 129, 127, 1, 0, 256, 257], 16),
    ((8, 2, 128), [700, 3, 1300, 640, 0, 2049], 24),
    ((16, 16, 64), [385, 384, 383, 1000], 7),
    ((8, 1, 128), [3000], 128),                       # many partitions of one sequence
    ((8, 8, 64), [1025] * 5, 32),                     # the plain grid
    ((2, 1, 64), [70 + i % 3 for i in range(520)], 16),  # past 512 unequal sequences: the nominal split
]


@pytest.mark.parametrize("kv", ["f32", "f16", "i8"])
@pytest.mark.parametrize("heads,lens,page", CASES)
def test_library_partition(gpu, oracle, kv, heads, lens, page):
    kvb = gpu
    w = kvb.Workload(kvb.Shape(len(lens), *heads), kv, lens, seed=sum(lens) + page, varied=(kv == "i8"))
    c = kvb.PagedCache(w, page, 3 * page + 1, pool_factor=1.25, poison=True)
    dev = kvb.DeviceCase(w, c)
    dev.out.fill(0xFF)
    dev.run(0)
    fused = dev.output().copy()
    err = pb.check_output(kvb, oracle, w, c, fused)
    dev.out.fill(0xFF)
    dev.run_split(0)
    assert np.array_equal(dev.output(), fused), "two-kernel"
    graph = dev.capture_graph(0, 2)
    dev.out.fill(0xFF)
    graph.launch()
    assert np.array_equal(dev.output(), fused), "graph"
    graph.free()
    a = dev.args(0)
    dev.out.fill(0xFF)
    kvb.check(kvb.hip.kvb_run_paged_noalloc(ctypes.byref(a)), "noalloc")
    kvb.synchronize()
    assert np.array_equal(dev.output(), fused), "noalloc"
    # with a workspace of the caller's: the slots of kvb_auto_part_tokens, as the header lays them out
    part = kvb.auto_part_tokens(w.shape.batch, w.shape.num_kv_heads, w.max_len)
    outs = []
    for p in (0, part):
        ws = kvb.Buffer(dev.workspace_bytes(0))
        ws.fill(0xFF)
        dev.out.fill(0xFF)
        dev.run(p, workspace=ws)
        outs.append((dev.output().copy(), ws.download(np.uint32, ws.nbytes // 4)))
        ws.free()
    assert np.array_equal(outs[0][0], outs[1][0]) and np.array_equal(outs[0][1], outs[1][1])
    dev.free()
    progress(f"[split] {heads} {kv} page {page}: max err {err:.3g}")


def test_fp32_error_does_not_grow_with_the_partition(gpu, oracle):
    """A tile's products are summed on their own before they join the walk's sum, which is rounded once a
    tile and not once a token: a partition eight times as long errs no more (2-norm against the fp64 oracle;
    summed one by one, 1.5 times as much)."""
    kvb = gpu
    w = kvb.Workload(kvb.Shape(1, 16, 2, 64), "f32", [8192], seed=5, q_amp=1.0, dist="normal")
    c = kvb.PagedCache(w, 64, 3)
    want = oracle.attention(w.shape, w.lens, w.max_len, w.q, w.k, w.v)
    dev = kvb.DeviceCase(w, c)
    errs = []
    for part in (512, 4096):
        dev.run(part)
        errs.append(float(np.linalg.norm(dev.output().astype(np.float64) - want) / np.linalg.norm(want)))
    dev.free()
    assert errs[1] <= 1.1 * errs[0], errs
    progress(f"[split] fp32 error at 512 and 4096 tokens: {errs[0]:.3g} {errs[1]:.3g}")
