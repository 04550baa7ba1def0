"""Workgroups of 16 and 32 query heads, which a step runs when its grid fills at least half the CUs
with them (a smaller step runs 8- or 16-head workgroups, whatever kvb_heads_per_workgroup says): batches
of 130 and more sequences with one KV head, so that the wide builds run, and the same sequences a few at
a time, so that the narrow ones do. Both against the oracle, and against each other: to the bit for 16 of
32 heads, to fp32 rounding for 8."""
import numpy as np
import pytest

import parity_battery as pb
from conftest import progress

pytestmark = pytest.mark.gpu

# group, head_dim, lengths of three sequences (repeated), page, partition
CASES = [
    (16, 128, [70, 33, 129], 16, 64),      # 2, 1 and 3 partitions
    (16, 64, [200, 1, 97], 24, 256),       # one partition, any page
    (32, 64, [300, 257, 0], 16, 128),      # the shared tiles of fp16, three partitions and an empty sequence
    (32, 128, [520, 31, 161], 32, 1024),   # five tiles a stream: each LDS slot reused
    (64, 64, [96, 40, 65], 7, 64),         # two 32-head workgroups per KV head, any page and partition
]


def kernel_heads(name):
    return int(name.split("<")[1].split(",")[2])


@pytest.mark.parametrize("kv", ["f16", "i8"])
@pytest.mark.parametrize("group,dim,lens,page,part", CASES)
def test_wide_workgroups_on_full_grids(gpu, oracle, kv, group, dim, lens, page, part):
    kvb = gpu
    wide = kvb.heads_per_workgroup(kvb.Shape(1, group, 1, dim), kv)
    many = (lens * 87)[: 260 if wide == group else 130]
    w = kvb.Workload(kvb.Shape(len(many), group, 1, dim), kv, many, seed=group + page, varied=(kv == "i8"))
    c = kvb.PagedCache(w, page, page + 5, pool_factor=1.1, poison=True)
    dev = kvb.DeviceCase(w, c)
    assert kernel_heads(dev.kernel_name(part)) == wide
    dev.out.fill(0xFF)
    dev.run(part)
    full = dev.output().copy()
    dev.out.fill(0xFF)
    dev.run_split(part)
    assert np.array_equal(dev.output(), full), "two-kernel"
    dev.free()
    err = pb.check_output(kvb, oracle, w, c, full)
    heads = set()
    for at, n in ((0, 3), (3, 45)):
        sub = kvb.Workload.from_arrays(kv, w.lens[at:at + n], w.q[at:at + n], w.k[at:at + n], w.v[at:at + n])
        part_c = kvb.PagedCache(sub, page, page + 5, pool_factor=1.1, poison=True)
        few = kvb.DeviceCase(sub, part_c)
        heads.add(kernel_heads(few.kernel_name(part)))
        few.out.fill(0xFF)
        few.run(part)
        got = few.output().copy()
        few.free()
        if kernel_heads(few_name := dev_name(kvb, sub, part_c, part)) == 16 and wide == 32:
            assert np.array_equal(got, full[at:at + n]), few_name
        else:  # (the bound of the 8-head and 16-head waves' agreement: 2e-7 of the largest |v|)
            assert np.abs(got - full[at:at + n]).max() <= 2e-7 * max(1.0, float(np.abs(sub.v).max()))
    assert min(heads) < wide, heads
    progress(f"[wide] group {group} D{dim} {kv} page {page} part {part}: {wide} heads, narrow {sorted(heads)}, err {err:.3g}")


def dev_name(kvb, w, c, part):
    dev = kvb.DeviceCase(w, c)
    name = dev.kernel_name(part)
    dev.free()
    return name
