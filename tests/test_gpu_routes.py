"""Which build of paged_decode a step runs (kvb_paged_kernel_name), on both sides of each rule of the
dispatch that sizes and types draw, and the builds those rules alone reach against the oracle."""
import ctypes

import numpy as np
import pytest

import parity_battery as pb
from conftest import progress

pytestmark = pytest.mark.gpu

FIELDS = ("kind", "dim", "heads", "fast", "loads", "pair", "part", "share", "stage", "refill")


def build_of(kvb, dev, part, share_kv=True):
    """The template arguments of the kernel a step launches."""
    buf = ctypes.create_string_buffer(512)
    a = dev.args(part, share_kv=share_kv)
    kvb.check(kvb.hip.kvb_paged_kernel_name(ctypes.byref(a), 0, buf, 512), "paged_kernel_name")
    values = buf.value.decode().split("<")[1].split(">")[0].split(", ")
    return dict(zip(FIELDS, values))


# heads, KV heads, share_kv: workgroups of 1, 2 and 4 heads, several per KV head
SIBLINGS = [((8, 2, 64), False), ((22, 2, 128), True), ((44, 2, 64), True), ((44, 1, 128), True)]


@pytest.mark.parametrize("kv", ["f32", "f16", "i8"])
@pytest.mark.parametrize("heads,share_kv", SIBLINGS)
@pytest.mark.parametrize("page,part,lens", [(24, 128, [300, 130]), (3, 64, [100, 64, 1, 0]), (7, 1024, [700] * 8)])
def test_siblings_share_pages_of_any_size(gpu, oracle, kv, heads, share_kv, page, part, lens):
    """Workgroups that read the same pages run the SHARE build (int8: from 32 MB of cache on)."""
    kvb = gpu
    w = kvb.Workload(kvb.Shape(len(lens), *heads), kv, lens, seed=page + sum(lens), varied=(kv == "i8"))
    c = kvb.PagedCache(w, page, 3 * page, pool_factor=1.2, poison=True)
    dev = kvb.DeviceCase(w, c)
    build = build_of(kvb, dev, part, share_kv)
    assert build["fast"] == "false" and build["share"] == ("false" if kv == "i8" else "true")
    dev.out.fill(0xFF)
    dev.run(part, share_kv=share_kv)
    err = pb.check_output(kvb, oracle, w, c, dev.output())
    dev.free()
    progress(f"[routes] siblings {heads} {kv} page {page}: max err {err:.3g}")


def test_int8_siblings_share_large_caches(gpu, oracle):
    kvb = gpu
    for length in (1023, 1025):  # 16 KV heads x 128 x 8 sequences x 2 = 32 KB a token
        w = kvb.Workload(kvb.Shape(8, 32, 16, 128), "i8", [length] * 8, seed=length)
        c = kvb.PagedCache(w, 100, 7, poison=True)
        dev = kvb.DeviceCase(w, c)
        assert build_of(kvb, dev, 256, share_kv=False)["share"] == ("true" if length > 1024 else "false")
        dev.out.fill(0xFF)
        dev.run(256, share_kv=False)
        pb.check_output(kvb, oracle, w, c, dev.output())
        dev.free()


@pytest.mark.parametrize("kv", ["f32", "f16"])
@pytest.mark.parametrize("heads,page", [((8, 8, 64), 24), ((14, 2, 128), 3), ((16, 1, 64), 7)])
def test_small_caches_are_read_with_ordinary_loads(gpu, oracle, kv, heads, page):
    """One workgroup per KV head (of 1, 7 and 16 heads): the SHARE build and its ordinary loads."""
    kvb = gpu
    lens = [300, 131, 0, 77]
    w = kvb.Workload(kvb.Shape(len(lens), *heads), kv, lens, seed=page)
    c = kvb.PagedCache(w, page, page, pool_factor=1.2, poison=True)
    dev = kvb.DeviceCase(w, c)
    assert build_of(kvb, dev, 128)["share"] == "true"
    dev.out.fill(0xFF)
    dev.run(128)
    pb.check_output(kvb, oracle, w, c, dev.output())
    dev.free()


def test_large_caches_are_read_with_streaming_loads(gpu):
    """Past 256 MB of cache, by the lengths alone (nothing is launched, so the pool need not hold them)."""
    kvb = gpu
    w = kvb.Workload(kvb.Shape(2, 8, 8, 128), "f16", [24, 24], seed=1)
    c = kvb.PagedCache(w, 24, 1)
    dev = kvb.DeviceCase(w, c)
    a = dev.args(512)
    buf = ctypes.create_string_buffer(512)
    for n, share in ((32768, "true"), (32769, "false")):  # 8 KV heads x 128 x 2 sequences x 2 x 2 = 8 KB a token
        lens = np.array([n, n], np.int32)
        a.max_len, a.max_blocks, a.host_seq_lens = n, n // 24 + 1, lens.ctypes.data
        kvb.check(kvb.hip.kvb_paged_kernel_name(ctypes.byref(a), 0, buf, 512), "paged_kernel_name")
        assert buf.value.decode().split("<")[1].split(">")[0].split(", ")[7] == share
    dev.free()


@pytest.mark.parametrize("heads", [(8, 2, 64), (8, 2, 128), (24, 2, 64), (12, 2, 128)])
@pytest.mark.parametrize("page", [16, 24])
@pytest.mark.parametrize("lens,part", [([1000, 600], 256), ([1000, 600], 128), ([257] * 2, 300), ([300] * 64, 256),
                                       ([300] * 65, 256), ([300] * 32, 256), ([300] * 33, 256)])
def test_fp32_refills_where_a_workgroup_has_its_cu(gpu, oracle, heads, page, lens, part):
    """The build that loads the next tile under the present one: at most one workgroup per CU (of 256), and
    two tiles a wave."""
    kvb = gpu
    w = kvb.Workload(kvb.Shape(len(lens), *heads), "f32", lens, seed=page + part)
    c = kvb.PagedCache(w, page, part, pool_factor=1.1, poison=True)
    dev = kvb.DeviceCase(w, c)
    groups = heads[0] // kvb.heads_per_workgroup(w.shape, kvb.KV_F32) * sum(-(-n // part) for n in lens)
    assert build_of(kvb, dev, part)["refill"] == ("true" if part >= 256 and groups <= 256 else "false")
    dev.out.fill(0xFF)
    dev.run(part)
    pb.check_output(kvb, oracle, w, c, dev.output())
    dev.free()


# kv, group, head_dim, sequences of 1000 tokens with 4 partitions each, heads per workgroup: the wide
# workgroups where they fill half the CUs (of 256), int8 groups of 16 at head_dim 64 an eighth of them
@pytest.mark.parametrize("kv,group,dim,batch,heads", [
    ("f16", 16, 64, 32, 8), ("f16", 16, 64, 33, 16), ("i8", 16, 128, 32, 8), ("i8", 16, 128, 33, 16),
    ("i8", 16, 64, 8, 8), ("i8", 16, 64, 9, 16), ("i8", 16, 64, 33, 16),
    ("i8", 32, 64, 16, 8), ("i8", 32, 64, 17, 16), ("i8", 32, 64, 32, 16), ("i8", 32, 64, 33, 32),
])
def test_wide_groups_on_few_workgroups(gpu, kv, group, dim, batch, heads):
    kvb = gpu
    w = kvb.Workload(kvb.Shape(batch, group, 1, dim), kv, [1000] * batch, seed=batch)
    c = kvb.PagedCache(w, 64, 1)
    dev = kvb.DeviceCase(w, c)
    assert build_of(kvb, dev, 256)["heads"] == str(heads)
    dev.free()


# page, sequences, their length: fewer and fuller workgroups than at 512 tokens would suit the batch
LONG = [(1, 16, 32768), (1, 32, 16384), (1, 64, 8192), (3, 16, 32768), (24, 64, 8192), (64, 64, 8192)]


@pytest.mark.parametrize("kv,most", [("f32", 4096), ("f16", 1024), ("i8", 1024)])
@pytest.mark.parametrize("page,batch,n", LONG)
@pytest.mark.parametrize("ragged", [False, True])
def test_library_partitions_stay_exact_and_staged(gpu, kv, most, page, batch, n, ragged):
    """Left to the library, no partition is so long that its error grows or that its block ids no longer fit
    in LDS (by the lengths alone: nothing is launched, so the pool need not hold them)."""
    kvb = gpu
    w = kvb.Workload(kvb.Shape(batch, 16, 2, 128), kv, [24] * batch, seed=1)
    c = kvb.PagedCache(w, page, 1)
    dev = kvb.DeviceCase(w, c)
    a = dev.args(0)
    lens = np.array([n - 5 * i * ragged for i in range(batch)], np.int32)
    a.max_len, a.max_blocks, a.host_seq_lens = n, -(-n // page), lens.ctypes.data
    part = kvb.hip.kvb_paged_part_tokens(ctypes.byref(a))
    assert 0 < part <= most
    buf = ctypes.create_string_buffer(512)
    kvb.check(kvb.hip.kvb_paged_kernel_name(ctypes.byref(a), 0, buf, 512), "paged_kernel_name")
    values = dict(zip(FIELDS, buf.value.decode().split("<")[1].split(">")[0].split(", ")))
    if page % 16:
        assert values["stage"] != "0"
    dev.free()


# page, partition, the build's table: a block either side of what each holds
@pytest.mark.parametrize("kv", ["f32", "f16", "i8"])
@pytest.mark.parametrize("page,part,table", [(1, 512, 512), (1, 513, 4096), (1, 4096, 4096), (1, 4097, 0),
                                             (3, 1536, 512), (3, 1537, 4096), (3, 1529, 512)])
def test_block_ids_at_the_edges_of_their_tables(gpu, oracle, kv, page, part, table):
    kvb = gpu
    lens = [part + 130, part, 1]
    w = kvb.Workload(kvb.Shape(len(lens), 4, 1, 64), kv, lens, seed=part, varied=(kv == "i8"))
    c = kvb.PagedCache(w, page, part, pool_factor=1.1, poison=True)
    dev = kvb.DeviceCase(w, c)
    assert build_of(kvb, dev, part)["stage"] == str(4096 if table and kv == "f16" else table)  # (fp16: one table)
    dev.out.fill(0xFF)
    dev.run(part)
    pb.check_output(kvb, oracle, w, c, dev.output())
    dev.free()
