"""The work a user of this framework has it do, as cases that can be timed and checked: decode steps
over a paged KV cache (fp32, fp16 and int8 pages), the writers that fill such a cache from a prompt's
contiguous K and V, and the three-pass baseline over the contiguous cache.

A case is a dict of plain values. ``op`` is one of

- ``decode``: one step of paged attention. ``call`` "queued" is kvb_run_paged_noalloc, the form of a
  serving loop, where the layers' steps follow each other on one stream and nobody waits in between;
  "run" is kvb_run_paged, the reference's synchronous call. ``part`` is the split-K partition: 0 (the
  default: the library's own rule), "policy" (mi355x_part_tokens_for) or a number.
- ``write``: the prompt's K and then its V into the paged pool (kvb_write_paged).
- ``naive``: kvb_run_naive, the reference's comparison point in every row of its benchmark.

``lens`` is "equal" (every sequence max_len tokens) or "ragged" (uniform lengths from ``lens_seed``,
one of them max_len; from 8 sequences on, one of them empty).
"""
import ctypes
import importlib
import math
import random

import torch

kvb = importlib.import_module("kv-cache-bench_amd")

ESZ = {"f32": 4, "f16": 2, "i8": 1}
DTYPE = {"f32": torch.float32, "f16": torch.float16, "i8": torch.int8}
DEV = "cuda"
SCRATCH = 16 << 20  # KVB_NOALLOC_WORKSPACE_BYTES


def _decode(name, kv, batch, heads, kv_heads, dim, max_len, lens, page, part, call, pool=1.25, lens_seed=0):
    return dict(name=name, op="decode", kv=kv, batch=batch, heads=heads, kv_heads=kv_heads, dim=dim, max_len=max_len,
                lens=lens, lens_seed=lens_seed, page=page, part=part, call=call, pool=pool)


def listed():
    return [
        # One short fp32 sequence, called and waited for: the latency of a single step.
        _decode("f32_1x512", "f32", 1, 32, 8, 128, 512, "equal", 16, 128, "run", 2.0),
        # The first row of the reference's sweep in fp16, queued: a few short chats.
        _decode("f16_2x512", "f16", 2, 32, 8, 128, 512, "equal", 16, 0, "queued"),
        # A small batch of medium prompts with small pages, partition left to the library.
        _decode("f16_8x4k", "f16", 8, 32, 8, 128, 4096, "equal", 16, 0, "queued", 1.5),
        # int8 cache, a batch of 16 medium-long contexts, with the MI355X partition policy.
        _decode("i8_16x8k", "i8", 16, 32, 8, 128, 8192, "equal", 64, "policy", "queued", 1.0),
        # Long contexts, 8 query heads per KV head: the repository's headline step.
        _decode("f16_4x32k", "f16", 4, 64, 8, 128, 32768, "equal", 128, "policy", "queued"),
        # A large ragged serving batch; partition left to the library, the synchronous call.
        _decode("f16_ragged72", "f16", 72, 32, 8, 128, 16384, "ragged", 64, 0, "run", 1.5, 5),
        # The longest fp32 row of the reference's sweep, with its defaults.
        _decode("f32_2x32k", "f32", 2, 32, 8, 128, 32768, "equal", 16, 0, "queued", 1.0),
        # A small multi-head model (one query head per KV head, head_dim 64) in int8, ragged, with a
        # page size that is no multiple of a tile.
        _decode("i8_mha_page24", "i8", 24, 16, 16, 64, 6000, "ragged", 24, 0, "queued", 1.25, 3),
        # Many query heads on few KV heads: a group of 32.
        _decode("f16_gqa32", "f16", 8, 64, 2, 128, 8192, "ragged", 32, "policy", "queued", 1.25, 7),
        # Prompts written to small fp16 pages, ragged.
        dict(name="write_f16_page16", op="write", kv="f16", batch=16, kv_heads=8, dim=128, max_len=4096, lens="ragged",
             lens_seed=11, page=16, pool=1.25),
        # Prompts quantised to int8 pages.
        dict(name="write_i8_page64", op="write", kv="i8", batch=8, kv_heads=8, dim=128, max_len=8192, lens="equal",
             lens_seed=0, page=64, pool=1.0),
        # The three-pass baseline at the reference's middle length.
        dict(name="naive_f16_2x4k", op="naive", kv="f16", batch=2, heads=32, kv_heads=8, dim=128, max_len=4096,
             lens="equal", lens_seed=0),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choices(("decode", "write", "naive"), (8, 2, 1))[0]
    kv = rng.choice(("f32", "f16", "i8"))
    lens = rng.choice(("equal", "ragged"))
    seed = rng.randrange(1 << 16)
    dim = rng.choice((64, 128, 128))
    kv_heads = rng.choice((1, 2, 4, 8, 8, 16))
    if op == "naive":
        kv = rng.choice(("f32", "f16"))
        group = rng.choice((1, 4, 8))
        max_len = _log_int(rng, 64, 4096)
        batch = _log_int(rng, 1, max(1, min(8, (1 << 18) // (max_len * kv_heads * group))))
        return dict(op=op, kv=kv, batch=batch, heads=kv_heads * group, kv_heads=kv_heads, dim=dim, max_len=max_len,
                    lens=lens, lens_seed=seed)
    page = rng.choice((8, 16, 16, 24, 32, 48, 64, 64, 100, 128, 256))
    max_len = _log_int(rng, 64, 32768)
    # at most half the largest listed case's cache (1 GB of pages; 512 MB of a prompt's K and V)
    token = kv_heads * dim * 2 * (4 if op == "write" and kv == "i8" else ESZ[kv])
    batch = _log_int(rng, 1, max(1, min(72, (1 << 29 if op == "write" else 1 << 30) // (max_len * token))))
    if op == "write":
        return dict(op=op, kv=kv, batch=batch, kv_heads=kv_heads, dim=dim, max_len=max_len, lens=lens, lens_seed=seed,
                    page=page, pool=1.25)
    group = rng.choice((1, 2, 3, 4, 4, 5, 6, 7, 8, 8, 12, 16, 32))
    part = rng.choice((0, 0, "policy", 256))
    c = dict(op=op, kv=kv, batch=batch, heads=kv_heads * group, kv_heads=kv_heads, dim=dim, max_len=max_len, lens=lens,
             lens_seed=seed, page=page, part=part, call="queued", pool=1.25)
    # the queued call holds its split-K state in 16 MB of static scratch: larger steps take kvb_run_paged
    slots = batch * c["heads"] * -(-max_len // (64 if part == 0 else 256))
    if slots * (dim * 4 + 8) > SCRATCH or rng.random() < 0.2:
        c["call"] = "run"
    return c


def _lens(c):
    if c["lens"] == "equal":
        return [c["max_len"]] * c["batch"]
    r = random.Random(c["lens_seed"])
    n = [r.randint(1, c["max_len"]) for _ in range(c["batch"])]
    n[0] = c["max_len"]
    if c["batch"] >= 8:
        n[c["batch"] // 2] = 0
    return n


def _shape(c):
    return kvb.Shape(c["batch"], c.get("heads", c["kv_heads"]), c["kv_heads"], c["dim"])


def _part(c):
    if c["part"] != "policy":
        return int(c["part"])
    kind = kvb.KV_BY_NAME[c["kv"]]
    return kvb.mi355x_part_tokens_for(_shape(c), _lens(c), min_groups=kvb.mi355x_min_groups(kind, c["dim"]))


class _State:
    """A program's buffers and the argument structs that point at them."""


def _quantised(blocks, kv_heads, page, dim, gen):
    """Pages of N(0, 1) values as int8 with a scale per (block, KV head), as the cache writer leaves them."""
    q = torch.empty(blocks, kv_heads, page, dim, dtype=torch.int8, device=DEV)
    s = torch.empty(blocks, kv_heads, dtype=torch.float32, device=DEV)
    step = max(1, (1 << 26) // (kv_heads * page * dim))
    for i in range(0, blocks, step):
        x = torch.randn(min(step, blocks - i), kv_heads, page, dim, device=DEV, generator=gen)
        a = x.abs().amax(dim=(2, 3)) / 127.0
        s[i:i + step] = a
        q[i:i + step] = (x / a[:, :, None, None]).round().clamp(-127, 127).to(torch.int8)
    return q, s


def _layout(c, seed):
    """A shuffled block table over a pool of ceil(live * pool) blocks."""
    lens, page = _lens(c), c["page"]
    used = [-(-n // page) for n in lens]
    live, width = sum(used), max(1, max(used))
    blocks = max(1, math.ceil(live * c["pool"]))
    ids = torch.randperm(blocks, generator=torch.Generator().manual_seed(seed))[:live].to(torch.int32)
    table = torch.full((c["batch"], width), -1, dtype=torch.int32)
    at = 0
    for b, n in enumerate(used):
        table[b, :n] = ids[at:at + n]
        at += n
    return lens, blocks, table


def prepare(case, seed):
    """The buffers of one call, made on the GPU from the seed: q, K and V are N(0, 1) as in the
    repository's configurations. The library runs on its own stream, so the buffers are finished
    before it is called."""
    c, st = case, _State()
    gen = torch.Generator(device=DEV).manual_seed(seed)
    B, Hkv, D = c["batch"], c["kv_heads"], c["dim"]
    st.case, st.ms = c, ctypes.c_double()
    lens = _lens(c)
    st.host_lens = torch.tensor(lens, dtype=torch.int32)
    st.lens = st.host_lens.to(DEV)

    def rand(*shape, dtype=torch.float32):
        return torch.randn(*shape, device=DEV, dtype=dtype, generator=gen)

    if c["op"] == "write":
        _, blocks, table = _layout(c, seed)
        src = torch.float32 if c["kv"] == "i8" else DTYPE[c["kv"]]
        st.table = table.to(DEV)
        st.contig = [rand(B, Hkv, c["max_len"], D, dtype=src) for _ in range(2)]
        st.pool = [torch.zeros(blocks, Hkv, c["page"], D, dtype=DTYPE[c["kv"]], device=DEV) for _ in range(2)]
        st.scale = [torch.zeros(blocks, Hkv, device=DEV) for _ in range(2)] if c["kv"] == "i8" else [None, None]
        st.args = []
        for x, pool, scale in zip(st.contig, st.pool, st.scale):
            a = kvb.CacheArgsC()
            a.batch, a.num_kv_heads, a.head_dim, a.kv_type = B, Hkv, D, kvb.KV_BY_NAME[c["kv"]]
            a.page_size, a.max_blocks, a.max_len = c["page"], table.shape[1], c["max_len"]
            a.contig, a.paged, a.block_table, a.seq_lens = x.data_ptr(), pool.data_ptr(), st.table.data_ptr(), st.lens.data_ptr()
            a.scales = scale.data_ptr() if scale is not None else None
            a.host_seq_lens = st.host_lens.data_ptr()
            st.args.append(a)
    elif c["op"] == "naive":
        dt = DTYPE[c["kv"]]
        st.q = rand(B, c["heads"], D)
        st.k, st.v = (rand(B, Hkv, c["max_len"], D, dtype=dt) for _ in range(2))
        st.out = torch.empty_like(st.q)
        a = st.args = kvb.NaiveArgsC()
        a.batch, a.num_heads, a.num_kv_heads, a.head_dim = B, c["heads"], Hkv, D
        a.kv_type, a.max_len = kvb.KV_BY_NAME[c["kv"]], c["max_len"]
        a.q, a.k, a.v, a.seq_lens, a.out = (t.data_ptr() for t in (st.q, st.k, st.v, st.lens, st.out))
        a.host_seq_lens = st.host_lens.data_ptr()
    else:
        _, blocks, table = _layout(c, seed)
        st.table = table.to(DEV)
        st.q = rand(B, c["heads"], D)
        st.out = torch.empty_like(st.q)
        st.ks = st.vs = None
        if c["kv"] == "i8":
            st.k, st.ks = _quantised(blocks, Hkv, c["page"], D, gen)
            st.v, st.vs = _quantised(blocks, Hkv, c["page"], D, gen)
        else:
            st.k, st.v = (rand(blocks, Hkv, c["page"], D, dtype=DTYPE[c["kv"]]) for _ in range(2))
        a = st.args = kvb.PagedArgsC()
        a.batch, a.num_heads, a.num_kv_heads, a.head_dim = B, c["heads"], Hkv, D
        a.kv_type, a.page_size, a.max_blocks = kvb.KV_BY_NAME[c["kv"]], c["page"], table.shape[1]
        a.max_len, a.part_tokens, a.share_kv = c["max_len"], _part(c), 1
        a.q, a.k, a.v, a.block_table, a.seq_lens, a.out = (t.data_ptr() for t in (st.q, st.k, st.v, st.table, st.lens, st.out))
        a.host_seq_lens = st.host_lens.data_ptr()
        if st.ks is not None:
            a.k_scale, a.v_scale = st.ks.data_ptr(), st.vs.data_ptr()
    torch.cuda.synchronize()
    return st


def run(state):
    c, hip = state.case, kvb.hip
    if c["op"] == "write":
        for a in state.args:
            kvb.check(hip.kvb_write_paged(ctypes.byref(a), ctypes.byref(state.ms)), "write_paged")
        return [t for t in state.pool + state.scale if t is not None]
    if c["op"] == "naive":
        kvb.check(hip.kvb_run_naive(ctypes.byref(state.args), ctypes.byref(state.ms)), "run_naive")
    elif c["call"] == "queued":
        kvb.check(hip.kvb_run_paged_noalloc(ctypes.byref(state.args)), "run_paged_noalloc")
    else:
        kvb.check(hip.kvb_run_paged(ctypes.byref(state.args), ctypes.byref(state.ms)), "run_paged")
    return state.out


def work(case):
    c = case
    lens = _lens(c)
    tokens = sum(lens)
    rows = tokens * c["kv_heads"] * c["dim"] * 2  # K and V values
    if c["op"] == "write":
        blocks = sum(-(-n // c["page"]) for n in lens)
        if c["kv"] == "i8":
            return {"bytes": rows * 5 + blocks * c["kv_heads"] * 8, "flops": 3 * rows}
        return {"bytes": rows * ESZ[c["kv"]] * 2, "flops": 0}
    bytes_ = rows * ESZ[c["kv"]] + c["batch"] * c["heads"] * c["dim"] * 8
    if c["op"] == "decode":
        blocks = sum(-(-n // c["page"]) for n in lens)
        bytes_ += 4 * blocks + (blocks * c["kv_heads"] * 8 if c["kv"] == "i8" else 0)
    return {"bytes": bytes_, "flops": 4 * tokens * c["heads"] * c["dim"]}


def tolerance(case):
    if case["op"] == "write":
        return "exact"  # a copy, or the reference's quantiser byte for byte
    # fp32 sums over exact products (fp16 and int8 keep q and p to about 22 bits). Against exact() the
    # decode is off by 2e-7 to 7e-7 (2-norm), the baseline's one-by-one sums by 1.2e-6.
    return {"rel": 5e-6 if case["op"] == "naive" else 3e-6}


def exact(case, seed):
    """The same inputs through plain torch in 64 bits."""
    st, c = prepare(case, seed), case
    lens, B, Hkv, D = _lens(c), c["batch"], c["kv_heads"], c["dim"]
    if c["op"] == "write":
        return _exact_write(st, c, lens)
    out = torch.zeros(B, c["heads"], D, dtype=torch.float64, device=DEV)
    for b, n in enumerate(lens):
        if n == 0:
            continue
        if c["op"] == "naive":
            k, v = (t[b, :, :n].double() for t in (st.k, st.v))
        else:
            ids = st.table[b, :-(-n // c["page"])].long()

            def rows(pool, scale):
                x = pool[ids].double()
                if scale is not None:
                    x = x * scale[ids].double()[:, :, None, None]
                return x.transpose(0, 1).reshape(Hkv, -1, D)[:, :n]

            k, v = rows(st.k, st.ks), rows(st.v, st.vs)
        q = st.q[b].double().reshape(Hkv, -1, D)
        for h in range(Hkv):
            p = torch.softmax(q[h] @ k[h].t() / math.sqrt(D), dim=-1)
            out[b].view(Hkv, -1, D)[h] = p @ v[h]
    return out


def _exact_write(st, c, lens):
    page = c["page"]
    pools = [t.double() for t in st.pool]
    scales = [t.double() if t is not None else None for t in st.scale]
    for b, n in enumerate(lens):
        used = -(-n // page)
        if used == 0:
            continue
        ids = st.table[b, :used].long()
        for x, pool, scale in zip(st.contig, pools, scales):
            rows = torch.zeros(c["kv_heads"], used * page, c["dim"], dtype=torch.float64, device=DEV)
            rows[:, :n] = x[b, :, :n].double()
            rows = rows.reshape(c["kv_heads"], used, page, c["dim"]).transpose(0, 1)
            if scale is not None:
                a = rows.abs().amax(dim=(2, 3)) / 127.0
                scale[ids] = a
                rows = (rows / a[:, :, None, None]).round().clamp(-127, 127)
            pool[ids] = rows
    if c["kv"] == "i8":
        return [None, None] + scales  # the bytes are whole numbers: rounding decides their ties
    return pools
