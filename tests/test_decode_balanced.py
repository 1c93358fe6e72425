"""Balanced decode (csrc/decode_sched.hpp): the keys of all sequences shared evenly between a fixed
number of workgroups by the lengths on the device. On the CPU: the schedule's arithmetic, restated
here, covers every key of every work head once, gives every segment a partial slot of its own inside
the workspace and every work head consecutive slots, over random and extreme lengths; and the plan's
choices. On the GPU: both split kernels through the public op, contiguous and paged, against the fp64
oracle, with lengths that cross, fill and leave empty the workgroups' shares.
"""

import ctypes
import random

import pytest
import torch

import flash_lab
from flash_lab import _hip
from parity import check_decode, normwise_rel
from oracle import reference


ROW_SLOTS = 8


def schedule(lens, rows, wgs, unit_keys, min_units, ramp_units):
    """(chunk, start of every row, size of every row): make_schedule's arithmetic."""
    units = [-(-n // unit_keys) for n in lens]
    sizes = [u + ramp_units if u else 0 for u in units]
    filled = sum(u > 0 for u in units)
    least = max(-(-sum(units) * rows // wgs), min_units)
    chunk = max(-(-sum(sizes) * rows // wgs), min_units)
    if filled * rows <= wgs:
        for c in (least, chunk):
            if sum(-(-u // c) for u in units) * rows <= wgs:
                sizes, chunk = [-(-u // c) * c for u in units], c
                break
    starts, every, pos = [], [], 0
    for size in sizes:
        for _ in range(rows):
            starts.append(pos)
            every.append(size)
            pos += size
    return chunk, starts, every


@pytest.mark.parametrize("rows,wgs,unit_keys,min_units,ramp_units", [
    (2, 256, 32, 2, 1), (8, 256, 32, 2, 4), (1, 256, 64, 1, 1), (32, 768, 64, 1, 1), (3, 7, 32, 2, 4),
])
def test_schedule_covers_every_key_once(rows, wgs, unit_keys, min_units, ramp_units):
    rng = random.Random(rows * wgs)
    cases = [[0] * 5, [1], [0, 1, 0], [32768] * 8, [1] * 256, [0] * 63 + [30000], [700, 701, 64, 63, 65, 0, 32]]
    cases += [[rng.choice([0, 1, rng.randrange(70), rng.randrange(9000)]) for _ in range(rng.randrange(1, 70))]
              for _ in range(8)]
    for lens in cases:
        chunk, starts, sizes = schedule(lens, rows, wgs, unit_keys, min_units, ramp_units)
        total = starts[-1] + sizes[-1]
        assert wgs * chunk >= total
        slots, keys, counts, written = set(), [0] * len(starts), [0] * len(starts), {}
        for w in range(wgs):
            pos, end = w * chunk, min((w + 1) * chunk, total)
            while pos < end:
                row = next(r for r in range(len(starts)) if starts[r] <= pos < starts[r] + sizes[r])
                first, n = pos - starts[row], lens[row // rows]
                after = min(end, starts[row] + sizes[row])
                begin, stop = min(n, first * unit_keys), min(n, (first + after - pos) * unit_keys)
                first_wg = starts[row] // chunk
                if first == 0:
                    units = -(-n // unit_keys)
                    written[row] = ((starts[row] + units - 1) // chunk - first_wg + 1, first_wg + row)
                pos = after
                if begin == stop:  # only the row's start cost
                    continue
                assert begin == keys[row]
                keys[row] = stop
                split = counts[row]
                counts[row] += 1
                assert split == w - first_wg
                slot = row * ROW_SLOTS + split if split < ROW_SLOTS else len(starts) * ROW_SLOTS + w + row
                assert split < ROW_SLOTS or slot == len(starts) * ROW_SLOTS + written[row][1] + split
                assert slot not in slots and slot < (ROW_SLOTS + 1) * len(starts) + wgs
                slots.add(slot)
        assert keys == [n for n in lens for _ in range(rows)]
        assert all(written[r][0] == counts[r] if lens[r // rows] else r not in written for r in range(len(starts)))


def test_floor_by_reciprocal():
    # floor_div: one float reciprocal per divisor, corrected by the remainder.
    rng = random.Random(0)
    top = 1 << 22
    for c in [1, 2, 3, 5, 7, 31, 64, 100, 999, 65536, top] + [rng.randrange(1, top) for _ in range(40)]:
        r = torch.tensor(1.0) / torch.tensor(float(c))
        n = torch.tensor([0, 1, c - 1, c, min(c + 1, top), top] +
                         [min(top, max(0, rng.randrange(1, top // c + 1) * c + d))
                          for _ in range(100) for d in (-1, 0, 1)])
        for off in (-1, 0, 1):  # the reciprocal one unit in its last place off
            approx = torch.nextafter(r, r + off) if off else r
            q = (n.float() * approx).int()
            rem = n - q * c
            q = q + (rem >= c).int() - (rem < 0).int()
            assert torch.equal(q.long(), n // c), c


DTYPES = {0: torch.bfloat16, 2: torch.float32}


def plan(batch, heads, heads_kv, head_dim, max_seqlen, dtype=0, page_size=0):
    return _hip.decode_schedule(batch, heads, heads_kv, head_dim, max_seqlen, DTYPES[dtype], page_size)


def test_plan():
    # 24 sequences of 8 KV heads, four per workgroup on the matrix-core kernel: 48 rows, 16 heads each.
    assert plan(24, 32, 8, 128, 8192, page_size=16) == (0, 256, (256 + 48 * 9) * 16 * 130 * 4 + 48 * 8)
    assert plan(8, 32, 32, 128, 8192)[1] == 256  # vector kernel, contiguous
    # Splits: a contiguous cache of grouped heads, few or more than 256 sequences, a small cache, segments
    # whose 1-row pages do not fit LDS, a line past 2^22 units.
    assert plan(24, 32, 8, 128, 8192)[1] == 0
    assert plan(5, 32, 8, 128, 32768, page_size=16)[1] == 0
    assert plan(257, 32, 8, 128, 8192, page_size=16)[1] == 0
    assert plan(24, 32, 8, 128, 1024, page_size=16)[1] == 0
    assert plan(8, 32, 8, 128, 131072, page_size=16)[1] == 256
    assert plan(8, 32, 8, 128, 131072, page_size=1)[1] == 0
    assert plan(64, 32, 8, 128, 1 << 20, page_size=64)[1] == 0
    assert plan(2, 8, 8, 64, 64) == (1, 0, 0)  # too short to be worth a merge pass


def test_split_counts():
    # One workgroup per CU where nobody asked for a count: matrix cores down to 64 keys, several query
    # heads on the vector kernel (fp32 here), and no more than that for short caches of one.
    assert plan(1, 32, 8, 128, 640)[:2] == (8, 0)
    assert plan(1, 32, 8, 128, 8448)[:2] == (32, 0)
    assert plan(8, 32, 8, 128, 32768)[:2] == (16, 0)  # four KV heads per workgroup, as planned
    assert plan(8, 32, 8, 128, 16000, dtype=2)[:2] == (4, 0)
    assert plan(4, 8, 8, 128, 3000)[:2] == (8, 0)
    assert plan(1, 32, 32, 128, 32768)[:2] == (16, 0)  # long: as planned
    # Groups of 3: three heads per workgroup (32 splits), and in fp32, where three workgroups read the same
    # keys, splits of 180 keys or more.
    assert plan(1, 24, 8, 128, 8192)[:2] == (32, 0)
    assert plan(4, 24, 8, 128, 4000, dtype=2)[:2] == (16, 0)
    # ... and one head per workgroup for smaller caches.
    assert plan(4, 24, 8, 64, 528)[0] == 1 and plan(8, 24, 8, 128, 304)[0] == 1
    # Two of them, or four of small rows, are left as planned.
    assert plan(6, 24, 8, 64, 576)[0] == 1 and plan(6, 24, 8, 64, 800)[0] == 1
    assert plan(10, 24, 8, 128, 400, dtype=2)[0] == 1 and plan(6, 24, 8, 128, 800, dtype=2)[0] == 4
    # A paged call keeps a split's block numbers within LDS.
    assert plan(1, 16, 8, 128, 131072, page_size=1)[0] == 128


@pytest.mark.parametrize("shape", [(2, 32, 8, 128, 352), (8, 16, 2, 128, 300), (13, 64, 8, 128, 176)], ids=str)
def test_short_fp32_caches_of_512_byte_rows_are_split_as_planned(shape):
    assert plan(*shape, dtype=2)[:2] == (_hip.decode_plan(*shape, torch.float32)[0], 0)
    assert plan(*shape, dtype=2)[0] > 1 and plan(*shape)[0] == 1  # bf16: one split


@pytest.mark.parametrize("shape", [(1, 24, 8, 128, 144), (1, 32, 8, 128, 144), (18, 32, 8, 128, 128), (2, 64, 8, 128, 48)], ids=str)
def test_the_shortest_fp32_caches_take_one_split(shape):
    assert plan(*shape, dtype=2) == (1, 0, 0)


def test_workgroups_that_share_keys_are_not_balanced():
    # Groups of 3 in fp32: three workgroups read the same keys, and short splits keep those reads together.
    assert plan(10, 24, 8, 128, 10848, dtype=2, page_size=16)[:2] == (8, 0)
    assert plan(24, 24, 8, 128, 2048, dtype=2, page_size=16)[:2] == (4, 0)
    assert plan(8, 24, 8, 64, 4096, dtype=2, page_size=16)[:2] == (16, 0)
    assert plan(10, 24, 8, 128, 10848, page_size=16)[0] == 0  # bf16: one workgroup for the three heads
    assert plan(16, 32, 8, 128, 8192, dtype=2, page_size=16)[0] == 0  # fp32, four heads per workgroup


@pytest.mark.parametrize("shape,span", [
    ((8, 32, 4, 128, 32768), 1), ((6, 32, 4, 128, 49152), 1),  # 8 and 6 rows with four KV heads in each
    ((64, 32, 8, 128, 2048), 4), ((10, 32, 8, 64, 16384), 4),  # 128 and 20 rows
], ids=str)
def test_balanced_spans(shape, span):
    batch, heads, heads_kv, head_dim = shape[:4]
    rows = batch * heads_kv // span
    want = (256 + rows * 9) * (batch * heads // rows) * (head_dim + 2) * 4 + rows * 8
    assert plan(*shape, page_size=16) == (0, 256, want)


@pytest.mark.parametrize("span", [1, 2, 3, 4])
def test_forced_spans(span, knobs):
    # 4 KV heads per workgroup, or, at any other value of the knob, one: 48 rows of 16 heads or 192 of 4.
    knobs("decode_mfma_span", span)
    rows = 48 if span == 4 else 192
    want = (256 + rows * 9) * (24 * 32 // rows) * 130 * 4 + rows * 8
    assert plan(24, 32, 8, 128, 8192, page_size=16) == (0, 256, want)


@pytest.mark.parametrize("shape", [(1, 8, 8, 128, 300), (16, 32, 8, 128, 320), (2, 8, 8, 64, 90), (4, 32, 8, 128, 4000)],
                         ids=str)
def test_workgroups_per_cu_knob_gives_the_plans_count(shape, knobs):
    knobs("decode_wg_per_cu", 4)
    assert plan(*shape)[:2] == (_hip.decode_plan(*shape, torch.bfloat16)[0], 0)


def test_balanced_call_is_checked_before_any_launch():
    p = _hip.DecodeParams()
    p.q = p.k_cache = p.v_cache = p.o = p.lse = p.seq_lens = 256
    p.batch, p.heads, p.heads_kv, p.head_dim, p.max_seqlen, p.softmax_scale = 24, 32, 8, 128, 8192, 0.1
    p.block_tables, p.page_size, p.num_blocks = 256, 16, 1 << 14
    p.workspace, p.workspace_bytes = 256, plan(24, 32, 8, 128, 8192, page_size=16)[2] - 4
    for wgs in (0, -1, 1 << 17, 256):
        assert _hip.LIB.fl_decode_balanced(ctypes.byref(p), wgs, None) == 1
    p.batch, p.workspace_bytes = 257, 1 << 40
    assert _hip.LIB.fl_decode_balanced(ctypes.byref(p), 256, None) == 1


CASES = [
    # batch, heads, heads_kv, max_seqlen, head_dim, lens
    (5, 32, 8, 3000, 128, [3000, 1, 0, 1777, 64]),  # matrix cores, one KV head per workgroup
    (33, 32, 8, 4100, 128, "random"),  # four per workgroup
    (70, 8, 2, 900, 64, "random"),  # two sequences per lane
    (3, 8, 8, 5000, 128, [5000, 31, 4999]),  # vector kernel, one query head
    (6, 16, 8, 2100, 64, [2100, 0, 0, 63, 65, 128]),  # vector kernel, two query heads
    (256, 4, 4, 300, 64, "random"),
    (2, 24, 8, 1500, 128, [1500, 700]),  # group of 3
]


def inputs(case, dtype):
    batch, heads, heads_kv, max_seqlen, head_dim, lens = case
    gen = torch.Generator(device="cuda").manual_seed(3)
    q = torch.randn(batch, 1, heads, head_dim, device="cuda", dtype=dtype, generator=gen)
    k, v = (torch.randn(batch, max_seqlen, heads_kv, head_dim, device="cuda", dtype=dtype, generator=gen)
            for _ in range(2))
    if lens == "random":
        lens = torch.randint(0, max_seqlen + 1, (batch,), device="cuda", generator=gen)
    else:
        lens = torch.tensor(lens, device="cuda")
    return q, k, v, lens.to(torch.int32)


def paged(cache, page):
    batch, rows, heads_kv, head_dim = cache.shape
    blocks = -(-rows // page)
    padded = torch.zeros(batch, blocks * page, heads_kv, head_dim, device="cuda", dtype=cache.dtype)
    padded[:, :rows] = cache
    order = torch.randperm(batch * blocks, device="cuda", generator=torch.Generator(device="cuda").manual_seed(4))
    pool = torch.empty(batch * blocks, page, heads_kv, head_dim, device="cuda", dtype=cache.dtype)
    pool[order] = padded.reshape(batch * blocks, page, heads_kv, head_dim)
    return pool, order.to(torch.int32).reshape(batch, blocks)


def balanced(q, k, v, lens, workgroups, tables=None):
    """fl_decode_balanced on these inputs, whatever the plan would choose."""
    q = q[:, 0]
    batch, heads, head_dim = q.shape
    out, lse = torch.empty_like(q), torch.empty(batch, heads, device="cuda")
    p = _hip._decode_params(q, k, v, lens, out, lse, head_dim**-0.5, tables)
    rows = batch * k.shape[2]  # at most: one row per KV head, whatever the span
    workspace = torch.full(((workgroups + rows * 9) * heads * (head_dim + 2) + 2 * rows,), float("nan"),
                           device="cuda")
    p.workspace, p.workspace_bytes = workspace.data_ptr(), 4 * workspace.numel()
    _hip._check(_hip.LIB.fl_decode_balanced(ctypes.byref(p), workgroups, torch.cuda.current_stream().cuda_stream))
    return out[:, None], lse


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "fp16", "fp32"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"B{c[0]}-H{c[1]}-Hkv{c[2]}-S{c[3]}-D{c[4]}")
def test_balanced_decode_matches_reference(case, dtype):
    q, k, v, lens = inputs(case, dtype)
    k_pool, tables = paged(k, 16)
    v_pool, _ = paged(v, 16)
    full = lens > 0
    for workgroups in (7, 256, 700):
        print(f"balanced decode {case} {dtype} workgroups={workgroups}", flush=True)
        out, lse = balanced(q, k, v, lens, workgroups)
        check_decode(out[full], lse[full], q[full], k[full], v[full], lens[full])
        if dtype == torch.float32:
            ref = reference.decode(q[full].cpu(), k[full].cpu(), v[full].cpu(), lens[full].cpu())
            assert normwise_rel(out[full].cpu(), ref) <= 1e-5
        assert torch.all(out[~full] == 0) and torch.isneginf(lse[~full]).all()
        # The same keys in the same order from a paged pool, and on every run, give the same bits.
        for got in (balanced(q, k_pool, v_pool, lens, workgroups, tables), balanced(q, k, v, lens, workgroups)):
            assert torch.equal(got[0], out) and torch.equal(got[1], lse)


@pytest.mark.gpu
def test_planned_balanced_decode_replays_on_new_lengths():
    # The public entry point on a planned call, captured once and replayed after the lengths changed in
    # place: each replay equals the eager call, and the oracle.
    gen = torch.Generator(device="cuda").manual_seed(5)
    batch, heads, heads_kv, pages, head_dim = 40, 32, 8, 256, 128
    assert plan(batch, heads, heads_kv, head_dim, pages * 16, page_size=16)[1] == 256
    q = torch.randn(batch, 1, heads, head_dim, device="cuda", dtype=torch.bfloat16, generator=gen)
    k, v = (torch.randn(batch * pages, 16, heads_kv, head_dim, device="cuda", dtype=torch.bfloat16, generator=gen)
            for _ in range(2))
    tables = torch.randperm(batch * pages, device="cuda", generator=gen).to(torch.int32).reshape(batch, pages)
    lens = torch.full((batch,), pages * 16, device="cuda", dtype=torch.int32)
    flash_lab.decode(q, k, v, lens, block_tables=tables)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out, lse = flash_lab.decode(q, k, v, lens, block_tables=tables, return_lse=True)
    for low, high in ((4096, 4097), (0, 4097), (1, 40), (3000, 3200)):
        lens.copy_(torch.randint(low, high, (batch,), device="cuda", generator=gen))
        print(f"balanced replay, lengths in [{low}, {high})", flush=True)
        graph.replay()
        torch.cuda.synchronize()
        want = flash_lab.decode(q, k, v, lens, block_tables=tables, return_lse=True)
        assert torch.equal(out, want[0]) and torch.equal(lse, want[1])
        for b in (0, batch - 1):
            n = int(lens[b])
            if n == 0:
                assert torch.all(out[b] == 0) and torch.isneginf(lse[b]).all()
                continue
            blocks = tables[b, : -(-n // 16)].long()
            kc, vc = (t[blocks].flatten(0, 1)[None, :n] for t in (k, v))
            check_decode(out[b : b + 1], lse[b : b + 1], q[b : b + 1], kc, vc, lens[b : b + 1])


# One long sequence among short ones on one KV head, its row cut into more partials than the merge pass
# takes at a time (128): (batch, longest, workgroups, partials that the long row has at least). The last
# one's rows are not padded to whole chunks.
LONG_ROWS = [(2, 20000, 300, 129), (2, 36000, 300, 257), (64, 32000, 229, 129)]


def long_row_lens(batch, longest):
    lens = [1 + 7 * i % 32 for i in range(batch)]
    lens[batch // 2 - 1] = longest
    return lens


@pytest.mark.parametrize("ramp_units", [2, 4])  # vector and matrix-core kernel
def test_long_rows_have_more_partials_than_one_merge_step(ramp_units):
    for batch, longest, workgroups, least in LONG_ROWS:
        lens = long_row_lens(batch, longest)
        chunk, starts, sizes = schedule(lens, 1, workgroups, 32, 4, ramp_units)
        row = batch // 2 - 1
        assert (starts[row] + -(-longest // 32) - 1) // chunk - starts[row] // chunk + 1 >= least
        assert (starts[row] % chunk != 0) == (batch == 64)


@pytest.mark.gpu
@pytest.mark.parametrize("heads,dtype", [(8, torch.bfloat16), (8, torch.float32), (3, torch.bfloat16),
                                         (2, torch.float16), (1, torch.float32)], ids=str)
@pytest.mark.parametrize("case", LONG_ROWS, ids=str)
def test_rows_of_many_partials_match_reference(case, heads, dtype):
    batch, longest, workgroups, _ = case
    print(f"balanced long row {case} heads={heads} {dtype}", flush=True)
    q, k, v, lens = inputs((batch, heads, 1, longest, 64, long_row_lens(batch, longest)), dtype)
    out, lse = balanced(q, k, v, lens, workgroups)
    check_decode(out, lse, q, k, v, lens)
    if dtype == torch.float32:
        assert normwise_rel(out.cpu(), reference.decode(q.cpu(), k.cpu(), v.cpu(), lens.cpu())) <= 1e-5
    again = balanced(q, k, v, lens, workgroups)
    assert torch.equal(again[0], out) and torch.equal(again[1], lse)


# Layouts beside the contiguous [B, S, H_kv, D] one: transposed caches, query heads a stride apart, pages
# of 1 and 7 rows. 8 rows of 992 keys on 8 workgroups of the matrix-core kernel: with pages of one row
# every segment's block numbers nearly fill their 1,024 places in LDS.
LAYOUT_CASES = [
    (4, 8, 2, 992, 128, [992, 992, 992, 992], 8),
    (9, 16, 4, 2002, 64, "random", 256),
    (6, 4, 4, 1500, 64, [1500, 0, 1, 33, 999, 1499], 100),
]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("case", LAYOUT_CASES, ids=lambda c: f"B{c[0]}-H{c[1]}-Hkv{c[2]}-S{c[3]}-D{c[4]}")
def test_balanced_decode_on_other_layouts(case, dtype):
    *shape, workgroups = case
    print(f"balanced layouts {case} {dtype}", flush=True)
    q, k, v, lens = inputs(tuple(shape), dtype)
    q = q.repeat_interleave(2, dim=2)[:, :, ::2]
    kt, vt = (x.transpose(1, 2).contiguous().transpose(1, 2) for x in (k, v))
    out, lse = balanced(q, kt, vt, lens, workgroups)
    full = lens > 0
    check_decode(out[full], lse[full], q[full], k[full], v[full], lens[full])
    assert torch.all(out[~full] == 0) and torch.isneginf(lse[~full]).all()
    for page in (1, 7):
        (k_pool, tables), (v_pool, _) = paged(k, page), paged(v, page)
        print(f"pages of {page}", flush=True)
        got = balanced(q, k_pool, v_pool, lens, workgroups, tables)
        if tables.shape[1] * page == k.shape[1]:  # the same capacity: the same keys per workgroup
            assert torch.equal(got[0], out) and torch.equal(got[1], lse)
        check_decode(got[0][full], got[1][full], q[full], k[full], v[full], lens[full])


# Infinities and NaN in one sequence's cache: what a fixed split count gives for it, and no effect on the
# others. fp32 (eight query heads) and groups of 1 and 3 run on the vector kernel. An infinite value is at
# every place of a 32-key unit in turn, among them the last keys of workgroups' segments.
@pytest.mark.gpu
@pytest.mark.parametrize("heads_kv,group,dtype", [(2, 1, torch.bfloat16), (1, 3, torch.bfloat16),
                                                  (1, 8, torch.float32), (1, 8, torch.float16)], ids=str)
def test_balanced_decode_with_infinities_and_nan(heads_kv, group, dtype):
    batch, longest = 3, 3000
    q, k, v, lens = inputs((batch, heads_kv * group, heads_kv, longest, 64, [2990, 700, 3000]), dtype)
    q = q * 0.1  # no probability underflows
    workgroups = 45 * heads_kv  # five units each: a segment ends within a batch of 64 or 128 keys
    assert schedule([2990, 700, 3000], heads_kv, workgroups, 32, 4, 2)[0] == 5
    want, want_lse = balanced(q, k, v, lens, workgroups)
    vector = dtype == torch.float32 or group < 4
    print(f"balanced non-finite {heads_kv} {group} {dtype}", flush=True)
    infinite = v.clone()
    places = 2528 + 33 * torch.arange(14, device="cuda")  # from its 79th unit on, each at another place in it
    places = places[places < 2990 - 1]
    infinite[0, places, 0, 3] = float("inf")
    infinite[0, 127:2528:32, 0, 5] = -float("inf")  # last keys of units
    for num_splits in (None, 1, 7):
        if num_splits is None:
            out, lse = balanced(q, k, infinite, lens, workgroups)
            assert torch.equal(out[1:], want[1:]) and torch.equal(lse, want_lse)
        else:
            out, lse = flash_lab.decode(q, k, infinite, lens, num_splits=num_splits, return_lse=True)
        assert torch.isposinf(out[0, 0, :group, 3]).all() and torch.isneginf(out[0, 0, :group, 5]).all()
        rest = out.clone()
        rest[0, 0, :group, [3, 5]] = 0
        assert torch.isfinite(rest).all()
    for bad in (float("nan"), float("inf")):
        broken = k.clone()
        broken[0, 1234, 0] = bad
        out, lse = balanced(q, broken, v, lens, workgroups)
        assert torch.equal(out[1:], want[1:]) and torch.equal(lse[1:], want_lse[1:])
        if vector:
            fixed, fixed_lse = flash_lab.decode(q, broken, v, lens, num_splits=7, return_lse=True)
            assert torch.equal(out[0, 0, :group], fixed[0, 0, :group])
            assert torch.equal(lse[0, :group], fixed_lse[0, :group])
            assert torch.equal(out[0, 0, group:], want[0, 0, group:])
