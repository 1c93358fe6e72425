"""Prefill calls whose keys are split over several workgroups per block of rows (csrc/prefill_pp.hip,
the plan in prefill_splits): the plan and the workspace checks on the CPU, and on the GPU the split
counts at their edges (one tile per split, more splits than tiles, splits past a causal block's last
key, rows without keys, ragged last tiles and blocks) against the fp64 oracle.
"""

import ctypes

import pytest
import torch

import flash_lab
from flash_lab import _hip
from parity import PrefillOracle, check_prefill


def params(shape, causal=1):
    batch, seqlen_q, seqlen_k, heads, heads_kv, head_dim = shape
    p = _hip.AttnParams()
    p.batch, p.seqlen_q, p.seqlen_k = batch, seqlen_q, seqlen_k
    p.heads, p.heads_kv, p.head_dim, p.causal, p.dtype = heads, heads_kv, head_dim, causal, 0
    p.softmax_scale = 0.125
    return p


def plan(shape, requested=0, causal=1):
    splits, nbytes = ctypes.c_int32(), ctypes.c_size_t()
    rc = _hip.LIB.fl_attention_plan(ctypes.byref(params(shape, causal)), requested, 256,
                                    ctypes.byref(splits), ctypes.byref(nbytes))
    return rc, splits.value, nbytes.value


def test_plan():
    # Few rows and many keys are split, within one split per tile; grids that fill the CUs are not.
    for shape in [(1, 300, 8492, 32, 8, 128), (1, 16, 8192, 32, 8, 128), (2, 40, 200, 64, 1, 64)]:
        rc, splits, nbytes = plan(shape)
        assert rc == 0 and 1 <= splits <= min(64, -(-shape[2] // 64))
        assert (nbytes == 0) == (splits == 1)
    assert plan((1, 300, 8492, 32, 8, 128))[1] > 1
    for shape in [(4, 4096, 4096, 32, 32, 128), (1, 512, 512, 32, 8, 128), (1, 1, 1, 1, 1, 64)]:
        assert plan(shape) == (0, 1, 0)
    # Five blocks of 256 packed rows per KV head: partials of 256 rows, 128 + 2 floats each.
    assert plan((1, 300, 8492, 32, 8, 128), 6) == (0, 6, 8 * 5 * 256 * 6 * 130 * 4)
    for requested in (-1, 65):
        assert plan((1, 300, 8492, 32, 8, 128), requested)[0] == 1


def test_knobs_that_pin_a_kernel_keep_the_keys_unsplit(knobs):
    shape = (1, 300, 8492, 32, 8, 128)
    want = plan(shape)
    knobs("prefill_causal_stream", 0)  # the default's own value changes nothing
    assert plan(shape) == want and want[1] > 1
    knobs("prefill_causal_stream", 1)
    assert plan(shape) == (0, 1, 0)
    knobs("prefill_causal_stream", None)
    knobs("prefill_pp_min_wg", 256)
    assert plan(shape) == (0, 1, 0)


def test_workspace_is_checked_before_any_launch():
    p = params((1, 300, 8492, 32, 8, 128))
    buf = torch.empty(1024, dtype=torch.int64)
    ptr = buf.data_ptr() + (-buf.data_ptr()) % 64
    p.q = p.k = p.v = p.o = p.lse = ptr
    for t in "qkvo":
        for s, n in (("batch", 0), ("seq", 4096), ("head", 128)):
            setattr(p, f"{t}_{s}_stride", n)
    need = plan((1, 300, 8492, 32, 8, 128), 6)[2]
    for splits, workspace, nbytes, want in [(6, None, need, 1), (6, ptr, need - 4, 1), (6, ptr + 4, need, 1),
                                            (-1, ptr, need, 1), (65, ptr, need, 1),
                                            (0, None, 0, _hip.ERR_WORKSPACE), (0, ptr, 64, _hip.ERR_WORKSPACE)]:
        rc = _hip.LIB.fl_attention_fwd_split(ctypes.byref(p), splits, 256, workspace, nbytes, None)
        assert rc == want, (splits, workspace, nbytes)


def split_prefill(q, k, v, causal, scale, num_splits):
    """fl_attention_fwd_split with this split count, whatever the plan would choose."""
    batch, seqlen_q, heads, head_dim = q.shape
    shape = (batch, seqlen_q, k.shape[1], heads, k.shape[2], head_dim)
    out, lse = torch.empty(q.shape, dtype=q.dtype, device="cuda"), torch.empty(batch, heads, seqlen_q, device="cuda")
    p = _hip.AttnParams(*(t.data_ptr() for t in (q, k, v, out, lse)), *q.stride()[:3], *k.stride()[:3],
                        *v.stride()[:3], *out.stride()[:3], *shape, int(causal), _hip.DTYPE_CODES[q.dtype], scale)
    nbytes = plan(shape, num_splits)[2]
    workspace = torch.full((nbytes // 4,), float("nan"), device="cuda")
    _hip._check(_hip.LIB.fl_attention_fwd_split(ctypes.byref(p), num_splits, 256, workspace.data_ptr(), nbytes,
                                                torch.cuda.current_stream().cuda_stream))
    return out, lse


SHAPES = [
    # batch, seqlen_q, seqlen_k, heads, heads_kv, head_dim
    (1, 1, 65, 8, 2, 128),  # two tiles, the second with one key
    (2, 70, 300, 12, 4, 128),  # 210 packed rows: a block whose last wave has 18
    (1, 300, 300, 8, 8, 128),  # causal from the first key: blocks of different lengths
    (2, 130, 40, 4, 2, 128),  # S_q > S_k: positions without keys, a block with none
    (1, 97, 513, 20, 4, 64),  # 485 packed rows: two 384-row blocks
    (3, 33, 128, 2, 1, 64),  # whole tiles only
]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_split_counts_match_reference(shape, causal, dtype):
    batch, seqlen_q, seqlen_k, heads, heads_kv, head_dim = shape
    q = torch.randn(batch, heads, seqlen_q, head_dim, device="cuda", dtype=dtype).transpose(1, 2)
    k = torch.randn(batch, seqlen_k, heads_kv, head_dim, device="cuda", dtype=dtype)
    v = torch.randn(batch, heads_kv, seqlen_k, head_dim, device="cuda", dtype=dtype).transpose(1, 2)
    oracle = PrefillOracle(q, k, v, causal)
    scale = head_dim**-0.5
    for num_splits in (2, 3, 9, 64):
        print(f"split prefill {shape} {dtype} causal={causal} splits={num_splits}", flush=True)
        out, lse = split_prefill(q, k, v, causal, scale, num_splits)
        oracle.check(out, lse)
        again = split_prefill(q, k, v, causal, scale, num_splits)
        assert torch.equal(out, again[0]) and torch.equal(lse, again[1])


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 300, 4000, 32, 8, 128), (4, 17, 3000, 32, 4, 64)], ids=str)
def test_planned_splits_match_reference_and_replay(shape):
    # The public entry point on planned splits, eager and captured: every replay gives the eager bits.
    batch, seqlen_q, seqlen_k, heads, heads_kv, head_dim = shape
    assert plan(shape)[1] > 1
    q = torch.randn(batch, seqlen_q, heads, head_dim, device="cuda", dtype=torch.bfloat16)
    k, v = (torch.randn(batch, seqlen_k, heads_kv, head_dim, device="cuda", dtype=torch.bfloat16)
            for _ in range(2))
    print(f"planned splits {shape}", flush=True)
    out, lse = flash_lab.attention(q, k, v, causal=True, return_lse=True)
    check_prefill(out, lse, q, k, v, True)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got, got_lse = flash_lab.attention(q, k, v, causal=True, return_lse=True)
    for _ in range(3):
        got.fill_(7)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, out) and torch.equal(got_lse, lse)
        flash_lab.attention(q, k, v, causal=True)


# Infinities and NaN in the keys and values of one KV head: what the unsplit forms and torch give (an
# infinite value is the output's, a NaN score makes the row NaN), wherever in the splits' shares and in the
# halves of a tile they are, and no effect on the other heads. (1, 150, 300, 8, 2): half tiles where not split.
@pytest.mark.gpu
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("num_splits", [1, 2, 3, 9])
def test_infinities_and_nan(num_splits, head_dim, knobs):
    knobs("prefill_pp_min_wg", 1 << 30)
    q = torch.randn(1, 150, 8, head_dim, device="cuda", dtype=torch.bfloat16) * 0.1  # no probability underflows
    k, v = (torch.randn(1, 300, 2, head_dim, device="cuda", dtype=torch.bfloat16) for _ in range(2))

    def call(k, v):
        if num_splits == 1:
            return flash_lab.attention(q, k, v, return_lse=True)
        return split_prefill(q, k, v, False, head_dim**-0.5, num_splits)

    want, want_lse = call(k, v)
    for key in (0, 31, 40, 63, 64, 191, 256, 299):
        print(f"non-finite prefill splits={num_splits} D={head_dim} key={key}", flush=True)
        infinite = v.clone()
        infinite[0, key, 0, 3], infinite[0, key, 0, 5] = float("inf"), -float("inf")
        out, lse = call(k, infinite)
        assert torch.isposinf(out[:, :, :4, 3]).all() and torch.isneginf(out[:, :, :4, 5]).all()
        out[:, :, :4, [3, 5]] = want[:, :, :4, [3, 5]]
        assert torch.equal(out, want) and torch.equal(lse, want_lse)
        for bad in (float("nan"), float("inf")):
            broken = k.clone()
            broken[0, key, 0] = bad
            out, lse = call(broken, v)
            assert torch.isnan(out[:, :, :4]).all() and not torch.isfinite(lse[:, :4]).any()
            assert torch.equal(out[:, :, 4:], want[:, :, 4:]) and torch.equal(lse[:, 4:], want_lse[:, 4:])
