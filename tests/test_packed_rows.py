"""The prefill kernels' packed rows: the query heads of one KV head run as one sequence of rows, row r
being position r / group of head r % group, with the division done as a multiplication on the host's
constants (csrc/abi.hip, csrc/launch.hpp). The CPU test checks that arithmetic over its range; the GPU
tests run both kernels, both causal orders of the ping-pong kernel and group sizes that are not powers
of two across the edges of 32-row waves and 128-, 256- and 384-row blocks, against the fp64 oracle.
"""

import random

import pytest
import torch

import flash_lab
from parity import check_prefill


def magic(pack):
    shift = 31
    while (1 << (shift - 31)) < pack:
        shift += 1
    return (1 << shift) // pack + 1, shift


@pytest.mark.parametrize("pack", [1, 2, 3, 4, 5, 6, 7, 8, 12, 16, 31, 32, 64, 71, 128, 1000, 65535])
def test_division_by_multiplication(pack):
    mul, shift = magic(pack)
    assert mul < 1 << 32
    rng = random.Random(pack)
    rows = {0, 1, pack - 1, pack, pack + 1, (1 << 31) - 1, (1 << 30) - 1}
    for _ in range(2000):
        multiple = rng.randrange((1 << 31) // pack) * pack
        rows |= {multiple, max(0, multiple - 1), rng.randrange(1 << 31)}
    assert all((r * mul) >> shift == r // pack for r in rows)


SHAPES = [
    # batch, seqlen_q, seqlen_k, heads, heads_kv, head_dim; packed rows per KV head in the comment
    (8, 43, 43, 24, 8, 128),  # 129: one row past a 128-row block
    (16, 85, 150, 12, 4, 64),  # 255, and S_q < S_k
    (8, 37, 37, 56, 8, 64),  # 259, group 7
    (8, 129, 64, 48, 16, 128),  # 387 rows, S_q > S_k: positions without keys
    (16, 1, 77, 32, 2, 128),  # 16, one position
    (4, 200, 200, 40, 8, 64),  # 1,000, group 5: three 384-row blocks
]


@pytest.mark.gpu
@pytest.mark.parametrize("min_wg", [0, 1 << 30], ids=["pingpong", "wg128"])
@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_packed_rows_match_reference(shape, causal, min_wg, knobs):
    knobs("prefill_pp_min_wg", min_wg)
    batch, seqlen_q, seqlen_k, heads, heads_kv, head_dim = shape
    print(f"packed rows {shape} causal={causal} min_wg={min_wg}", flush=True)
    q = torch.randn(batch, heads, seqlen_q, head_dim, device="cuda", dtype=torch.bfloat16).transpose(1, 2)
    k = torch.randn(batch, seqlen_k, heads_kv, head_dim, device="cuda", dtype=torch.bfloat16)
    v = torch.randn(batch, heads_kv, seqlen_k, head_dim, device="cuda", dtype=torch.bfloat16).transpose(1, 2)
    out, lse = flash_lab.attention(q, k, v, causal=causal, return_lse=True)
    check_prefill(out, lse, q, k, v, causal)


# Causal orders of the ping-pong kernel at head_dim 128: 130 work heads of four 256-row blocks are 260
# pairs, 51% of two rounds of 256 (single blocks, heaviest first); 128 work heads are one full round
# (pairs). The last block is partly empty in both.
@pytest.mark.gpu
@pytest.mark.parametrize("batch", [65, 64])
def test_causal_block_orders(batch):
    print(f"causal order, batch {batch}", flush=True)
    q, k, v = (torch.randn(batch, 490, h, 128, device="cuda", dtype=torch.bfloat16) for h in (4, 2, 2))
    out, lse = flash_lab.attention(q, k, v, causal=True, return_lse=True)
    check_prefill(out, lse, q, k, v, True, rows=torch.arange(0, 490, 7))


# Causal calls with one ping-pong block per query head in one round: separate heads where the packed rows
# would be fewer than 128 pairs of that kernel's blocks and more than 256 of the 4-wave kernel's, packed at 256
# of these.
@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(8, 186, 186, 32, 4, 128), (8, 128, 200, 32, 4, 128), (3, 250, 594, 64, 8, 64)],
                         ids=str)
def test_one_round_of_heads(shape):
    print(f"one round of heads {shape}", flush=True)
    batch, seqlen_q, seqlen_k, heads, heads_kv, head_dim = shape
    q = torch.randn(batch, seqlen_q, heads, head_dim, device="cuda", dtype=torch.bfloat16)
    k, v = (torch.randn(batch, heads_kv, seqlen_k, head_dim, device="cuda", dtype=torch.bfloat16).transpose(1, 2)
            for _ in range(2))
    out, lse = flash_lab.attention(q, k, v, causal=True, return_lse=True)
    check_prefill(out, lse, q, k, v, True)
