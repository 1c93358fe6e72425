"""The 4-wave prefill kernel with two waves to each 32 rows, one 32-key half of every 64-key tile each
(csrc/prefill_fwd.hip, kParts = 2), at its edges: keys that end inside the first half, at its end and
one past it, causal rows whose last tile is only in the first half, rows without keys, one-row blocks,
and a dominant key that only one of the halves sees, against the fp64 oracle.
"""

import pytest
import torch

import flash_lab
from parity import check_prefill

pytestmark = pytest.mark.gpu

SHAPES = [
    # batch, seqlen_q, seqlen_k, heads, heads_kv, head_dim
    (1, 65, 65, 8, 8, 128),  # a second block of one row, a second tile of one key
    (1, 70, 96, 4, 1, 128),  # the last tile is one half
    (1, 64, 97, 4, 2, 64),  # ... and one key of the other
    (1, 33, 127, 8, 2, 64),
    (2, 130, 90, 4, 4, 128),  # S_q > S_k: positions without keys
    (1, 200, 650, 4, 4, 128),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("causal", [False, True], ids=["full", "causal"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_half_tiles_match_reference(shape, causal, dtype, knobs):
    knobs("prefill_pp_min_wg", 1 << 30)  # the 4-wave kernel, unsplit
    print(f"half tiles {shape} {dtype} causal={causal}", flush=True)
    batch, seqlen_q, seqlen_k, heads, heads_kv, head_dim = shape
    q = torch.randn(batch, seqlen_q, heads, head_dim, device="cuda", dtype=dtype)
    k, v = (torch.randn(batch, heads_kv, seqlen_k, head_dim, device="cuda", dtype=dtype).transpose(1, 2)
            for _ in range(2))
    out, lse = flash_lab.attention(q, k, v, causal=causal, return_lse=True)
    check_prefill(out, lse, q, k, v, causal)
    again = flash_lab.attention(q, k, v, causal=causal, return_lse=True)
    assert torch.equal(out, again[0]) and torch.equal(lse, again[1])


@pytest.mark.parametrize("key", [5, 40, 100])
def test_dominant_key_in_one_half(key, knobs):
    knobs("prefill_pp_min_wg", 1 << 30)
    print(f"half tiles, dominant key {key}", flush=True)
    q, k, v = (torch.randn(1, 150, 2, 128, device="cuda") for _ in range(3))
    k[:, key] = q[:, 20] / q[:, 20].norm(dim=-1, keepdim=True) * 60
    q, k, v = (x.to(torch.bfloat16) for x in (q, k, v))
    out, lse = flash_lab.attention(q, k, v, return_lse=True)
    check_prefill(out, lse, q, k, v, False)
