"""The reference ABI's flat call at the edges of the flat kernel's launch
shapes: list segments of 8192 and 4096 slots, both sides of the 384-workgroup rule,
head dims that fill, straddle and miss the lane layouts."""

import numpy as np
import pytest
import torch

from helpers import pkg
from oracle import attention as oa

pytestmark = pytest.mark.gpu

ops = pkg("paged_ops")


def flat_case(tokens, heads, kv_heads, dim, context, density, seed):
    rng = np.random.Generator(np.random.PCG64(seed))
    blocks, bs = 61, 16
    kc = rng.standard_normal((2, blocks, bs, kv_heads, dim), dtype=np.float32)
    vc = rng.standard_normal((2, blocks, bs, kv_heads, dim), dtype=np.float32)
    q = rng.standard_normal((1, heads, tokens, dim), dtype=np.float32)
    slots = rng.integers(0, blocks * bs, size=context).astype(np.int32)
    mask = (rng.random((tokens, context)) < density).astype(np.uint8)
    if tokens > 1:
        mask[1] = 0  # attends nothing: zeros
    return q, kc, vc, slots, mask


# (tokens, heads, kv heads, head dim, context slots, attended share).  384
# workgroups (of 1-4 heads) are the last of 16 waves each (segments of 8192
# slots), 385 the first of 4 (4096).
CASES = [
    (1, 1, 1, 4, 1, 1.0),
    (3, 4, 2, 12, 63, 0.5),
    (2, 6, 2, 64, 8192, 0.02),
    (2, 6, 2, 64, 8193, 1.0),
    (48, 8, 8, 64, 257, 0.3),
    (55, 7, 7, 64, 4097, 0.05),
    (99, 8, 4, 72, 129, 0.5),
    (3, 8, 1, 128, 1471, 0.2),
    (130, 4, 4, 128, 65, 1.0),
    (130, 9, 3, 128, 300, 0.4),
    (385, 4, 1, 100, 40, 0.6),
    (5, 20, 4, 64, 900, 0.4),
    (2, 3, 3, 132, 300, 0.7),
    (2, 2, 1, 256, 8200, 0.1),
    (390, 2, 1, 256, 70, 0.9),
    # Groups of 4 and 3 on rows of 256: at 16 waves the kernel's largest LDS.
    (3, 8, 2, 256, 8200, 0.1),
    (2, 6, 2, 192, 300, 0.7),
    (200, 8, 2, 256, 90, 0.8),
    (200, 6, 2, 252, 4099, 0.05),
    (3, 2, 2, 6, 200, 0.5),  # rows of half pieces: the one-wave kernel
]


@pytest.mark.parametrize("tokens,heads,kv_heads,dim,context,density", CASES)
def test_flat_call_matches_oracle(tokens, heads, kv_heads, dim, context, density):
    device = torch.device("cuda", 0)
    q, kc, vc, slots, mask = flat_case(tokens, heads, kv_heads, dim, context, density, seed=dim * 1000 + context)
    scale = 1.0 / np.sqrt(dim)
    ref = oa.paged_attention(q, kc, vc, 1, slots, mask[None, None], scale)
    # Slots outside the pool are skipped: the oracle masks them instead.
    live = slots.copy()
    bad = np.arange(context) % 5 == 3
    live[bad] = np.where(np.arange(context)[bad] % 2 == 0, -1, kc.shape[1] * kc.shape[2])
    ref_bad = oa.paged_attention(q, kc, vc, 1, slots, (mask * ~bad).astype(np.uint8)[None, None], scale)
    on = lambda x: torch.from_numpy(x).to(device)
    for s, want in ((slots, ref), (live, ref_bad)):
        got = ops.paged_attention_flat(on(q), on(kc), on(vc), 1, on(s), on(mask)[None, None], scale)
        # fp32 dots of up to 256 terms and sums of up to 8200 weights: errors
        # of a few 1e-6 of values of order 1; the path's bound is 1e-4.
        assert np.max(np.abs(got.cpu().numpy() - want.reshape(got.shape))) <= 1e-4


def test_flat_call_takes_unaligned_rows():
    """A query and caches that start 4 bytes past a 16-byte boundary."""
    device = torch.device("cuda", 0)
    q, kc, vc, slots, mask = flat_case(3, 4, 2, 64, 300, 0.5, seed=1)
    ref = oa.paged_attention(q, kc, vc, 0, slots, mask[None, None], 0.125)

    def shifted(x):
        t = torch.empty(x.size + 1, device=device)[1:].view(x.shape)
        t.copy_(torch.from_numpy(x))
        return t

    got = ops.paged_attention_flat(shifted(q), shifted(kc), shifted(vc), 0, torch.from_numpy(slots).to(device),
                                   torch.from_numpy(mask).to(device)[None, None], 0.125)
    assert np.max(np.abs(got.cpu().numpy() - ref.reshape(got.shape))) <= 1e-4
