"""The matrix-core decode kernel (16-bit heads of 64 to 128) where it can go
wrong: contexts at the edges of its 16- and 32-token tiles and of a partition,
every query-head count it pads to 16, small blocks, missing blocks, and cache
rows past a context that hold NaN and infinity."""

import numpy as np
import pytest
import torch

from helpers import pkg

pytestmark = pytest.mark.gpu

ops = pkg("paged_ops")

CONTEXTS = [1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 129, 160, 257, 500]


def build(heads, kv_heads, dim, dtype, block, contexts, holes=False, seed=0):
    device = torch.device("cuda", 0)
    gen = torch.Generator(device=device)
    gen.manual_seed(seed)
    need = [-(-c // block) for c in contexts]
    blocks = sum(need) + 3
    # Rows no context holds: NaN keys, infinite values.
    kc = torch.full((1, blocks, block, kv_heads, dim), float("nan"), device=device, dtype=dtype)
    vc = torch.full((1, blocks, block, kv_heads, dim), float("inf"), device=device, dtype=dtype)
    perm = np.random.Generator(np.random.PCG64(seed)).permutation(blocks)
    table = np.full((len(contexts), max(need)), -1, dtype=np.int32)
    live, at = [], 0
    for i, (c, n) in enumerate(zip(contexts, need)):
        table[i, :n] = perm[at:at + n]
        at += n
        pos = np.arange(c)
        slots = torch.from_numpy(table[i, pos // block].astype(np.int64) * block + pos % block).to(device)
        kc.view(-1, kv_heads, dim)[slots] = torch.randn((c, kv_heads, dim), generator=gen, device=device).to(dtype)
        vc.view(-1, kv_heads, dim)[slots] = torch.randn((c, kv_heads, dim), generator=gen, device=device).to(dtype)
        keep = np.ones(c, dtype=bool)
        if holes and n > 2:  # a missing block in the middle and one outside the pool
            table[i, n // 2] = -1
            keep &= pos // block != n // 2
            if n > 4:
                table[i, 1] = blocks
                keep &= pos // block != 1
        live.append(slots[torch.from_numpy(keep).to(device)])
    q = torch.randn((len(contexts), heads, dim), generator=gen, device=device).to(dtype)
    return q, kc, vc, torch.from_numpy(table).to(device), live


def reference(q, kc, vc, live, scale):
    """The attention in 64 bits, and the weighted mean of |v| beside it (what
    the errors of the probabilities scale with)."""
    kv_heads, dim = kc.shape[3], kc.shape[4]
    group = q.shape[1] // kv_heads
    out, size = [], []
    for i, slots in enumerate(live):
        k = kc.view(-1, kv_heads, dim)[slots].double().repeat_interleave(group, dim=1)
        v = vc.view(-1, kv_heads, dim)[slots].double().repeat_interleave(group, dim=1)
        p = torch.softmax((k * q[i].double()).sum(-1).t() * scale, dim=-1).t().unsqueeze(-1)
        out.append((p * v).sum(0))
        size.append((p * v.abs()).sum(0))
    return torch.stack(out), torch.stack(size)


def check(heads, kv_heads, dim, dtype, block, partition, contexts=CONTEXTS, holes=False):
    q, kc, vc, table, live = build(heads, kv_heads, dim, dtype, block, contexts, holes)
    scale = 1.0 / np.sqrt(dim)
    step = ops.pack_step(table, [c - 1 for c in contexts], [1] * len(contexts), block, num_kv_heads=kv_heads,
                         num_query_heads=heads, head_dim=dim, dtype=dtype, partition_size=partition)
    out = ops.decode(q, kc, vc, 0, step, scale).double()
    ref, size = reference(q, kc, vc, live, scale)
    assert torch.isfinite(out).all()
    # The result is rounded once, by half a unit in its last place (relative u).
    # A probability enters the product as two terms of the cache type, off by
    # u^2 at most; scores of up to 128 products, their exponentials and sums are
    # fp32: about 1e-5 of a probability.  (One rounded to the cache type alone
    # would be off by u, and a tile left out of 4096 tokens moves the result
    # by 100 times the bound.)
    u = 2.0**-8 if dtype == torch.bfloat16 else 2.0**-11
    excess = ((out - ref).abs() - (1 + 2 * u) * u * ref.abs() - (u * u + 1.5e-5) * size).max().item()
    assert excess <= 0, excess


@pytest.mark.parametrize("heads,kv_heads", [(1, 1), (3, 3), (9, 3), (10, 2), (7, 1), (16, 2), (9, 1), (22, 2), (16, 1),
                                            (17, 1), (40, 2), (64, 1), (2, 2), (12, 4), (16, 4), (4, 4)])
@pytest.mark.parametrize("dim", [64, 80, 96, 128])
def test_groups(heads, kv_heads, dim):
    check(heads, kv_heads, dim, torch.bfloat16, 16, 128)


@pytest.mark.parametrize("block", [1, 2, 4, 8, 16, 32, 64])
@pytest.mark.parametrize("holes", [False, True])
@pytest.mark.parametrize("heads,kv_heads,dim", [(16, 1, 128), (15, 3, 64), (8, 2, 128), (4, 4, 64), (6, 3, 96)])
def test_blocks(block, holes, heads, kv_heads, dim):
    check(heads, kv_heads, dim, torch.float16, block, 96, holes=holes)


@pytest.mark.parametrize("partition", [32, 64, 4096])
@pytest.mark.parametrize("heads,kv_heads,dim", [(16, 1, 128), (10, 2, 64), (8, 2, 128), (6, 6, 64), (20, 2, 80)])
def test_partitions(partition, heads, kv_heads, dim):
    check(heads, kv_heads, dim, torch.bfloat16, 16, partition, contexts=[1, 31, 32, 33, 64, 700, 4095, 4096, 4097])
