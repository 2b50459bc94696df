"""bf16 attention over key ranges of few 64-key tiles: a tile's PV product is
taken in the next tile's step, from a ring of three V stages, so the first
steps, the last one and the ring's wrap are where it can go wrong.

Bound: P is rounded to bf16 (relative 2^-9) under weights that sum to 1 within
the same rounding, the output once more, so |out - exact| <= 3 * 2^-9 max|V|
+ the scores' fp32 error, which is below 1e-3 max|V| for |score| <= 64.
"""

import math

import pytest
import torch

from kvpersist import api

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _case(keys, heads, scale, seed):
    g = torch.Generator().manual_seed(seed)
    D = heads * 128
    q, k, v = (torch.randn(keys, D, generator=g) for _ in range(3))
    # scores grow with the key, so every tile raises the running maximum
    k = k * torch.linspace(0.2, scale, keys)[:, None]
    return tuple(x.to(torch.bfloat16).to(DEV) for x in (q, k, v))


def _exact(q, k, v, heads):
    q, k, v = (x.double().cpu().view(-1, heads, 128).transpose(0, 1).contiguous()
               for x in (q, k, v))
    p = torch.softmax(q @ k.transpose(1, 2).contiguous() / math.sqrt(128.0), dim=-1)
    return (p @ v).transpose(0, 1).reshape(q.shape[1], heads * 128)


def _run(q, k, v, heads, arena=None, kvmap=None):
    out = torch.full_like(q, float("nan"))
    api.attn_forward_single_frame_bf16(q, k, v, arena, kvmap, out, q.shape[0], heads * 128, heads,
                                       0, 0, 0)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("scale", [1.0, 4.0])
@pytest.mark.parametrize("keys", [1, 63, 64, 65, 128, 129, 191, 192, 193, 256, 320, 449])
def test_tile_counts(keys, scale):
    heads = 2
    q, k, v = _case(keys, heads, scale, seed=keys)
    got = _run(q, k, v, heads)
    err = (got.double().cpu() - _exact(q, k, v, heads)).abs().max()
    assert float(err) <= (3 * 2.0 ** -9 + 1e-3) * float(v.abs().max())

    # rows taken from the arena, one by one or as whole groups: same bits
    g = torch.Generator().manual_seed(keys + 1)
    group = torch.arange(keys) // 16 % 3
    chosen = (group == 1) | ((group == 2) & (torch.rand(keys, generator=g) < 0.5))
    chosen[0] = True
    rows = chosen.nonzero().flatten()
    arena = torch.cat([k.cpu()[rows], v.cpu()[rows]], dim=1)
    kvmap = torch.full((keys,), -1, dtype=torch.int64)
    kvmap[rows] = torch.arange(len(rows))
    kb, vb = k.clone(), v.clone()
    kb[rows.to(DEV)] = float("nan")  # the original rows must not reach the sums
    vb[rows.to(DEV)] = float("nan")
    via_map = _run(q, kb, vb, heads, arena.to(DEV), kvmap.to(DEV))
    assert torch.equal(via_map, got)


@pytest.mark.parametrize("keys", [1023, 1024, 1025, 1089])
def test_tile_counts_around_a_short_walk(keys):
    """Without a map, walks of up to 16 tiles run a kernel whose first step is one of
    its own, longer ones start with a product of zeros; with one, all do the former."""
    test_tile_counts(keys, 4.0)
