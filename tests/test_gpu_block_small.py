"""Block attention of at most 48 query tokens (attn.hip, HALVES): the edges of its row tiles and of
the 64-key tiles whose halves different waves take, with one key split and several, short
splits and long ones."""

import math

import pytest
import torch

from helpers import bf16_ulp

pytestmark = pytest.mark.gpu
BF, HQ, HKV, D = torch.bfloat16, 32, 8, 128


def _masks(B, T, tree, g):
    """Visibility [B, T, T] and, for trees, the ancestor words [B, T]."""
    vis = torch.eye(T, dtype=torch.bool).repeat(B, 1, 1)
    if not tree:
        return torch.ones(B, T, T, dtype=torch.bool).tril(), None
    for b in range(B):
        for j in range(1, T):
            vis[b, j] |= vis[b, int(torch.randint(0, j, (1,), generator=g))]
    words = [[sum(1 << j for j in range(T) if vis[b, t, j]) for t in range(T)] for b in range(B)]
    return vis, torch.tensor(words, dtype=torch.int64, device="cuda")


@pytest.mark.parametrize("tree", [True, False])
@pytest.mark.parametrize("T", [1, 15, 16, 17, 31, 32, 33, 47, 48, 49])
@pytest.mark.parametrize("B,base,spare", [(1, 0, 0), (2, 31, 5), (3, 33, 700), (2, 1500, 0), (9, 64, 3), (9, 2100, 3)])
def test_small_blocks(B, base, spare, T, tree):
    from qdecode import ops
    print(f"\n[case] B={B} T={T} base={base} spare={spare} tree={tree}", flush=True)
    g = torch.Generator()
    g.manual_seed(1000 * T + base + B)
    cap = base + T + spare
    rnd = lambda *s, std=1.0: (torch.randn(s, generator=g) * std).to(BF).cuda()  # noqa: E731
    q, k, v = rnd(B, T, HQ, D, std=2.0), rnd(B, HKV, cap, D), rnd(B, HKV, cap, D)
    k[:, :, base + T:] = float("nan")            # slots that no token sees
    v[:, :, base + T:] = 0
    vis, anc = _masks(B, T, tree, g)
    got = ops.block_attention(q, k, v, torch.full((B,), base, dtype=torch.int64, device="cuda"), anc=anc)
    n = base + T
    seen = torch.cat((torch.ones(B, T, base, dtype=torch.bool), vis), 2).cuda()
    qd = q.double().view(B, T, HKV, 4, D)
    for h in range(HKV):
        kk, vv = k[:, h, :n].double(), v[:, h, :n].double()
        for i in range(4):
            s = (qd[:, :, h, i] @ kk.transpose(1, 2).contiguous()) / math.sqrt(D)
            p = torch.softmax(s.masked_fill(~seen, -math.inf), -1)
            want = p @ vv
            # each probability is rounded to bf16 once (2^-9 relative; as much again covers the
            # fp32 scores, exponentials and sums), the result once
            bound = 2.0 ** -8 * (p @ vv.abs()) + bf16_ulp(want.float()).double()
            d = (got[:, :, 4 * h + i].double() - want).abs()
            assert bool((d <= bound).all()), f"head {4 * h + i}: {float((d - bound).max())}"


# a cache with room for much more than it holds, and keys on both sides of the counts (2 and 7 tiles of
# 64) from which a workgroup's split takes the half-tile form: 17..48 tokens
@pytest.mark.parametrize("tree", [True, False])
@pytest.mark.parametrize("T", [17, 32, 33, 48])
@pytest.mark.parametrize("keys", [60, 128, 129, 448, 449, 513, 1100])
def test_form_by_keys(keys, T, tree):
    test_small_blocks(2, keys - T, 4096 - keys, T, tree)
