"""GPU: the 16x16x32 key split (flash_fwd_ksplit) at the edges of its steps, parts and rows.

Lengths around a key tile, a step of two or four tiles, the switch to the 32x32x16 key split and
the four-way split's causal extension; inputs that leave the optimistic softmax (a row max that
jumps far past 2^16 in a later step, a part whose keys all lie far below the others', so that its
merge weight underflows); scales 0, negative and large; O and the LSE against the fp32 oracle.
CPU: the order of the two-round causal grids is a permutation that ends with the longest blocks'
partners.
"""

from __future__ import annotations

import pytest
import torch

from conftest import ATOL, RTOL
from oracle import attention as orc
from test_geometry import geo  # noqa: F401


def _check(q, k, v, causal, scale=None):
    import fa

    o, lse = fa.forward_lse(q.cuda(), k.cuda(), v.cuda(), causal=causal, softmax_scale=scale)
    o, lse = o.cpu(), lse.cpu()
    b, h = q.shape[:2]
    for bi, hi in {(0, 0), (b - 1, h - 1)}:
        sl = (slice(bi, bi + 1), slice(hi, hi + 1))
        torch.testing.assert_close(o[sl].float(),
                                   orc.attention_fp32(q[sl], k[sl], v[sl], causal, scale),
                                   atol=ATOL, rtol=RTOL)
        torch.testing.assert_close(lse[sl], orc.lse_fp32(q[sl], k[sl], causal, scale), atol=2e-3,
                                   rtol=0)


def _qkv(b, h, n, d, seed):
    g = torch.Generator().manual_seed(seed)
    return tuple(torch.randn(b, h, n, d, generator=g).half() for _ in range(3))


# (d, N): one to a few tiles (32 keys at d = 128, 64 at d = 64), steps of two and four tiles
EDGES = [(128, n) for n in (1, 31, 33, 64, 65, 96, 97, 129, 480, 481, 512, 545)] + \
        [(64, n) for n in (384, 385, 447, 449, 513, 577, 960, 961, 1025, 1089)]


@pytest.mark.gpu
@pytest.mark.parametrize("d,n", EDGES)
@pytest.mark.parametrize("causal", [False, True])
def test_edge_lengths(d, n, causal):
    print(f"case edge d={d} N={n} causal={causal}", flush=True)
    _check(*_qkv(2, 3, n, d, seed=n + d), causal)


# both sides of the rows' bounds: the grids over 400 blocks (32x32x16 up to 800 keys causal, 448 at
# d = 64), the four-way split's causal extension (2560 and 4096 keys), the two-round order
BOUNDS = [(1, 62, 500, 64, True), (1, 62, 801, 64, True), (1, 50, 449, 64, False),
          (1, 62, 700, 128, True), (1, 34, 768, 128, True), (1, 8, 2559, 128, True),
          (1, 8, 2560, 128, True), (1, 5, 4095, 64, True), (1, 5, 4097, 64, True),
          (1, 16, 2000, 128, True), (1, 20, 1800, 64, True)]


@pytest.mark.gpu
@pytest.mark.parametrize("b,h,n,d,causal", BOUNDS)
def test_both_sides_of_the_rules(b, h, n, d, causal):
    print(f"case bound B={b} H={h} N={n} d={d} causal={causal}", flush=True)
    _check(*_qkv(b, h, n, d, seed=n + h), causal)


@pytest.mark.gpu
@pytest.mark.parametrize("d,n", [(128, 300), (128, 700), (64, 700), (64, 1500)])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("kind", ["jump", "low part", "scales"])
def test_softmax_paths_and_merge(d, n, causal, kind):
    print(f"case {kind} d={d} N={n} causal={causal}", flush=True)
    q, k, v = _qkv(1, 3, n, d, seed=n)
    if kind == "scales":
        for scale in (0.0, -0.2, 1.5):
            _check(q, k, v, causal, scale)
        return
    q[..., 0] = 4.0
    level = torch.zeros(n)
    if kind == "jump":      # +40 log2 units from the middle on
        level[n // 2:] = 40.0
    else:                   # every second key tile 200 log2 units below the rest
        tile = 4096 // d
        level[torch.arange(n) // tile % 2 == 1] = -200.0
    k[..., 0] = (level * 0.6931 * d ** 0.5 / 4.0).half()
    _check(q, k, v, causal)


@pytest.mark.parametrize("total", [1, 256, 257, 288, 400, 511, 512, 513, 1000])
def test_two_round_order_is_a_permutation(geo, total):  # noqa: F811
    got = [geo.geom_two_round_turn(i, total) for i in range(total)]
    assert sorted(got) == list(range(total))
    if 256 < total <= 512:
        assert got[256] == total - 1 and got[:256] == list(range(256))
    else:
        assert got == list(range(total))
