"""The GEMM kernels behind the usual ones, against fp64 products: activation rows too far apart for
32-bit offsets."""

import pytest
import torch

from helpers import bf16_ulp

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.fixture(scope="module")
def ops():
    from qdecode import ops as o
    return o


def _rnd(g, *s, std=1.0):
    return torch.empty(s, dtype=BF, device="cuda").normal_(0, std, generator=g)


def _check(ops, epi, x, N, g, **kw):
    """ops.linear over x with random weights, each output within the roundings of its epilogue."""
    K = x.shape[1]
    w, res = _rnd(g, 2 * N if epi == ops.EPI_SWIGLU else N, K, std=0.05), _rnd(g, x.shape[0], N, std=2.0)
    got = ops.linear(x, w, epi, res=res if epi == ops.EPI_RES else None, **kw).float()
    a = (x.double() @ w.double().t()).to(BF).float()
    if epi == ops.EPI_SWIGLU:
        # one ulp in bf16(gate), bf16(up) and bf16(silu) each, propagated, and two of the output
        gate, up = a[:, :N], a[:, N:]
        sg = torch.sigmoid(gate)
        s = (gate * sg).to(BF).float()
        want = (s * up).to(BF).float()
        bound = (up.abs() * ((sg * (1 + gate * (1 - sg))).abs() * bf16_ulp(gate) + bf16_ulp(s))
                 + s.abs() * bf16_ulp(up) + 2 * bf16_ulp(torch.maximum(got.abs(), want.abs())) + 2 ** -12)
    elif epi == ops.EPI_RES:
        want = (res.float() + a).to(BF).float()
        bound = bf16_ulp(a) + 2 * bf16_ulp(torch.maximum(got.abs(), want.abs()))
    else:
        want = a
        bound = 2 * bf16_ulp(torch.maximum(got.abs(), want.abs())) + 2 ** -9
    d = (got - want).abs()
    assert bool((d <= bound).all()), f"max excess {float((d - bound).max())}"


# the skinny kernel's buffer extent (32 rows), the four-wave kernel's offsets (33 and 300 rows, in
# both plans) and the all-rows kernel's (100 and 200): each row count beyond its 32-bit reach
@pytest.mark.parametrize("epi", [0, 1, 2])
@pytest.mark.parametrize("M,stride", [(32, 70_000_000), (33, 8_400_000), (100, 21_800_000),
                                      (200, 10_900_000), (300, 8_400_000)])
def test_long_row_strides(ops, M, stride, epi):
    print(f"\n[case] {M} rows of stride {stride}, epilogue {epi}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(M + epi)
    K = 1024
    x = torch.empty((M - 1) * stride + K, dtype=BF, device="cuda").as_strided((M, K), (stride, 1))
    x.copy_(_rnd(g, M, K))
    _check(ops, epi, x, 512, g)                  # its workspace: K splits where the plan has them
    _check(ops, epi, x, 512, g, ws=torch.zeros(256, dtype=torch.uint8, device="cuda"))
