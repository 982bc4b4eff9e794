"""The GEMM kernels behind the usual ones, against fp64 products: activation rows too far apart for
32-bit offsets, and at 33 to 64 rows the widths, alignments and vocabularies that the four-wave kernel does
not take."""

import pytest
import torch

from helpers import check_linear

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.fixture(scope="module")
def ops():
    from qdecode import ops as o
    return o


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
    x.normal_(0, 1, generator=g)
    check_linear(ops, epi, x, 512, g)                  # its workspace: K splits where the plan has them
    check_linear(ops, epi, x, 512, g, ws=torch.zeros(256, dtype=torch.uint8, device="cuda"))


# N is not a multiple of 128 (SwiGLU: 64): the LDS-staged kernel (K a multiple of 512) and the plain
# one, at odd widths too
@pytest.mark.parametrize("epi", [0, 1, 2])
@pytest.mark.parametrize("N,K", [(192, 1024), (96, 512), (72, 512), (161, 1024), (192, 640), (96, 128)])
@pytest.mark.parametrize("M", [33, 48, 64])
def test_widths_at_33_to_64_rows(ops, M, N, K, epi):
    if epi == ops.EPI_SWIGLU and N % 64 == 0:
        N += 32
    print(f"\n[case] {M} x {N} x {K}, epilogue {epi}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(M + N + K + epi)
    x = torch.empty((M, K), dtype=BF, device="cuda").normal_(0, 1, generator=g)
    check_linear(ops, epi, x, N, g)


# on both sides of the columns and K at which whole products of 33 to 64 rows stay on the LDS-staged
# kernel, with room for split partials and without
@pytest.mark.parametrize("epi", [0, 1, 2])
@pytest.mark.parametrize("N,K", [(128, 512), (1024, 1024), (2048, 1536), (2048, 2048), (1024, 2560), (1152, 2560),
                                 (2048, 4096), (2176, 1024)])
@pytest.mark.parametrize("M", [33, 64])
def test_narrow_products_at_33_to_64_rows(ops, M, N, K, epi):
    print(f"\n[case] {M} x {N} x {K}, epilogue {epi}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(M + N + K + epi)
    x = torch.empty((M, K), dtype=BF, device="cuda").normal_(0, 1, generator=g)
    check_linear(ops, epi, x, N, g)
    check_linear(ops, epi, x, N, g, ws=torch.zeros(256, dtype=torch.uint8, device="cuda"))


@pytest.mark.parametrize("M", [33, 64])
def test_unaligned_output_at_33_to_64_rows(ops, M):
    """Output rows that start 2 bytes off: not the four-wave kernel's 8-byte stores."""
    g = torch.Generator(device="cuda")
    g.manual_seed(M)
    x = torch.empty((M, 1024), dtype=BF, device="cuda").normal_(0, 1, generator=g)
    buf = torch.full((M, 260), 7.0, dtype=BF, device="cuda")
    check_linear(ops, 0, x, 256, g, out=buf[:, 1:257])
    assert bool((buf[:, :1] == 7).all()) and bool((buf[:, 257:] == 7).all())


# a vocabulary that is no multiple of 4, or under 256: the weight-streaming kernel (K a multiple of 512)
# and the LDS-staged and plain ones
@pytest.mark.parametrize("V,K", [(50257, 1024), (4099, 2560), (250, 512), (1001, 640), (37, 256)])
@pytest.mark.parametrize("M", [33, 48, 64])
def test_lm_head_vocabularies_at_33_to_64_rows(ops, M, V, K):
    print(f"\n[case] lm_head_argmax {M} rows, vocabulary {V}, K {K}", flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(M + V)
    rnd = lambda *s, std: torch.empty(s, dtype=BF, device="cuda").normal_(0, std, generator=g)  # noqa: E731
    x, w, nw = rnd(M, K, std=1.0), rnd(V, K, std=0.02), rnd(K, std=0.1) + 1
    logits = torch.empty((M, V), dtype=torch.float32, device="cuda")
    tok = ops.lm_head_argmax(x, w, nw, 1e-6, logits=logits)
    # against the kernel's own normalised rows the logits carry fp32 accumulation error only
    want = ops.rmsnorm(x, nw, 1e-6).double() @ w.double().t()
    assert float((logits.double() - want).abs().max()) <= 1e-4
    assert torch.equal(tok.cpu(), torch.argmax(logits.to(BF).float().cpu(), dim=-1))


# the vocabularies from which 33 to 64 rows take the four-wave kernel (48 blocks of 320), and the tile
# shapes of 129 rows and more
@pytest.mark.parametrize("M,V", [(33, 15040), (64, 15044), (129, 256), (129, 16000), (192, 40064), (193, 40064),
                                 (257, 33152)])
def test_lm_head_tile_shapes(ops, M, V):
    test_lm_head_vocabularies_at_33_to_64_rows(ops, M, V, 1024)
