"""Tiled products whose blocks are no more than the compute units: a ring in LDS as deep as it holds."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("slabs", [1, 2, 6, 7, 8, 9, 15, 31])
@pytest.mark.parametrize("M,N", [(65, 1100), (449, 1030)])
def test_a_deep_ring_gives_the_bits_of_a_shallow_one(M, N, slabs):
    """Small tiles: one accumulator an output, products in ascending k, so that the rows of a product of few blocks (ring of eight) come out as among many rows (ring of three)."""
    from alofa_amd import ops
    g = torch.Generator(device=DEV).manual_seed(slabs)
    many, K = 1100, 64 * slabs
    a, w, b = torch.randn(many, K, generator=g, device=DEV).bfloat16(), torch.randn(N, K, generator=g, device=DEV).bfloat16(), torch.randn(N, generator=g, device=DEV)
    want, out = torch.empty(many, N, device=DEV), torch.full((M, N), float("nan"), device=DEV)
    ops.gemm(want, a, w, b, kernel="tiled")
    ops.gemm(out, a[:M], w, b, kernel="tiled")
    assert torch.equal(out, want[:M])
    exact = a.double() @ w.double().T + b
    assert (want - exact).abs().max().item() <= (K + 1) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T).max().item() + 1e-5      # (a float sum of K products and the bias)


@pytest.mark.parametrize("M,N,K", [(17, 4000, 320), (64, 4000, 576), (33, 11000, 2048), (64, 3000, 2112), (100, 1000, 64), (200, 1000, 384), (300, 4000, 256), (200, 3000, 4096),
                                   (40, 500, 4096), (500, 1000, 8192), (1000, 1500, 4160)])
def test_every_form_with_a_deep_ring(M, N, K):
    """Gate and up, and sums onto the residual stream, in tiles of 64 and of 128 rows, whole and with K in shares; fewer slabs than the ring holds and more, edges in both directions."""
    from alofa_amd import ops
    g = torch.Generator(device=DEV).manual_seed(K)
    a, w, u = (torch.randn(n, K, generator=g, device=DEV).bfloat16() for n in (M, N, N))
    ws, us = (w.float() * K ** -0.5).bfloat16(), (u.float() * K ** -0.5).bfloat16()
    x, y = a.double() @ ws.double().T, a.double() @ us.double().T
    bound = (K + 1) * 2.0 ** -24 * (a.double().abs() @ ws.double().abs().T).max().item()
    acc = torch.ones(M, N, device=DEV)
    ops.gemm(acc, a, ws, add_to_out=True, kernel="tiled")
    assert (acc - (x + 1)).abs().max().item() <= bound + 1e-5
    out = torch.full((M, N), float("nan"), device=DEV, dtype=torch.bfloat16)
    ops.gemm_swiglu(out, a, ws, us, kernel="tiled")
    want = torch.nn.functional.silu(x) * y
    assert (out.double() - want).abs().max().item() <= want.abs().max().item() * 2.0 ** -8 + 2 * bound
