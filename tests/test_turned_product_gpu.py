"""The product of a step's queries, keys and values that turns them and writes the cache on its way out."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def both(M, heads, kv_heads, K, d=64, page=16, start=0, bias=True, strided=False, shuffled=False, seed=0):
    """([queries, key cache, value cache] by two launches, by ``gemm_turned``)"""
    from alofa_amd import ops
    g = torch.Generator().manual_seed(seed)
    N, hd = (heads + 2 * kv_heads) * d, heads * d
    a, w = torch.randn(M, K, generator=g).bfloat16().to(DEV), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16().to(DEV)
    b = torch.randn(N, generator=g).to(DEV) if bias else None
    angles = torch.rand(M + start + 3, d // 2, generator=g) * 6
    cos, sin = angles.cos().to(DEV), angles.sin().to(DEV)
    n_pages = (M + start) // page + 2
    slots = torch.arange(start, start + M) if not shuffled else torch.randperm(n_pages * page, generator=g)[:M]
    positions = torch.randint(0, M + start + 3, (M,), generator=g).int().to(DEV)
    out = []
    for how in (0, 1):
        wide = torch.zeros(M, N + (24 if strided else 0), dtype=torch.bfloat16, device=DEV)
        qkv = wide[:, 8 * strided:8 * strided + N]
        k, v = torch.full((n_pages, kv_heads, page, d), 7., dtype=torch.bfloat16, device=DEV), torch.full((n_pages, kv_heads, d, page), 7., dtype=torch.bfloat16, device=DEV)
        if how:
            ops.gemm_turned(qkv, a, w, b, cos, sin, positions, slots.to(DEV), k, v, heads, kv_heads, d)
        else:
            ops.gemm(qkv, a, w, b)
            ops.rope_kv_write(qkv, cos, sin, positions, heads, kv_heads, d, slots.to(DEV), k, v)
        out.append((qkv[:, :hd].clone(), k, v, qkv[:, hd:].clone()))
    return out


@pytest.mark.parametrize("M,heads,kv_heads,K", [(17, 1, 1, 64), (63, 4, 1, 256), (64, 14, 2, 896), (17, 64, 8, 1984), (40, 40, 4, 1984), (65, 3, 3, 512), (65, 1, 1, 64), (201, 14, 2, 896),
                                                (1100, 14, 2, 640), (1030, 9, 3, 1984), (1500, 28, 4, 768), (600, 40, 8, 128)])
@pytest.mark.parametrize("page,start,shuffled,strided", [(16, 0, False, False), (8, 3, False, True), (64, 8, True, False), (1, 0, True, False)])
def test_the_bits_of_two_launches(M, heads, kv_heads, K, page, start, shuffled, strided):
    """Few blocks and many, one slab of K and more than the ring holds, rows that end inside a tile and inside eight of a page; runs of slots that begin at a page, inside one, and none; pages of a token.
    Against the product as ``gemm`` runs it, whichever kernel that is: up to 64 rows of the smaller matrices go by two launches."""
    from alofa_amd import ops
    from alofa_amd.csrc.build import load
    N = (heads + 2 * kv_heads) * 64
    assert load().alofa_gemm_turns(M, N, K, 64)
    two, one = both(M, heads, kv_heads, K, page=page, start=start, shuffled=shuffled, strided=strided, bias=not strided, seed=M)
    assert all(torch.equal(x, y) for x, y in zip(two[:3], one[:3]))
    assert bool(one[3].any()) == (ops.few_rows_kernel(M, N, K) != "tiled")      # (one launch: keys and values are in the cache only)


@pytest.mark.parametrize("M,K,d,page", [(16, 256, 64, 16), (70, 2048, 64, 16), (70, 256, 32, 16), (70, 256, 128, 16), (70, 264, 64, 16), (70, 256, 64, 12), (40, 2048, 64, 16), (40, 256, 64, 12)])
def test_what_the_product_does_not_take_is_two_launches(M, K, d, page):
    two, one = both(M, 4, 2, K, d=d, page=page)
    assert all(torch.equal(x, y) for x, y in zip(two[:3], one[:3]))
    assert one[3].any()


def test_under_capture():
    from alofa_amd import ops
    M, H, KV, K = 70, 4, 2, 256
    (q, k, v, _), _ = both(M, H, KV, K)
    g = torch.Generator().manual_seed(0)
    N = (H + 2 * KV) * 64
    a, w = torch.randn(M, K, generator=g).bfloat16().to(DEV), (torch.randn(N, K, generator=g) * K ** -0.5).bfloat16().to(DEV)
    b, angles = torch.randn(N, generator=g).to(DEV), torch.rand(M + 3, 32, generator=g) * 6
    cos, sin, slots, positions = angles.cos().to(DEV), angles.sin().to(DEV), torch.arange(M, device=DEV), torch.randint(0, M + 3, (M,), generator=g).int().to(DEV)
    qkv, kc, vc = torch.zeros(M, N, dtype=torch.bfloat16, device=DEV), torch.full_like(k, 7.), torch.full_like(v, 7.)
    run = lambda: ops.gemm_turned(qkv, a, w, b, cos, sin, positions, slots, kc, vc, H, KV, 64)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        run()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            run()
    for _ in range(3):
        qkv.zero_(), kc.fill_(7.), vc.fill_(7.)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(qkv[:, :H * 64], q) and torch.equal(kc, k) and torch.equal(vc, v)
