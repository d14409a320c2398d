"""The 32-bit path's kernels with float64 sums on the matrix cores, at the edges of their tiles, against float64 on the host."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
ONCE = 2.0 ** -23      # an output is rounded to float once (half a unit in the last place), a sum with the residual stream twice


def ops():
    from alofa_amd import ops as o
    return o


def t(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV)


def within(got, want, parts):
    """|got - want| <= parts roundings of the terms' size."""
    got, want = got.cpu().double().numpy(), np.asarray(want, dtype=np.float64)
    assert np.all(np.isfinite(got)) and np.all(np.abs(got - want) <= ONCE * parts), np.abs((got - want) / parts).max()


# rows up to 16, 32 and beyond (three kernels' forms), tiles' edges, K short, ragged and shared out, unaligned rows
@pytest.mark.parametrize("M,N,K,shift", [(1, 16, 32, 0), (8, 896, 4864, 0), (16, 17, 31, 0), (16, 5000, 36, 0), (5, 70000, 64, 0), (17, 33, 260, 0), (32, 129, 1000, 0),
                                         (33, 64, 128, 0), (64, 896, 4864, 0), (65, 130, 2056, 0), (200, 97, 1030, 0), (8, 130, 200, 1), (40, 70, 512, 1), (450, 1152, 896, 0)])
def test_exact_products(M, N, K, shift):
    rng = np.random.default_rng(M * 1000 + N)
    a, w, w2, b, res = (rng.standard_normal(s).astype(np.float32) for s in ((M, K + shift), (N, K + shift), (N, K + shift), (N,), (M, N)))
    ta, tw, tw2 = t(a)[:, shift:], t(w)[:, shift:], t(w2)[:, shift:]
    want = a[:, shift:].astype(np.float64) @ w[:, shift:].astype(np.float64).T
    up = a[:, shift:].astype(np.float64) @ w2[:, shift:].astype(np.float64).T
    out = torch.full((M, N + 3), 7.0, device=DEV)
    ops().gemm(out[:, :N], ta, tw, t(b), exact=True)
    within(out[:, :N], want + b, np.abs(want + b) + 1e-7)
    assert bool((out[:, N:] == 7.0).all())
    acc = t(res)
    ops().gemm(acc, ta, tw, add_to_out=True, exact=True)
    within(acc, want + res, np.abs(want) + np.abs(want + res) + 1e-7)
    ops().gemm_swiglu(out[:, :N], ta, tw, tw2, exact=True)
    gate = want / (1.0 + np.exp(-want))
    within(out[:, :N], gate * up, 4 * np.abs(gate * up) * (1 + np.abs(want)) + 1e-7)      # (gate and up are rounded before the activation, whose slope is its size at most)
    again = torch.empty(M, N, device=DEV)
    ops().gemm(again, ta, tw, t(b), exact=True)
    ops().gemm(out[:, :N], ta, tw, t(b), exact=True)
    assert torch.equal(again, out[:, :N])      # a fixed order, whatever the timing


@pytest.mark.parametrize("heads,kv_heads,d,bs,requests", [(14, 2, 64, 16, 3), (20, 1, 32, 4, 2), (33, 1, 16, 12, 2), (4, 4, 112, 16, 2), (2, 1, 160, 8, 2), (8, 2, 128, 64, 70)])
@pytest.mark.parametrize("window", [None, 19])
def test_exact_attention(heads, kv_heads, d, bs, requests, window):
    rng = np.random.default_rng(heads + d)
    lens = [1 + (i * 37) % 90 + (100 if i == 0 else 0) for i in range(requests)]      # from one key on, past a page's and a tile's end
    brings = [n if i == 1 else min(n, 1 + i % 2) for i, n in enumerate(lens)]      # a whole prompt and single tokens
    per = [(n + bs - 1) // bs for n in lens]
    order = rng.permutation(sum(per) + 1)
    kc = torch.full((sum(per) + 1, kv_heads, bs, d), float("nan"), dtype=torch.float32)      # (what no token has written is never read into a result)
    vc = torch.full((sum(per) + 1, kv_heads, d, bs), float("nan"), dtype=torch.float32)
    table = torch.full((requests, max(per)), -1, dtype=torch.int32)
    rows, req, pos, want, used = [], [], [], [], 0
    for i, (n, m) in enumerate(zip(lens, brings)):
        pages = order[used:used + per[i]]
        used += per[i]
        lowest = 0 if window is None else max(0, n - m - window + 1)
        k, v, q = (torch.from_numpy(rng.standard_normal(s).astype(np.float32)) for s in ((n, kv_heads, d), (n, kv_heads, d), (m, heads, d)))
        for j in range(n):
            kc[pages[j // bs], :, j % bs], vc[pages[j // bs], :, :, j % bs] = k[j], v[j]
        for j, page in enumerate(pages):
            table[i, j] = -1 if (j + 1) * bs <= lowest else int(page)      # (pages that a window has passed are given back)
        rows.append(q.reshape(m, heads * d)), req.extend([i] * m), pos.extend(range(n - m, n))
        for j in range(m):
            p = n - m + j
            lo = 0 if window is None else max(0, p - window + 1)
            kk, vv = (x[lo:p + 1].double().repeat_interleave(heads // kv_heads, 1) for x in (k, v))
            s = torch.einsum("hd,khd->hk", q[j].double(), kk) * float(np.float32(d ** -0.5))
            want.append(torch.einsum("hk,khd->hd", torch.softmax(s, -1), vv).reshape(-1))
    out = torch.empty(len(req), heads * d, device=DEV)
    to = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)      # noqa: E731
    ops().paged_attention(out, torch.cat(rows).to(DEV), kc.to(DEV), vc.to(DEV), table.to(DEV), to(req), to(pos), heads, kv_heads, d, window, float(np.float32(d ** -0.5)), True)
    # a weight: its score's rounding (some units of 2^-23 at scores of up to six), expf's two units; the values are of order one
    within(out, torch.stack(want).numpy(), 12.0)


# gate and up of tiles of 96 rows (where they are the fewer rounds of the chip): their edges, K ragged, columns of no whole tile
@pytest.mark.parametrize("M,N,K", [(66, 4864, 896), (96, 4864, 100), (95, 4833, 68), (450, 4864, 128), (385, 4810, 36)])
def test_exact_gate_and_up_of_taller_tiles(M, N, K):
    gen = torch.Generator(device=DEV).manual_seed(M)
    a, g, u = (torch.randn(s, generator=gen, device=DEV) * K ** -0.25 for s in ((M, K), (N, K), (N, K)))
    out = torch.full((M, N + 1), 7.0, device=DEV)
    ops().gemm_swiglu(out[:, :N], a, g, u, exact=True)
    gate, up = ((a.double() @ w.double().T.contiguous()).cpu().numpy() for w in (g, u))
    want = gate / (1.0 + np.exp(-gate)) * up
    within(out[:, :N], want, 4 * np.abs(want) * (1 + np.abs(gate)) + 1e-7)
    assert bool((out[:, N:] == 7.0).all())
    for first, n in ((0, 1), (60, 5), (1, 40), (0, 64)):      # (the same bits as in the other forms)
        part = torch.empty(n, N, device=DEV)
        ops().gemm_swiglu(part, a[first:first + n], g, u, exact=True)
        assert torch.equal(part, out[first:first + n, :N])


# slabs of 32 k: none whole, one to seven, with and without a rest, rows that are not 16-byte aligned, shares of unequal length
def test_taller_tiles_where_their_rounds_are_the_shorter():
    """A tile of 96 rows takes 1.55 times as long as one of 64: two rounds of the one do not make up for three of the other."""
    from alofa_amd.csrc.build import load
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    for M in (65, 96, 130, 190, 240, 390, 450, 480, 576, 960):
        for N in (1024, 2432, 4864, 5632, 8960, 11008, 13824, 18944):
            low, tall = (-(-(-(-N // 32) * -(-M // rows)) // cus) for rows in (64, 96))
            assert load().alofa_gemm_swiglu_exact_tile(M, N) == (96 if 1.55 * tall < low else 64), (M, N, low, tall)
    assert [load().alofa_gemm_swiglu_exact_tile(M, 4864) for M in (16, 17, 32, 33, 64)] == [16, 32, 32, 64, 64]


@pytest.mark.parametrize("M,N,K,shift", [(17, 40, 20, 0), (33, 70, 32, 0), (33, 70, 52, 0), (65, 70, 64, 0), (20, 140, 96, 0), (65, 70, 99, 0), (40, 64, 128, 0), (64, 64, 160, 1), (90, 70, 190, 1),
                                         (40, 70, 228, 0), (200, 64, 1100, 0)])
def test_exact_products_by_slabs(M, N, K, shift):
    rng = np.random.default_rng(K)
    a, w = (rng.standard_normal(s).astype(np.float32) for s in ((M, K + shift), (N, K + shift)))
    want = a[:, shift:].astype(np.float64) @ w[:, shift:].astype(np.float64).T
    out = torch.empty(M, N, device=DEV)
    ops().gemm(out, t(a)[:, shift:], t(w)[:, shift:], exact=True)
    within(out, want, np.abs(want) + 1e-7)


# up to 16 rows against few columns and K so long that a share of 1,024 k a block would make more shares than are added up
@pytest.mark.parametrize("M,N,K", [(8, 64, 18944), (1, 128, 27648), (16, 16, 32768), (3, 240, 17408), (16, 31, 17500)])
def test_exact_products_of_few_rows_and_very_long_k(M, N, K):
    gen = torch.Generator(device=DEV).manual_seed(K + N)
    a, w, b, res = (torch.randn(s, generator=gen, device=DEV) for s in ((M, K), (N, K), (N,), (M, N)))
    want = (a.double() @ w.double().T.contiguous()).cpu().numpy()
    out = torch.empty(M, N, device=DEV)
    ops().gemm(out, a, w, b, exact=True)
    within(out, want + b.cpu().numpy(), np.abs(want + b.cpu().numpy()) + 1e-7)
    acc = res.clone()
    ops().gemm(acc, a, w, add_to_out=True, exact=True)
    within(acc, want + res.cpu().numpy(), np.abs(want) + np.abs(want + res.cpu().numpy()) + 1e-7)


# Every form (rows up to 16, 32 and beyond; chains of K in one block, over blocks, in rounds; two matrices; a vocabulary) adds up in one order: a row alone and the same row among
# others are the same bits. Pairs of 2^40 that cancel exactly lie far apart in k: what is summed between them loses its low bits, and another order loses others.
@pytest.mark.parametrize("N,K,shift", [(896, 896, 0), (896, 4864, 0), (17, 1030, 0), (130, 2056, 1), (70000, 200, 0), (33, 20000, 0), (4100, 3584, 0), (64, 127, 0), (48, 160, 0)])
def test_a_row_of_an_exact_product_does_not_depend_on_the_others(N, K, shift):
    gen = torch.Generator(device=DEV).manual_seed(N + K)
    rows = 40 if N > 10000 else 300
    a, w, b = (torch.randn(s, generator=gen, device=DEV) for s in ((rows, K + shift), (N, K + shift), (N,)))
    order = torch.randperm(K, generator=gen, device=DEV)[:K // 8 * 2] + shift
    plus, minus = order[::2], order[1::2]
    w[:, minus] = w[:, plus]
    a[:, plus] = torch.ldexp(a[:, plus], torch.tensor(40, device=DEV))
    a[:, minus] = -a[:, plus]
    a, w = a[:, shift:], w[:, shift:]
    want = torch.empty(rows, N, device=DEV)
    ops().gemm(want, a, w, b, exact=True)
    gate = torch.empty(rows, N // 2, device=DEV)
    ops().gemm_swiglu(gate, a, w[:N // 2], w[N // 2:N // 2 * 2], exact=True)
    stream = torch.randn(rows, N, generator=gen, device=DEV)
    added = stream.clone()
    ops().gemm(added, a, w, add_to_out=True, exact=True)
    for first, n in ((0, 1), (7, 5), (0, 16), (3, 17), (0, 32), (1, 33), (0, 64), (9, 65), (0, 200)):
        if first + n > rows:
            continue
        part = slice(first, first + n)
        out, half, acc = torch.empty(n, N, device=DEV), torch.empty(n, N // 2, device=DEV), stream[part].clone()
        ops().gemm(out, a[part], w, b, exact=True)
        ops().gemm_swiglu(half, a[part], w[:N // 2], w[N // 2:N // 2 * 2], exact=True)
        ops().gemm(acc, a[part], w, add_to_out=True, exact=True)
        assert torch.equal(out, want[part]) and torch.equal(acc, added[part]) and torch.equal(half, gate[part]), (first, n)


def test_exact_sums_of_many_rows_stay_bounded():
    from alofa_amd.csrc.build import load
    for M, N, K in ((64, 152064, 3584), (4096, 896, 4864), (100000, 896, 4864), (64, 20000, 8192), (65, 8192, 8192), (1, 128, 27648), (16, 240, 17408)):
        assert load().alofa_gemm_exact_parts(M, N, K) * 8 <= 64 << 20


def test_exact_products_whose_sums_go_to_memory_in_pieces():
    M, N, K = 1100, 500, 16384      # 16 chains, 64 KB of sums a row
    gen = torch.Generator(device=DEV).manual_seed(1)
    a, w, res = (torch.randn(s, generator=gen, device=DEV) for s in ((M, K), (N, K), (M, N)))
    acc = res.clone()
    ops().gemm(acc, a, w, add_to_out=True, exact=True)
    want = (a.double() @ w.double().T.contiguous()).cpu().numpy()
    within(acc, want + res.cpu().numpy(), np.abs(want) + np.abs(want + res.cpu().numpy()) + 1e-7)


@pytest.mark.parametrize("heads,kv_heads,d", [(14, 2, 64), (8, 1, 32), (6, 2, 160)])
def test_a_row_of_exact_attention_does_not_depend_on_the_others(heads, kv_heads, d):
    bs, rows, history = 16, 300, 500
    gen = torch.Generator(device=DEV).manual_seed(d)
    pages = -(-(rows + history) // bs)
    q = torch.randn(rows, heads * d, generator=gen, device=DEV) * 2
    kc, vc = torch.randn(pages, kv_heads, bs, d, generator=gen, device=DEV), torch.randn(pages, kv_heads, d, bs, generator=gen, device=DEV)
    table = torch.arange(pages, dtype=torch.int32, device=DEV)[None].contiguous()
    req, pos = torch.zeros(rows, dtype=torch.int32, device=DEV), torch.arange(history, history + rows, dtype=torch.int32, device=DEV)

    def attend(part):
        out = torch.empty_like(q[part])
        ops().paged_attention(out, q[part], kc, vc, table, req[part], pos[part], heads, kv_heads, d, None, d ** -0.5, True)
        return out
    want = attend(slice(0, rows))
    for first, n in ((0, 1), (299, 1), (5, 8), (17, 100), (100, 200)):
        assert torch.equal(attend(slice(first, first + n)), want[first:first + n])


def test_sums_of_chains_lie_in_the_callers_buffers(tiny_dirs):
    a, w, out = torch.ones(64, 4864, device=DEV), torch.ones(896, 4864, device=DEV), torch.empty(64, 896, device=DEV)
    room, asked = torch.empty(1 << 23, dtype=torch.float64, device=DEV), []

    def scratch(name, shape, dtype):
        asked.append((name, dtype))
        return room[:shape[0]]
    ops().gemm(out, a, w, exact=True)
    before = torch.cuda.memory_stats()["allocation.all.allocated"]
    ops().gemm(out, a, w, exact=True, scratch=scratch)
    assert torch.cuda.memory_stats()["allocation.all.allocated"] == before and asked == [("product_sums", torch.float64)] and bool((out == 4864).all())
    # an engine's steps, cut kernel by kernel and captured: the sums are among the buffers that its account of memory counts
    from alofa_amd.replay import Replayer
    r = Replayer(tiny_dirs["D"], "float32", 128)
    r.step({"step": 0, "entries": [{"id": "a", "tokens": list(range(20)), "want": []}], "end": []})
    for i in range(2):
        r.step({"step": 1 + i, "entries": [{"id": "a", "tokens": [7], "want": [0]}], "end": ["a"] if i else []})
    fn = r.fn
    eager, captured = fn._eager_scratch["product_sums", torch.float64], fn._graph_buffers[1]["scratch"]["product_sums", torch.float64]
    assert fn.graph_replays == 1 and fn.scratch_bytes() > 8 * (eager.numel() + captured.numel())


def test_exact_products_name_the_operand_that_is_not_float32():
    from alofa_amd.errors import AlofaError
    f, h = torch.ones(8, 64, device=DEV), torch.ones(8, 64, device=DEV, dtype=torch.bfloat16)
    out = torch.empty(8, 8, device=DEV)
    for operands, name in (((out, h, f), "operand=a"), ((out, f, h), "operand=w"), ((out.bfloat16(), f, f), "operand=out")):
        with pytest.raises(AlofaError, match=name):
            ops().gemm(*operands, exact=True)
    for operands, name in (((out, h, f, f), "operand=a"), ((out, f, h, h), "operand=w_gate"), ((out.bfloat16(), f, f, f), "operand=out")):
        with pytest.raises(AlofaError, match=name):
            ops().gemm_swiglu(*operands, exact=True)


# rows up to 16, 32, 64 and beyond, sums in one piece and in several, columns that fill a block's threads and more; where no sums go to memory the norm is a launch of its own
@pytest.mark.parametrize("M,N,K", [(1, 896, 896), (8, 896, 4864), (16, 64, 4864), (8, 1028, 2048), (3, 2052, 700), (17, 896, 4864), (64, 1024, 1024), (450, 896, 896), (1100, 500, 16384), (5, 4100, 1024), (9, 131, 3000)])
def test_exact_products_with_the_norm_behind_them(M, N, K):
    gen = torch.Generator(device=DEV).manual_seed(M + N)
    draw = lambda *s: torch.randn(s, generator=gen, device=DEV)      # noqa: E731
    a, w, weight, stream = draw(M, K), draw(N, K) * K ** -0.5, draw(N), draw(M, N)
    got = []
    for rides in (False, True):
        out, rows = stream.clone(), torch.empty(M, N, device=DEV)
        if rides:
            ops().gemm(out, a, w, add_to_out=True, exact=True, then_norm=(weight, 1e-6, rows))
        else:
            ops().gemm(out, a, w, add_to_out=True, exact=True)
            ops().rmsnorm(rows, out, weight, 1e-6, True)
        got.append((out, rows))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


# the new token at a tile's, a page's and a quad's first and last place, alone, behind a window; more heads to a key head than a tile holds
@pytest.mark.parametrize("heads,kv_heads,d,bs", [(14, 2, 64, 16), (20, 1, 32, 4), (4, 4, 96, 16), (6, 2, 64, 12)])
@pytest.mark.parametrize("window", [None, 19])
def test_a_decode_step_of_the_exact_path_turns_its_tokens(heads, kv_heads, d, bs, window):
    positions = [0, 1, 3, 4, 15, 16, 17, 31, 63, 64, 130, 255]
    n = len(positions)
    gen = torch.Generator(device=DEV).manual_seed(heads)
    draw = lambda *s: torch.randn(s, generator=gen, device=DEV)      # noqa: E731
    per = [p // bs + 1 for p in positions]
    pages = torch.randperm(sum(per), generator=gen, device=DEV).to(torch.int32)
    table = torch.full((n, max(per)), -1, dtype=torch.int32, device=DEV)
    used, slots = 0, []
    for i, p in enumerate(positions):
        mine = pages[used:used + per[i]]
        lowest = 0 if window is None else max(0, p - window + 1)
        table[i, :per[i]] = torch.where((torch.arange(per[i], device=DEV) + 1) * bs <= lowest, -1, mine)
        slots.append(int(mine[-1]) * bs + p % bs)
        used += per[i]
    kc, vc = draw(sum(per), kv_heads, bs, d), draw(sum(per), kv_heads, d, bs)
    for slot in slots:      # (what stands at a new token's place, and behind it, is not data)
        kc[slot // bs, :, slot % bs:], vc[slot // bs, :, :, slot % bs:] = float("nan"), float("nan")
    qkv, cos, sin = draw(n, (heads + 2 * kv_heads) * d), draw(300, d // 2), draw(300, d // 2)
    to = lambda x, t=torch.int32: torch.tensor(x, dtype=t, device=DEV)      # noqa: E731
    pos, req, slots = to(positions), to(range(n)), to(slots, torch.int64)
    got = []
    for turned in (False, True):
        rows, k, v, out = qkv.clone(), kc.clone(), vc.clone(), torch.empty(n, heads * d, device=DEV)
        if not turned:
            ops().rope_kv_write(rows, cos, sin, pos, heads, kv_heads, d, slots, k, v)
        assert ops().can_turn_exactly(rows, k, v, d)
        ops().paged_attention(out, rows, k, v, table, req, pos, heads, kv_heads, d, window, d ** -0.5, True, rope=(cos, sin, slots) if turned else None)
        got.append((out, k.nan_to_num(7.0), v.nan_to_num(7.0)))
    assert all(torch.equal(a, b) for a, b in zip(*got)) and bool(torch.isfinite(got[0][0]).all())
    assert torch.equal(rows, qkv)


# gate and up of up to 16 rows dealt out over the compute units (256 here): 17 to 24 outputs a block, the last block with fewer, one before and one behind the range; K ragged and of several rounds of chains
@pytest.mark.parametrize("M", [1, 8, 16])
@pytest.mark.parametrize("N,K", [(4096, 64), (4097, 64), (4113, 896), (4864, 896), (4865, 99), (6144, 132), (6145, 64), (5000, 2100)])
def test_exact_gate_and_up_of_few_rows_dealt_out(M, N, K):
    gen = torch.Generator(device=DEV).manual_seed(N + K)
    a, g, u = (torch.randn(s, generator=gen, device=DEV) * K ** -0.25 for s in ((M, K), (N, K), (N, K)))
    out = torch.full((M, N + 1), 7.0, device=DEV)
    ops().gemm_swiglu(out[:, :N], a, g, u, exact=True)
    gate, up = ((a.double() @ w.double().T.contiguous()).cpu().numpy() for w in (g, u))
    want = gate / (1.0 + np.exp(-gate)) * up
    within(out[:, :N], want, 4 * np.abs(want) * (1 + np.abs(gate)) + 1e-7)
    assert bool((out[:, N:] == 7.0).all())
    for first in (0, N - 1000):      # (the same bits as in blocks of sixteen outputs)
        part = torch.empty(M, 1000, device=DEV)
        ops().gemm_swiglu(part, a, g[first:first + 1000].contiguous(), u[first:first + 1000].contiguous(), exact=True)
        assert torch.equal(part, out[:, first:first + 1000])
