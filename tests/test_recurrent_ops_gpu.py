"""Each mechanism of the layers with state alone: the kernel against the plain function of the same equation, with
rows of several requests in one call, state carried from call to call, and sizes that no tile divides."""
import numpy as np
import pytest
import torch

from plain import tugalix as pt

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def rows_of(spans, n_slots):
    """spans: [(slot, rows)] in the order of the step's rows."""
    from alofa_amd import ops
    slots = torch.tensor([s for s, _ in spans], dtype=torch.int32, device=DEV)
    total = sum(n for _, n in spans)
    if all(n == 1 for _, n in spans):
        return ops.RowsOfRequests(slots, None, None, len(spans), total, n_slots)
    offsets = torch.tensor(np.concatenate([[0], np.cumsum([n for _, n in spans])]), dtype=torch.int32, device=DEV)
    req = torch.tensor([i for i, (_, n) in enumerate(spans) for _ in range(n)], dtype=torch.int32, device=DEV)
    return ops.RowsOfRequests(slots, offsets, req, len(spans), total, n_slots)


def dev(x, dtype=torch.float32):
    return torch.tensor(np.asarray(x), dtype=dtype, device=DEV).contiguous()


def cuts(n, sizes):
    out, at, k = [], 0, 0
    while at < n:
        m = min(sizes[k % len(sizes)], n - at)
        out.append((at, at + m))
        at, k = at + m, k + 1
    return out


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("width", [48, 1000])
def test_layer_norm(width, exact):
    from alofa_amd import ops
    rng = np.random.default_rng(0)
    x, w, b = rng.normal(2.0, 3.0, (9, width)), rng.normal(1, 0.2, width), rng.normal(0, 0.5, width)
    want = pt.layer_norm(x.astype(np.float32).astype(np.float64), w.astype(np.float32), b.astype(np.float32), 1e-5)
    out = torch.empty(9, width, device=DEV)
    ops.layernorm(out, dev(x), dev(w), dev(b), 1e-5, exact)
    assert np.abs(out.cpu().numpy() - want).max() <= (2e-6 if exact else 2e-5)
    rows = torch.tensor([8, 0, 3], dtype=torch.int32, device=DEV)
    some = torch.empty(3, width, device=DEV)
    ops.layernorm(some, dev(x), dev(w), dev(b), 1e-5, exact, rows)
    assert torch.equal(some, out[[8, 0, 3]])
    inplace = dev(x)
    ops.layernorm(inplace, inplace, dev(w), dev(b), 1e-5, exact)
    assert torch.equal(inplace, out)


@pytest.mark.parametrize("taps", [1, 2, 3, 4, 9, 16])
def test_short_convolution_in_portions_of_two_requests(taps):
    """Two requests whose rows arrive in unequal portions within the same calls; the state carries the last rows."""
    from alofa_amd import ops
    rng = np.random.default_rng(taps)
    width, n_slots = 40, 5
    h = {5: rng.normal(0, 1, (23, width)), 2: rng.normal(0, 1, (17, width))}      # by slot
    w = rng.normal(0, 0.5, (width, taps))
    want = {s: x + pt.causal_filter(x, w) for s, x in h.items()}
    n_slots = 6
    state = torch.zeros(n_slots, taps - 1, width, device=DEV)
    state[1] = 7.0      # another request's slot: must stay as it is
    parts = {5: cuts(23, (1, 4, 2, 1, 1, 9)), 2: cuts(17, (3, 1, 1, 2, 8))}
    got = {5: [], 2: []}
    for step in range(max(len(p) for p in parts.values())):
        live = [(s, parts[s][step]) for s in (5, 2) if step < len(parts[s])]
        x = np.concatenate([h[s][a:b] for s, (a, b) in live])
        rows = rows_of([(s, b - a) for s, (a, b) in live], n_slots)
        out = torch.empty(x.shape[0], width, device=DEV)
        ops.short_conv(out, dev(x), dev(w), state, rows, exact=True)
        if taps > 1:
            ops.keep_last_rows(state, dev(x), rows)
        at = 0
        for s, (a, b) in live:
            got[s].append(out[at:at + b - a].cpu().numpy())
            at += b - a
    for s in (5, 2):
        assert np.abs(np.concatenate(got[s]) - want[s]).max() <= 1e-5
    if taps > 1:
        assert bool((state[1] == 7.0).all())


def test_mix_with_the_token_before():
    from alofa_amd import ops
    rng = np.random.default_rng(1)
    width = 24
    x, mu = rng.normal(0, 1, (11, width)).astype(np.float32), rng.uniform(0, 1, (5, width)).astype(np.float32)
    before = np.vstack([np.zeros((1, width)), x[:-1]])
    want = np.stack([x + (before - x) * m for m in mu])
    state = torch.zeros(3, 1, width, device=DEV)
    got = []
    for a, b in cuts(11, (1, 1, 4, 2, 1, 1, 1)):
        rows = rows_of([(2, b - a)], 3)
        out = torch.empty(5, b - a, width, device=DEV)
        if b - a == 1 and a % 2:      # a single row: the state may move on in the same launch
            ops.shift_mix(out, dev(x[a:b]), dev(mu), state, rows, keep=True)
        else:
            ops.shift_mix(out, dev(x[a:b]), dev(mu), state, rows)
            ops.keep_last_rows(state, dev(x[a:b]), rows)
        got.append(out.cpu().numpy())
    assert np.abs(np.concatenate(got, axis=1) - want).max() <= 1e-6


DECAYS = ["per_head", "sigmoid_root", "exp_neg_exp"]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("kind", DECAYS)
@pytest.mark.parametrize("heads,dk,dv", [(2, 16, 16), (1, 40, 72), (3, 24, 8), (2, 128, 128), (1, 130, 66), (1, 300, 20)])
def test_linear_recurrence(heads, dk, dv, kind, dtype):
    """Two requests side by side in unequal portions (single rows among them) against the plain recurrence of each."""
    from alofa_amd import ops
    rng = np.random.default_rng(dk + dv)
    n_slots, T = 4, {3: 141, 0: 29}      # (steps of more than 64 rows make their decays in a launch of their own)
    data = {}
    for s, n in T.items():
        q, k, v = rng.normal(0, 1, (n, heads * dk)), rng.normal(0, 1, (n, heads * dk)), rng.normal(0, 1, (n, heads * dv))
        if dtype is torch.bfloat16:
            q, k, v = (pt.to_bfloat16(a) for a in (q, k, v))
        data[s] = (q.astype(np.float32), k.astype(np.float32), v.astype(np.float32), rng.normal(0.5, 1.5, (n, heads * dk)).astype(np.float32))
    per_head = rng.uniform(0.8, 1.0, heads).astype(np.float32)
    bonus = rng.normal(0, 1, (heads, dk)).astype(np.float32) if kind == "exp_neg_exp" else None
    tau, qs, ks = 7.0, 0.37, 1.9

    def weights(z):
        if kind == "per_head":
            return np.repeat(per_head.astype(np.float64), dk)[None, :].repeat(z.shape[0], 0)
        z = z.astype(np.float64)
        return (1 / (1 + np.exp(-z))) ** (1 / tau) if kind == "sigmoid_root" else np.exp(-np.exp(z - 2.0))
    want = {}
    for s, (q, k, v, z) in data.items():
        w = weights(z)
        want[s] = np.concatenate([pt.decayed_outer_sum(q[:, i * dk:(i + 1) * dk].astype(np.float64) * np.float32(qs), k[:, i * dk:(i + 1) * dk].astype(np.float64) * np.float32(ks),
                                                       v[:, i * dv:(i + 1) * dv].astype(np.float64), w[:, i * dk:(i + 1) * dk], None if bonus is None else bonus[i].astype(np.float64))
                                  for i in range(heads)], axis=1)
    state = torch.zeros(n_slots, heads, dk, dv, device=DEV)
    state[1] = 3.0
    parts = {3: cuts(141, (1, 17, 1, 2, 100, 5, 15)), 0: cuts(29, (6, 1, 1, 16, 2, 9))}
    got = {3: [], 0: []}
    code = {"per_head": ops.DECAY_PER_HEAD, "sigmoid_root": ops.DECAY_SIGMOID_ROOT, "exp_neg_exp": ops.DECAY_EXP_NEG_EXP}[kind]
    for step in range(max(len(p) for p in parts.values())):
        live = [(s, parts[s][step]) for s in (3, 0) if step < len(parts[s])]
        q, k, v, z = (np.concatenate([data[s][j][a:b] for s, (a, b) in live]) for j in range(4))
        rows = rows_of([(s, b - a) for s, (a, b) in live], n_slots)
        # (room for the read-outs in parts: the step of 100 rows deals the key channels out over blocks where the key size allows)
        room = torch.full((ops.recurrence_max_parts(dk), q.shape[0], heads * dv), float("nan"), device=DEV)
        decay = dev(per_head) if kind == "per_head" else dev(z - 2.0 if kind == "exp_neg_exp" else z)
        used = ops.linear_recurrence(room, dev(q, dtype), dev(k, dtype), dev(v, dtype), state, rows, heads, dk, dv, code, decay, tau=tau,
                                     bonus=None if bonus is None else dev(bonus), q_scale=qs, k_scale=ks, before_update=bonus is not None)
        assert 1 <= used <= room.shape[0] and (used > 1) == (q.shape[0] > 64 and dk >= 32)
        out = room[:used].sum(0)
        at = 0
        for s, (a, b) in live:
            got[s].append(out[at:at + b - a].cpu().numpy())
            at += b - a
    for s in (3, 0):
        g = np.concatenate(got[s])
        assert np.abs(g - want[s]).max() <= 2e-5 * max(1.0, np.abs(want[s]).max()), f"slot {s}"
    assert bool((state[1] == 3.0).all()) and bool((state[2] == 0.0).all())


@pytest.mark.parametrize("weighted", [False, True])
@pytest.mark.parametrize("heads,dv", [(3, 8), (2, 72), (1, 200)])
def test_head_norm_and_gate(heads, dv, weighted):
    from alofa_amd import ops
    rng = np.random.default_rng(heads)
    T = 7
    o, g = rng.normal(0, 2, (T, heads, dv)).astype(np.float32), rng.normal(0, 2, (T, heads * dv)).astype(np.float32)
    w = rng.normal(1, 0.3, heads * dv).astype(np.float32) if weighted else None
    want = pt.unit_rms(o.astype(np.float64), 1e-6).reshape(T, -1) * (1.0 if w is None else w) * pt.silu(g.astype(np.float64))
    wide = torch.zeros(T, heads * dv + 8, device=DEV)      # the gate as columns of a wider matrix
    wide[:, 8:] = dev(g)
    out = torch.empty(T, heads * dv, device=DEV)
    ops.headnorm_gate(out, dev(o.reshape(T, -1)), wide[:, 8:], None if w is None else dev(w), heads, dv, 1e-6, True)
    assert np.abs(out.cpu().numpy() - want).max() <= 1e-5 * max(1.0, np.abs(want).max())
    # the same read-outs in three parts, with room for four
    shares = rng.normal(0, 1, (4, T, heads * dv)).astype(np.float32)
    shares[2] = o.reshape(T, -1) - shares[0] - shares[1]
    ops.headnorm_gate(out, dev(shares), wide[:, 8:], None if w is None else dev(w), heads, dv, 1e-6, True, parts=3)
    assert np.abs(out.cpu().numpy() - want).max() <= 2e-5 * max(1.0, np.abs(want).max())


def test_activations():
    from alofa_amd import ops
    z = np.linspace(-9, 9, 1001).astype(np.float32).reshape(7, 143)
    out = torch.empty(7, 143, device=DEV)
    ops.activation(out, dev(z), ops.XIELU, pt.softplus(0.3), 0.5 + pt.softplus(-1.2), exact=True)
    assert np.abs(out.cpu().numpy() - pt.xielu(z.astype(np.float64), 0.3, -1.2)).max() <= 1e-5
    ops.activation(out, dev(z), ops.TANH, exact=True)
    assert np.abs(out.cpu().numpy() - np.tanh(z.astype(np.float64))).max() <= 1e-6
    half = dev(z, torch.bfloat16)
    ops.activation(half, half, ops.XIELU, pt.softplus(0.3), 0.5 + pt.softplus(-1.2))
    want = pt.xielu(pt.to_bfloat16(z), 0.3, -1.2)
    assert np.abs(half.float().cpu().numpy() - want).max() <= 2 ** -8 * np.abs(want).max()


def test_average_over_depth_and_sum_of_branches():
    from alofa_amd import ops
    rng = np.random.default_rng(3)
    levels, shape = 4, (5, 12)
    outs = [rng.normal(0, 1, shape).astype(np.float32) for _ in range(levels)]
    weights = [rng.normal(0.4, 0.3, n + 1).astype(np.float32) for n in range(levels)]
    stack = torch.zeros(levels, *shape, device=DEV)
    x = dev(outs[0])
    ops.depth_average(x, stack, None, 1)
    assert torch.equal(x, dev(outs[0])) and torch.equal(stack[0], x)
    for n in range(1, levels):
        x = dev(outs[n])
        ops.depth_average(x, stack, dev(weights[n]), n + 1, exact=True)
        want = sum(weights[n][j].astype(np.float64) * outs[j] for j in range(n + 1))
        assert np.abs(x.cpu().numpy() - want).max() <= 1e-6
    r, a, b = (rng.normal(0, 1, shape).astype(np.float32) for _ in range(3))
    res = dev(r)
    ops.add_scaled(res, dev(a), 1.25, dev(b), -0.5, exact=True)
    assert np.abs(res.cpu().numpy() - (r + 1.25 * a.astype(np.float64) - 0.5 * b)).max() <= 1e-6
    ops.scale_(res, 3.0)
    assert np.abs(res.cpu().numpy() - 3.0 * (r + 1.25 * a.astype(np.float64) - 0.5 * b)).max() <= 3e-6


def test_part_of_a_head_rotated():
    """Rotary positions on the first channels of a head only: the position part's table and channel order against the
    plain rotation, through the products q . k, which are what the order of channels must not change."""
    from alofa_amd import ops
    from alofa_amd.config.base import PartSpec
    from alofa_amd.parts.base import Runtime, build_part
    rng = np.random.default_rng(5)
    T, heads, d, dims, base = 19, 3, 40, 12, 10000.0
    q, k = rng.normal(0, 1, (T, heads, d)).astype(np.float32), rng.normal(0, 1, (T, heads, d)).astype(np.float32)
    want = np.einsum("thd,shd->hts", pt.rotate(q.astype(np.float64), dims, base), pt.rotate(k.astype(np.float64), dims, base))
    part = build_part("position", PartSpec("rotary", {"theta": base, "head_dim": d, "dims": dims}), {}, Runtime(torch.device(DEV), torch.float32))
    order = part.channel_order()
    assert sorted(order) == list(range(d))
    both = dev(np.concatenate([q[:, :, order].reshape(T, -1), k[:, :, order].reshape(T, -1)], axis=1))
    cos, sin = part.table(T)
    ops.rope_kv_write(both, cos, sin, torch.arange(T, dtype=torch.int32, device=DEV), 2 * heads, 0, d)
    got = both.cpu().numpy().astype(np.float64).reshape(T, 2, heads, d)
    assert np.abs(np.einsum("thd,shd->hts", got[:, 0], got[:, 1]) - want).max() <= 1e-4


@pytest.mark.parametrize("taps", [2, 4, 16])
@pytest.mark.parametrize("exact", [True, False])
def test_norm_filter_and_state_in_one_launch(taps, exact):
    """Single rows of three requests: the fused kernel against norm, filter and state update one after the other."""
    from alofa_amd import ops
    rng = np.random.default_rng(taps)
    width, n_slots = 200, 5
    w, nw, nb = dev(rng.normal(0, 0.5, (width, taps))), dev(rng.normal(1, 0.2, width)), dev(rng.normal(0, 0.3, width))
    fused, apart = torch.zeros(n_slots, taps - 1, width, device=DEV), torch.zeros(n_slots, taps - 1, width, device=DEV)
    rows = rows_of([(4, 1), (0, 1), (2, 1)], n_slots)
    for _ in range(6):
        x = dev(rng.normal(1.0, 2.0, (3, width)))
        normed, want, got = torch.empty(3, width, device=DEV), torch.empty(3, width, device=DEV), torch.empty(3, width, device=DEV)
        ops.layernorm(normed, x, nw, nb, 1e-5, exact)
        ops.short_conv(want, normed, w, apart, rows, exact)
        ops.keep_last_rows(apart, normed, rows)
        ops.norm_conv_step(got, x, nw, nb, 1e-5, w, fused, rows, exact)
        assert torch.equal(got, want) and torch.equal(fused, apart)


@pytest.mark.parametrize("shapes", [[(3, 4)], [(16, 64, 64), (3, 5), (1,), (1029,)], [(4097,), (7, 4096), (33, 257)]])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_the_slot_of_a_new_request_is_cleared_in_every_tensor_and_no_other(shapes, dtype):
    from alofa_amd import ops
    from alofa_amd.errors import AlofaError
    tensors = [torch.randn((3, *s), device="cuda").to(dtype) for s in shapes]
    want = [t.clone() for t in tensors]
    slots = ops.StateSlots(tensors)
    for slot in (1, 2, 0):
        slots.clear(slot)
        for w, t in zip(want, tensors):
            w[slot].zero_()
            assert torch.equal(w, t)
    with pytest.raises(AlofaError):
        slots.clear(3)


def test_a_slot_is_cleared_on_the_callers_stream():
    """Within a scope of another stream, as where another part of the program is in the middle of a step."""
    from alofa_amd import ops
    t = torch.ones((3, 1000), device="cuda")
    slots = ops.StateSlots([t])
    busy, mine = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(busy):
        scope = ops.stream_scope()
        scope.__enter__()
        torch.cuda._sleep(200_000_000)      # (a kernel that counts clock cycles, some 0.1 s, and ends)
    try:
        with torch.cuda.stream(mine):
            slots.clear(1)
            got = t.cpu()
            assert not busy.query()
    finally:
        scope.__exit__(None, None, None)
    busy.synchronize()
    assert bool((got[1] == 0).all()) and bool((got[[0, 2]] == 1).all())


STEP_HEADS = [(1, 1, 4), (3, 63, 20), (16, 64, 64), (5, 96, 40), (2, 128, 256), (3, 256, 252), (2, 256, 256)]


@pytest.mark.parametrize("turned,heads,dk,dv", [(turned, *sizes) for turned in (False, True) for sizes in STEP_HEADS if not turned or sizes[1] % 2 == 0])      # (a rotation takes pairs of channels)
@pytest.mark.parametrize("kind", ["per head", "sigmoid root", "exp of exp, bonus"])
def test_single_row_step_in_one_launch(heads, dk, dv, kind, turned):
    """Rotation, recurrence, head norm and gate in one launch beside the launches it replaces and beside float64; slots in any order, others left alone."""
    from alofa_amd import ops
    rng = np.random.default_rng(heads * dk + dv)
    T, n_slots, used = 5, 9, (7, 0, 3, 8, 4)
    rows = rows_of([(s, 1) for s in used], n_slots)
    proj = dev(rng.normal(0, 1, (T, heads * (2 * dk + 2 * dv) + 8)), torch.bfloat16)
    kd, vd = heads * dk, heads * dv
    q, k, v, gate = proj[:, :kd], proj[:, kd:2 * kd], proj[:, 2 * kd:2 * kd + vd], proj[:, 2 * kd + vd:2 * kd + 2 * vd]
    state = dev(rng.normal(0, 1, (n_slots, heads, dk, dv)))
    weight = None if kind == "per head" else dev(rng.normal(1, 0.2, vd))
    bonus = dev(rng.normal(0, 1, (heads, dk))) if kind.startswith("exp") else None
    code = {"per head": ops.DECAY_PER_HEAD, "sigmoid root": ops.DECAY_SIGMOID_ROOT}.get(kind, ops.DECAY_EXP_NEG_EXP)
    decay = dev(rng.uniform(0.5, 0.99, heads)) if code == ops.DECAY_PER_HEAD else dev(rng.normal(0, 1, (T, kd)))
    how = dict(tau=4.0, bonus=bonus, q_scale=0.5, k_scale=0.25, before_update=bonus is not None)
    cos, sin = (dev(rng.uniform(-1, 1, (11, max(dk // 2, 1)))) for _ in range(2))
    positions = torch.tensor([10, 0, 3, 5, 5], dtype=torch.int32, device=DEV)
    out, got_state, kept = torch.empty(T, vd, device=DEV, dtype=torch.bfloat16), state.clone(), proj.clone()
    ops.recurrence_step(out, q, k, v, gate, weight, got_state, rows, heads, dk, dv, 1e-5, code, decay, rope=(cos, sin, positions) if turned else None, **how)
    assert torch.equal(proj, kept)

    # launch by launch
    if turned:
        ops.rope_kv_write(proj, cos, sin, positions, 2 * heads, 0, dk)
    o, old_state, old = torch.empty(T, vd, device=DEV), state.clone(), torch.empty_like(out)
    ops.linear_recurrence(o, q, k, v, old_state, rows, heads, dk, dv, code, decay.clone(), **how)
    ops.headnorm_gate(old, o, gate, weight, heads, dv, 1e-5, False)
    # (a number of the state is one product and one sum in either, two roundings of at most 2^-24 of terms below 8)
    assert torch.allclose(got_state, old_state, rtol=1e-6, atol=1e-6)

    # in float64
    S = state.double()[rows.slots.long()]
    qd, kh, vh = (t.double().unflatten(1, (heads, -1)) for t in (q, k, v))
    qd, kh = qd * 0.5, kh * 0.25
    if code == ops.DECAY_PER_HEAD:
        w = decay.double()[None, :, None].expand(T, heads, dk)
    else:
        w = (torch.sigmoid(decay.double()) ** 0.25 if code == ops.DECAY_SIGMOID_ROOT else torch.exp(-torch.exp(decay.double()))).unflatten(1, (heads, -1))
    kv = kh[..., None] * vh[:, :, None]
    new = w[..., None] * S + kv
    read = ((S + bonus.double()[None, :, :, None] * kv if bonus is not None else new) * qd[..., None]).sum(2)
    y = (read / torch.sqrt((read * read).mean(2, keepdim=True) + 1e-5)).flatten(1) * (1 if weight is None else weight.double()) * torch.nn.functional.silu(gate.double())
    assert ((got_state[rows.slots.long()].double() - new).norm() / new.norm()).item() < 1e-6
    untouched = [s for s in range(n_slots) if s not in used]
    assert torch.equal(got_state[untouched], state[untouched])
    # a result is rounded once, to bfloat16: by at most 2^-9 of it; both ways are off by those roundings, and where a sum falls close to the middle of two of them they differ
    off = {n: ((x.double() - y).norm() / y.norm()).item() for n, x in (("one launch", out), ("launch by launch", old))}
    assert off["one launch"] < 2 ** -9 and off["one launch"] <= off["launch by launch"] * 1.01 + 1e-5, off


@pytest.mark.parametrize("width", [1, 255, 1025, 2048, 2049, 4100])
@pytest.mark.parametrize("taps", [2, 3, 4, 5])
def test_norm_filter_and_state_at_the_edges_of_its_forms(width, taps):
    """Widths around a block's channels and what a thread keeps of a row, the taps that have a form of their own and the next: norm, filter and state beside the launches for any rows."""
    from alofa_amd import ops
    rng = np.random.default_rng(width + taps)
    n_slots, rows = 6, rows_of([(4, 1), (0, 1), (5, 1)], 6)
    x, w, b, f = dev(rng.normal(1, 2, (3, width))), dev(rng.normal(1, 0.2, width)), dev(rng.normal(0, 0.5, width)), dev(rng.normal(0, 0.5, (width, taps)))
    state = dev(rng.normal(0, 1, (n_slots, taps - 1, width)))
    for dtype in (torch.float32, torch.bfloat16):
        one, got = state.clone(), torch.empty(3, width, device=DEV, dtype=dtype)
        ops.norm_conv_step(got, x, w, b, 1e-5, f, one, rows)
        apart, n, want = state.clone(), torch.empty(3, width, device=DEV), torch.empty(3, width, device=DEV)
        ops.layernorm(n, x, w, b, 1e-5, False)
        ops.short_conv(want, n, f, apart, rows)
        ops.keep_last_rows(apart, n, rows)
        # (a norm's sums of up to 4,100 numbers in another order: 1e-6 of numbers around 3; a rounding to bfloat16 is 2^-9 of a number)
        assert torch.allclose(one, apart, rtol=1e-5, atol=1e-5)
        assert torch.allclose(got.float(), want, rtol=2 ** -8 if dtype is torch.bfloat16 else 1e-5, atol=1e-4)


# what rides on the vector-unit product is the same bits as the launches one behind the other: K of one run, several, ragged and (depth) the long form; rows up to eight and, launch by launch, beyond; columns of no whole block
@pytest.mark.parametrize("M,N,K", [(1, 64, 512), (4, 4096, 1024), (5, 37, 520), (8, 130, 6144), (3, 64, 8192), (12, 96, 1024), (2, 8, 16)])
def test_products_with_what_follows_them(M, N, K):
    from alofa_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(M + N)
    draw = lambda *s: torch.randn(s, generator=gen, device=DEV)      # noqa: E731
    a, w, bias = draw(M, K).bfloat16(), (draw(N, K) * K ** -0.5).bfloat16(), draw(N)
    for b in (None, bias):
        for kind in ops.ACTIVATIONS:
            want, got = torch.empty(M, N, device=DEV, dtype=torch.bfloat16), torch.empty(M, N + 5, device=DEV, dtype=torch.bfloat16).fill_(7.0)
            ops.gemm(want, a, w, b)
            ops.activation(want, want, kind, 0.7, 1.1)
            ops.gemm(got[:, :N], a, w, b, act=(kind, 0.7, 1.1))
            assert torch.equal(got[:, :N], want) and bool((got[:, N:] == 7.0).all()), kind
    for n in (1, 2, 8, 9, 13):
        levels, weights, x = draw(14, M, N), draw(n), draw(M, N)
        stacks, xs = [levels.clone(), levels.clone()], [x.clone(), x.clone()]
        ops.gemm(xs[0], a, w, add_to_out=True)
        ops.depth_average(xs[0], stacks[0], weights, n)
        ops.gemm(xs[1], a, w, add_to_out=True, depth=(stacks[1], weights, n))
        assert torch.equal(xs[0], xs[1]) and torch.equal(*stacks), n


@pytest.mark.parametrize("M,K,columns", [(1, 512, (64, 64)), (4, 1024, (1024, 1024, 1024, 1024, 64)), (8, 520, (5, 130, 4)), (3, 4096, (33, 7, 64, 1)), (9, 256, (64, 32))])
def test_products_side_by_side(M, K, columns):
    from alofa_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(K)
    products, want = [], []
    wide = torch.zeros(M, sum(columns) + 8, device=DEV, dtype=torch.bfloat16)      # (results beside one another in one buffer)
    at = 0
    for i, n in enumerate(columns):
        a, w = torch.randn(M, K, generator=gen, device=DEV).bfloat16(), (torch.randn(n, K, generator=gen, device=DEV) * K ** -0.5).bfloat16()
        kind = (None, ops.TANH, ops.SILU, None, ops.GELU_TANH)[i]
        products.append((wide[:, at:at + n], a, w, kind))
        alone = torch.empty(M, n, device=DEV, dtype=torch.bfloat16)
        ops.gemm(alone, a, w)
        if kind is not None:
            ops.activation(alone, alone, kind)
        want.append(alone)
        at += n
    ops.gemm_side_by_side(products)
    assert torch.equal(wide[:, :at], torch.cat(want, 1)) and not bool(wide[:, at:].any())


@pytest.mark.parametrize("n", [1, 2, 5, 16])
@pytest.mark.parametrize("rank", [8, 16, 40, 64])
@pytest.mark.parametrize("heads,dk,dv,kind", [(3, 64, 64, "sigmoid_root"), (2, 40, 72, "exp_neg_exp"), (1, 256, 8, "exp_neg_exp")])
def test_single_row_step_that_makes_its_decays(heads, dk, dv, kind, rank, n):
    from alofa_amd import ops
    gen = torch.Generator(device=DEV).manual_seed(rank + dk)
    draw = lambda *s: torch.randn(s, generator=gen, device=DEV)      # noqa: E731
    wide = draw(n, 2 * heads * dk + 2 * heads * dv + rank).bfloat16()
    q, k, v, gate, low = wide.split([heads * dk, heads * dk, heads * dv, heads * dv, rank], 1)
    w, bias = (draw(heads * dk, rank) * rank ** -0.5).bfloat16(), draw(heads * dk)
    assert ops.recurrence_step_makes_decays(low, w, bias, n, heads * dk) and not ops.recurrence_step_makes_decays(low, w, bias, 17, heads * dk)
    z = torch.empty(n, heads * dk, device=DEV)
    ops.gemm(z, low, w, bias)      # (the launch that is saved)
    before = kind == "exp_neg_exp"
    code, rows = (ops.DECAY_EXP_NEG_EXP if before else ops.DECAY_SIGMOID_ROOT), rows_of([(s, 1) for s in range(n, 0, -1)], n + 1)
    bonus, first = draw(heads, dk) if before else None, draw(n + 1, heads, dk, dv)
    got = []
    for decay in (z, (low, w, bias)):
        state, out = first.clone(), torch.empty(n, heads * dv, device=DEV, dtype=torch.bfloat16)
        ops.recurrence_step(out, q, k, v, gate, None, state, rows, heads, dk, dv, 1e-6, code, decay, tau=5.0, bonus=bonus, before_update=before)
        got.append((out.float(), state))
    assert torch.equal(got[0][1], got[1][1]) and torch.equal(got[0][0], got[1][0]) and torch.equal(got[1][1][0], first[0])


# portions of one row, of fewer rows than the state keeps, of a block's rows and one more, and long ones; the widths at the edges of either form; the bits of three launches
@pytest.mark.parametrize("width", [4, 64, 260, 1020, 1024, 1028, 2044, 2048])
@pytest.mark.parametrize("taps", [2, 3, 4])
def test_norm_filter_and_state_of_portions_in_one_launch(width, taps):
    from alofa_amd import ops
    rng = np.random.default_rng(width + taps)
    lengths, slots = (1, 2, 3, 8, 9, 35, 16), (6, 0, 3, 7, 1, 2, 5)
    T = sum(lengths)
    x, nw, nb, w = dev(rng.normal(1.0, 2.0, (T, width))), dev(rng.normal(1, 0.2, width)), dev(rng.normal(0, 0.5, width)), dev(rng.normal(0, 0.5, (width, taps)))
    state = dev(rng.normal(0, 1, (8, taps - 1, width)))
    rows = rows_of(list(zip(slots, lengths)), 8)
    assert ops.norm_conv_rows_takes(x, nw, nb, w)
    assert not ops.norm_conv_rows_takes(torch.empty(3, 2052, device=DEV), torch.empty(2052, device=DEV), torch.empty(2052, device=DEV), torch.empty(2052, taps, device=DEV))      # (three launches are faster)
    # launch by launch, and in float64
    wide, old, old_state = torch.empty_like(x), torch.empty_like(x), state.clone()
    ops.layernorm(wide, x, nw, nb, 1e-5, False)
    ops.short_conv(old, wide, w, old_state, rows)
    ops.keep_last_rows(old_state, wide, rows)
    xd = x.double()
    dev2 = xd - xd.mean(1, keepdim=True)
    n = dev2 / torch.sqrt((dev2 * dev2).mean(1, keepdim=True) + 1e-5) * nw.double() + nb.double()
    want, want_state, at = torch.empty_like(n), state.double(), 0
    for s, m in zip(slots, lengths):
        both = torch.cat([want_state[s], n[at:at + m]])
        want[at:at + m] = both[taps - 1:] + sum(both[j:j + m] * w.double()[:, j] for j in range(taps))
        want_state[s] = both[m:]
        at += m
    for dtype in (torch.float32, torch.bfloat16):
        out, got_state = torch.empty(T, width, device=DEV, dtype=dtype), state.clone()
        ops.norm_conv_rows(out, x, nw, nb, 1e-5, w, got_state, rows, max(lengths))
        assert torch.equal(out, old.to(dtype)) and torch.equal(got_state, old_state)
        assert (out.double() - want).norm() / want.norm() < (2 ** -8 if dtype is torch.bfloat16 else 1e-6)
        assert (got_state.double() - want_state).abs().max() <= 1e-5 * want_state.abs().max()
        assert torch.equal(got_state[4], state[4])
