"""The binding: the calls of C entries, and the operand checks in front of them against the same rules written out here."""
import ctypes
import re
import shutil
import subprocess

import pytest
import torch

from alofa_amd import ops
from alofa_amd.csrc import build, calls
from alofa_amd.csrc.build import load_binding
from alofa_amd.errors import AlofaError

SOURCE = """
#include <stdint.h>
static int64_t seen[64];
int64_t* places(void) { return seen; }
int mixed(int a, float x, int64_t b, void* p, int c, int d, int e, int64_t f, float y, int g, int h, float z) {
  return a == 1 && x == 0.5f && b == -2 && !p && c == 3 && d == -4 && e == 5 && f == (INT64_C(1) << 40) && y == 1.5f && g == -7 && h == 8 && z == -2.5f;
}
int nothing(void) { return -3; }
int floats(float a, float b, float c, float d, float e, float f, float g, float h, int last) {
  return a == 1 && b == 2 && c == 3 && d == 4 && e == 5 && f == 6 && g == 7 && h == 8 && last == -9;
}
int memory(const float* t, int n) { float s = 0; for (int i = 0; i < n; ++i) s += t[i]; return (int)s; }
"""


@pytest.fixture(scope="module")
def entries(tmp_path_factory):
    cc = shutil.which("gcc") or shutil.which("cc") or shutil.which("clang")
    if cc is None:
        pytest.skip("no C compiler")
    d = tmp_path_factory.mktemp("entries")
    (d / "entries.c").write_text(SOURCE + "int many(" + ", ".join(f"int64_t a{i}" for i in range(48)) + ") { int64_t s = 0;" + " ".join(f"s += (a{i} == {i} - 20);" for i in range(48)) + " return (int)s; }\n")
    subprocess.run([cc, "-O2", "-shared", "-fPIC", "-o", str(d / "entries.so"), str(d / "entries.c")], check=True)
    lib = ctypes.CDLL(str(d / "entries.so"))
    return lambda name: ctypes.cast(getattr(lib, name), ctypes.c_void_p).value


def test_every_parameter_arrives(entries):
    call = load_binding().call
    assert call(entries("mixed"), 1, 0.5, -2, None, 3, -4, 5, 1 << 40, 1.5, -7, 8, -2.5) == 1
    assert call(entries("nothing")) == -3
    assert call(entries("floats"), 1.0, 2.0, 3.0, 4.0, 5.0, 6.0, 7.0, 8.0, -9) == 1
    assert call(entries("many"), *range(-20, 28)) == 48
    assert call(entries("memory"), torch.arange(5, dtype=torch.float32), 5) == 10
    assert call(entries("mixed"), True, 0.5, -2, None, 3, -4, 5, 1 << 40, 1.5, -7, 8, -2.5) == 1


def test_what_cannot_be_passed_is_refused(entries):
    call = load_binding().call
    for args, error in (((), TypeError), ((0,), ValueError), ((entries("nothing"), "x"), TypeError), ((entries("nothing"), 1 << 70), OverflowError),
                        ((entries("nothing"), *range(49)), TypeError), ((entries("nothing"), *[0.5] * 9), TypeError)):
        with pytest.raises(error):
            call(*args)


def test_operands_that_are_not_on_the_gpu_are_left_to_the_checks_that_say_so():
    t = torch.zeros(4, 16, dtype=torch.bfloat16)
    assert load_binding().product(t, t, t, None, None) is None and load_binding().caches(t, t, 1, 16) is None
    assert load_binding().product(None, 3, "x", None, None) is None and load_binding().norm(t) is None
    with pytest.raises(AlofaError):
        ops.gemm(t, t, t)
    with pytest.raises(AlofaError):
        ops.rmsnorm(t, t.float(), torch.ones(16), 1e-6, False)


def _rows(t):
    return t.dim() == 2 and (t.stride(1) == 1 or t.shape[1] <= 1)


def _ld(t):
    return t.stride(0) if t.shape[0] > 1 else max(t.stride(0), t.shape[1])


@pytest.mark.gpu
def test_operands_of_products_are_told_apart_as_the_rules_say():
    dev = "cuda"
    pool = torch.zeros(1 << 16, dtype=torch.bfloat16, device=dev)

    def forms(rows, columns):
        yield pool[:rows * columns].view(rows, columns)
        yield pool[:rows * (columns + 8)].view(rows, columns + 8)[:, :columns]           # padded rows
        yield pool[:rows * (columns + 8)].view(rows, columns + 8)[:, 8:]                 # ... that start behind the padding
        yield pool[:rows * (columns + 4)].view(rows, columns + 4)[:, :columns]           # rows in steps of 4
        yield pool[1:1 + rows * columns].view(rows, columns)                             # bases between two 16-byte places
        yield pool[:rows * columns].view(columns, rows).t()                              # the other order
        yield pool[:columns].view(1, columns).expand(rows, columns)                      # one row, many times
        yield pool[:rows * columns].view(1, rows, columns)                               # another rank
        yield pool[:rows * columns].view(rows, columns).float()
        yield pool[:rows * columns].view(rows, columns).half()
        yield pool[:rows * columns].view(rows, columns).cpu()
    bias = torch.zeros(24, device=dev)
    taken = 0
    for M, N, K in ((1, 24, 32), (3, 24, 32), (3, 24, 20), (3, 1, 32), (0, 24, 32)):
        for out in list(forms(M, N))[:1] + [torch.zeros(M, N, device=dev), torch.zeros(M, N, device=dev).half(), torch.zeros(M, N + 1, device=dev)]:
            for a in forms(M, K):
                for w in forms(N, K):
                    for b in (None, bias[:N], bias.half()[:N], bias[:N - 1]):
                        got = ops._native().product(out, a, w, None, b)
                        ok = (all(t.is_cuda and _rows(t) for t in (out, a, w)) and a.dtype is w.dtype is torch.bfloat16 and out.dtype in (torch.float32, torch.bfloat16)
                              and tuple(out.shape) == (M, N) and tuple(a.shape) == (M, K) and tuple(w.shape) == (N, K) and K % 8 == 0
                              and _ld(a) % 8 == 0 and _ld(w) % 8 == 0 and a.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0
                              and (b is None or (b.dtype is torch.float32 and b.shape[0] == N)))
                        assert (got is not None) == ok, (M, N, K, out.shape, a.shape, a.stride(), w.stride())
                        if ok:
                            taken += 1
                            assert got == (M, N, K, _ld(out), _ld(a), _ld(w), ops.dtype_code(out))
    assert taken > 20
    gate, up = pool[:24 * 32].view(24, 32), pool[24 * 32:48 * 32].view(24, 32)
    a, out = pool[:3 * 32].view(3, 32), torch.zeros(3, 24, dtype=torch.bfloat16, device=dev)
    product = ops._native().product
    assert product(out, a, gate, up, None) and product(out.float(), a, gate, up, None) is None and product(out, a, gate, up[:23], None) is None
    assert product(out, a, gate, pool[:24 * 40].view(24, 40)[:, :32], None) is None      # gate and up in different steps


@pytest.mark.gpu
def test_operands_of_attention_norm_and_rotation_are_told_apart_as_the_rules_say():
    dev, n = "cuda", ops._native()
    k, v = torch.zeros(5, 2, 16, 64, dtype=torch.bfloat16, device=dev), torch.zeros(5, 2, 64, 16, dtype=torch.bfloat16, device=dev)
    assert n.caches(k, v, 2, 64) == 16
    for kk, vv, h, d in ((k, k, 2, 64), (k, v.float(), 2, 64), (k, v[:4], 2, 64), (k, v, 4, 64), (k, v, 2, 32), (k[:, :, :, ::2], v, 2, 32), (k, v.transpose(2, 3), 2, 64), (k.cpu(), v.cpu(), 2, 64)):
        assert n.caches(kk, vv, h, d) is None
        with pytest.raises(AlofaError):
            ops.check_caches(kk, vv, h, d)
    q, out, table = torch.zeros(3, 4 * 64, dtype=torch.bfloat16, device=dev), torch.zeros(3, 4 * 64, dtype=torch.bfloat16, device=dev), torch.zeros(3, 7, dtype=torch.int32, device=dev)
    assert n.attention(out, q, k, v, table, 4, 2, 64) == (3, 16) and n.attention(out.float(), q, k, v, table, 4, 2, 64) == (3, 16)
    bad = [(out[:2], q, table, 4), (out, q.float(), table, 4), (out.half(), q, table, 4), (out, q, table.long(), 4), (out, q, table[:, ::2], 4), (out, q, table, 3), (out, q, table, 8),
           (out, torch.zeros(3 * 256 + 1, dtype=torch.bfloat16, device=dev)[1:].view(3, 256), table, 4), (out, torch.zeros(3, 260, dtype=torch.bfloat16, device=dev)[:, :256], table, 4)]
    for o, qq, t, h in bad:
        assert n.attention(o, qq, k, v, t, h, 2, 64) is None
        with pytest.raises(AlofaError):
            ops._attention_operands(o, qq, k, v, t, h, 2, 64)
    small = torch.zeros(5, 2, 4, 64, dtype=torch.bfloat16, device=dev), torch.zeros(5, 2, 64, 4, dtype=torch.bfloat16, device=dev)
    assert n.attention(out, q, *small, table, 4, 2, 64) is None and n.attention(out, q, k.float(), v.float(), table, 4, 2, 64) is None
    x, w, rows = torch.zeros(3, 40, device=dev), torch.zeros(40, device=dev), torch.zeros(2, dtype=torch.int32, device=dev)
    assert n.norm(x.clone(), x, w, None) == (3, 40, ops.F32) and n.norm(x[:2].bfloat16(), x, w, rows) == (2, 40, ops.BF16)
    for args in ((x[:2], x, w, None), (x, x, w, rows), (x.half(), x, w, None), (x, x.bfloat16(), w, None), (x, x, w[:39], None), (x, x, w.bfloat16(), None), (x.t(), x.t(), w, None), (x, x, w, rows.long())):
        assert n.norm(*args) is None
        with pytest.raises(AlofaError):
            ops.rmsnorm(args[0], args[1], args[2], 1e-6, False, rows=args[3])
    qkv, cos, at, slots = torch.zeros(3, 8 * 64, dtype=torch.bfloat16, device=dev), torch.zeros(9, 32, device=dev), torch.zeros(3, dtype=torch.int32, device=dev), torch.zeros(3, dtype=torch.int64, device=dev)
    assert n.turn(qkv, cos, cos, at, slots, k, v, 4, 2, 64) == (3, 512, ops.BF16, 16)
    for args in ((qkv.float(), cos, cos, at, slots), (qkv[:, :448], cos, cos, at, slots), (qkv, cos[:, :31], cos, at, slots), (qkv, cos, cos[:8], at, slots), (qkv, cos, cos, at[:2], slots),
                 (qkv, cos, cos, at, slots.int()), (qkv, cos, cos, at, slots[:2]), (qkv, cos, cos, at.long(), slots), (qkv, cos, cos, at, None)):
        assert n.turn(*args, k, v, 4, 2, 64) is None
        with pytest.raises(AlofaError):
            ops.rope_kv_write(*args[:4], 4, 2, 64, args[4], k, v)


def test_without_the_binding_ctypes_passes_the_same(entries):
    assert calls.call(entries("mixed"), 1, 0.5, -2, None, 3, -4, 5, 1 << 40, 1.5, -7, 8, -2.5) == 1
    assert calls.call(entries("nothing")) == -3
    assert calls.call(entries("floats"), 1.0, 2.0, 3.0, 4.0, 5.0, 6.0, 7.0, 8.0, -9) == 1
    assert calls.call(entries("many"), *range(-20, 28)) == 48
    assert calls.call(entries("memory"), torch.arange(5, dtype=torch.float32), 5) == 10
    for args, error in (((0,), ValueError), ((entries("nothing"), "x"), TypeError), ((entries("nothing"), 1 << 70), OverflowError)):
        with pytest.raises(error):
            calls.call(*args)


def test_a_binding_that_cannot_be_built_is_done_without(monkeypatch, capsys):
    def refuse():
        raise AlofaError("not_initialized", "no C++ compiler was found; the binding cannot be built")
    monkeypatch.setattr(build, "_binding", None)
    monkeypatch.setattr(build, "find_built_binding", lambda: None)
    monkeypatch.setattr(build, "build_binding", refuse)
    monkeypatch.setattr(ops, "_binding", None)
    assert ops._native() is calls and "no C++ compiler" in capsys.readouterr().err
    t = torch.zeros(4, 16, dtype=torch.bfloat16)
    with pytest.raises(AlofaError) as e:      # the check that says a tensor is not on the GPU needs no binding
        ops.gemm(t, t, t)
    assert e.value.name == "invalid_argument" and "GPU tensor" in str(e.value)


def test_every_entry_can_be_called():
    """The one signature behind ``call``: at most 48 integers and pointers, at most eight floats, and no double (it would be passed as a float)."""
    seen = 0
    for source in build.sources():
        for name, parameters in re.findall(r'extern "C" [\w ]+?\b(alofa_\w+)\(([^)]*)\)', source.read_text()):
            kinds = [re.sub(r"\b\w+$", "", p.strip()) for p in parameters.split(",") if p.strip()]
            floats = [k for k in kinds if "*" not in k and "float" in k]
            assert not any("double" in k and "*" not in k for k in kinds), name
            assert len(floats) <= 8 and len(kinds) - len(floats) <= 48, name
            seen += 1
    assert seen > 50


@pytest.mark.gpu
def test_without_the_binding_the_results_are_the_same(monkeypatch):
    dev = "cuda"
    gen = torch.Generator(device=dev).manual_seed(1)

    def results():
        gen.manual_seed(1)
        rand = lambda *s: torch.randn(*s, generator=gen, device=dev)      # noqa: E731
        a, w, w2, x = rand(70, 256).bfloat16(), rand(192, 256).bfloat16(), rand(192, 256).bfloat16(), rand(70, 192)
        out, gated, normed = torch.empty(70, 192, device=dev), torch.empty(70, 192, device=dev, dtype=torch.bfloat16), torch.empty(70, 192, device=dev, dtype=torch.bfloat16)
        ops.gemm(out, a, w, rand(192))
        ops.gemm_swiglu(gated, a, w, w2)
        ops.gemm(x, a, w, add_to_out=True, then_norm=(rand(192), 1e-6, normed))
        exact = torch.empty(70, 192, device=dev)
        ops.gemm(exact, a.float(), w.float(), exact=True)
        kc, vc = rand(5, 1, 16, 64).bfloat16(), rand(5, 1, 64, 16).bfloat16()
        qkv, cos = rand(70, 6 * 64).bfloat16(), rand(80, 32)
        at, slots = torch.arange(70, dtype=torch.int32, device=dev), torch.arange(70, dtype=torch.int64, device=dev)
        ops.rope_kv_write(qkv, cos, cos, at, 4, 1, 64, slots, kc, vc)
        attn, table = torch.empty(70, 256, device=dev, dtype=torch.bfloat16), torch.arange(5, dtype=torch.int32, device=dev)[None]
        tiles = torch.tensor(ops.pair_tiles([(0, 0, 64, 0), (0, 64, 6, 64)]), dtype=torch.int32, device=dev)
        ops.attention_prefill(attn, qkv[:, :256], kc, vc, table, tiles, 4, 1, 64, None, 0.125)
        return [out, gated, x, normed, exact, qkv, kc, vc, attn]
    want = results()
    monkeypatch.setattr(ops, "_binding", calls)
    for got, expected in zip(results(), want):
        assert torch.equal(got, expected)
