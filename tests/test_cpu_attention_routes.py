"""Which kernel the attention stages lower to, and what the emitted source says (no GPU)."""
import re

import pytest

from sanic_amd import ir
from tests import attn_forms as A


def _functions(src):
    """name -> body of the kernel's functions"""
    out = {}
    for m in re.finditer(r"(?:void|bool|float)[^(;{}]* (\w+)\([^{};]*Args&? a[^{;]*\{", src):
        out[m.group(1)] = src[m.end():src.find("\n}", m.end())]
    return out


@pytest.mark.parametrize("terms", [A.prefix, A.chunk, A.bias, lambda p, s: A.bias(p, s) + A.prefix(p, s)])
@pytest.mark.parametrize("NH,NKV,NQ,T,dt", [
    (4, 2, 128, 128, ir.BF16),      # whole tiles
    (4, 2, 100, 300, ir.BF16),      # any length
    (0, 0, 40, 1000, ir.BF16),      # no head dim
    (0, 0, 200, 200, ir.F32),
    (4, 2, 200, 200, ir.F32),
])
def test_every_function_of_an_attention_kernel_names_the_same_buffers(NH, NKV, NQ, T, dt, terms):
    """A mask or an epilogue that reads a buffer: the score, window and store functions and the
    kernel pass one argument struct, so the store goes to the output (the one float16 buffer)
    and to nothing else."""
    p = A.attention(NH, NKV, NQ, T, terms, dt=dt, out=ir.F16, epilogue=A.residual)
    kind, src = p.emit(0)
    assert kind.startswith("skeleton:flash_prefill" if dt == ir.BF16 else "skeleton:attn_f32"), kind
    types = re.findall(r"(\S+)\* __restrict__ (b\d+);", src)
    out = [b for t, b in types if t == "_Float16"]
    assert len(out) == 1 and len(types) == len(p.buffers)
    fns = _functions(src)
    assert "finish" in fns and "window" in fns
    for name, body in fns.items():
        stores = set(re.findall(r"a\.(b\d+)\[[^;=]*\] = ", body))
        assert stores == (set(out) if name == "finish" else set()), (name, stores)
    # the mask's and the bias's float buffers are read by the score function as float
    floats = {b for t, b in types if t == "float"}
    score = fns["score_part"] if "score_part" in fns else fns["score"]
    assert set(re.findall(r"a\.(b\d+)", score)) <= floats


@pytest.mark.parametrize("name", A.EDGES)
@pytest.mark.parametrize("NH,NKV,NQ,T,dt", [(8, 2, 512, 512, ir.BF16), (4, 2, 100, 300, ir.BF16), (0, 0, 200, 200, ir.F32)])
def test_windows_that_move_one_way_take_the_attention_kernels(NH, NKV, NQ, T, dt, name):
    kind = A.attention(NH, NKV, NQ, T, A.EDGES[name], dt=dt).emit(0)[0]
    assert kind.startswith("skeleton:flash_prefill" if dt == ir.BF16 else "skeleton:attn_f32"), kind


@pytest.mark.parametrize("name", A.UNORDERED)
@pytest.mark.parametrize("NH,NKV,NQ,T,dt", [(8, 2, 512, 512, ir.BF16), (4, 2, 100, 300, ir.BF16), (0, 0, 200, 200, ir.F32)])
def test_windows_not_bounded_by_their_end_rows_take_the_fold(NH, NKV, NQ, T, dt, name):
    assert A.attention(NH, NKV, NQ, T, A.UNORDERED[name], dt=dt).emit(0)[0].startswith("fold:")


def test_heads_that_share_no_window_do_not_take_the_decode_kernel():
    """The decode kernel cuts a group's keys by its first head's window."""
    assert A.heads(8, 2, 1000, A.edge_per_head).emit(0)[0].startswith("fold:")
    assert A.heads(4, 4, 1000, A.edge_per_head).emit(0)[0].startswith("skeleton:attn_decode[rep 1]")


def test_the_decode_kernel_compiles_for_row_major_values():
    """... which the ILP machine scheduler of the compiler does not survive (8 heads over 300 keys)."""
    p = A.heads(8, 1, 300, A.prefix)
    assert p.emit(0)[0].startswith("skeleton:attn_decode[rep 8]")
    p.precompile()


@pytest.mark.parametrize("rows", [2, 4, 8])
@pytest.mark.parametrize("T", [256, 4096, 16384])
def test_a_few_query_rows_without_heads_take_the_decode_kernel(rows, T):
    assert A.attention(0, 0, rows, T, A.prefix).emit(0)[0].startswith(f"skeleton:attn_decode[rep {rows}]")


def test_query_rows_that_share_no_window_do_not_take_the_decode_kernel():
    """The decode kernel cuts a group's keys by its first row's window."""
    for form in (A.chunk, A.causal):
        assert A.attention(0, 0, 8, 4096, form).emit(0)[0].startswith("skeleton:attn_f32")
        assert A.attention(0, 0, 8, 300, form).emit(0)[0].startswith("skeleton:flash_prefill")


@pytest.mark.parametrize("NH,NKV,NQ,T,kind", [
    (0, 0, 4, 65536, "attn_f32"), (0, 0, 17, 1024, "attn_f32"), (2, 2, 2, 32768, "attn_f32"), (32, 8, 32, 4096, "attn_f32"),
    (0, 0, 17, 1000, "flash_prefill"), (32, 8, 33, 4096, "flash_prefill"), (0, 0, 300, 1024, "flash_prefill"), (2, 2, 2, 1024, "flash_prefill"),
])
def test_a_few_rows_over_a_long_cache_take_the_kernel_that_splits_the_keys(NH, NKV, NQ, T, kind):
    assert A.attention(NH, NKV, NQ, T, A.prefix).emit(0)[0].startswith("skeleton:" + kind)
