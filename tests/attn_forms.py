"""Attention programs of many forms for the lowering and GPU tests: softmax(q·kᵀ·HD^-½ + terms)·v."""
import math

from sanic_amd import carrier as C
from sanic_amd import ir
from sanic_amd.program import STREAM, Program


def mask(a, b, when, other):
    """where(a < b, when, other)"""
    return ir.map_(ir.WHERE, ir.map_(ir.LT, a, b), ir.const(when), ir.const(other))


def row(s):
    return ir.coordinate(s, s.rank - 2)


def key(s):
    return ir.coordinate(s, s.rank - 1)


def attention(NH, NKV, NQ, T, terms=lambda p, s: [], HD=64, dt=ir.BF16, out=ir.BF16, epilogue=None, vt=False):
    """NH query heads over NKV key/value heads (NH = 0: no head dim), NQ rows over T keys; `terms`
    gives the nodes added to the scores, `epilogue` the node stored, from (p, fold value); `vt`: V is
    stored [heads, HD, T]."""
    p = Program()
    lead, klead = ((NH,), (NKV,)) if NH else ((), ())
    q, k = p.input("Q", lead + (NQ, HD), dt), p.input("K", klead + (T, HD), dt)
    v = p.input("V", klead + ((HD, T) if vt else (T, HD)), dt)
    if vt:
        v = ir.transpose(v, -2, -1)
    if NH:
        k, v = ir.expand_heads(k, 0, NH // NKV), ir.expand_heads(v, 0, NH // NKV)
        s = ir.reduce(ir.map_(ir.MUL, ir.unsqueeze(q, 2), ir.unsqueeze(k, 1)), 3, ir.M_ADD)
    else:
        s = ir.matmul(q, ir.transpose(k, 0, 1))
    s = ir.map_(ir.MUL, s, ir.const(HD ** -0.5))
    for t in terms(p, s):
        s = ir.map_(ir.ADD, s, t)
    sb, vb = ((0, 1, STREAM), (0, STREAM, 2)) if NH else ((0, STREAM), (STREAM, 1))
    grid = lead + (NQ, HD)
    epi = epilogue(p, ir.fold_value(grid)) if epilogue else None
    p.fused("O", grid, T, [(s, sb), (v, vb)], C.online_softmax_weighted(), out, epilogue=epi)
    return p


def causal(p, s):
    return [mask(row(s), key(s), -1e30, 0.0)]


def prefix(p, s):
    """Keys up to `position` (a decode step's mask)."""
    pos = p.input("position", (), ir.F32)
    return [mask(ir.iota(s.shape[-1]), ir.map_(ir.ADD, pos, ir.const(1.0)), 0.0, -math.inf)]


def chunk(p, s):
    """Row i sees the keys up to position + i (a later chunk of a prompt)."""
    pos = p.input("position", (), ir.F32)
    return [mask(ir.map_(ir.ADD, row(s), pos), key(s), -1e30, 0.0)]


def bias(p, s):
    """A stored value per key."""
    return [p.input("bias", (s.shape[-1],), ir.F32)]


def residual(p, fold):
    return ir.map_(ir.ADD, p.input("R", fold.shape, ir.BF16), fold)
