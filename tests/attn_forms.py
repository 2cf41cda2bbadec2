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


def attention(NH, NKV, NQ, T, terms=lambda p, s: [], HD=64, dt=ir.BF16, out=ir.BF16, epilogue=None, vt=False, qscale=False):
    """NH query heads over NKV key/value heads (NH = 0: no head dim), NQ rows over T keys; `terms`
    gives the nodes added to the scores, `epilogue` the node stored, from (p, fold value); `vt`: V is
    stored [heads, HD, T]; `qscale`: the query side is q times a stored value per dim."""
    p = Program()
    lead, klead = ((NH,), (NKV,)) if NH else ((), ())
    q, k = p.input("Q", lead + (NQ, HD), dt), p.input("K", klead + (T, HD), dt)
    v = p.input("V", klead + ((HD, T) if vt else (T, HD)), dt)
    if vt:
        v = ir.transpose(v, -2, -1)
    if qscale:
        q = ir.map_(ir.MUL, q, p.input("scale", (HD,), ir.F32))
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


def _half(s):
    return float(s.shape[-1] // 2)


# Window edges that move one way with the query row: mask terms by name.
EDGES = {
    "falling": lambda p, s: [mask(ir.map_(ir.SUB, ir.const(_half(s)), row(s)), key(s), -1e30, 0.0)],
    "falling product": lambda p, s: [mask(ir.map_(ir.ADD, ir.map_(ir.MUL, row(s), ir.const(-1.0)), ir.const(_half(s))), key(s), -1e30, 0.0)],
    "half": lambda p, s: [mask(ir.map_(ir.DIV, row(s), ir.const(2.0)), key(s), -1e30, 0.0)],
    "at most": lambda p, s: [mask(ir.map_(ir.MIN, row(s), ir.const(37.0)), key(s), -1e30, 0.0)],
    "at least": lambda p, s: [mask(ir.map_(ir.MAX, row(s), ir.const(37.0)), key(s), -1e30, 0.0)],
    "iota": lambda p, s: [mask(ir.unsqueeze(ir.iota(s.shape[-2]), 1), ir.iota(s.shape[-1]), -1e30, 0.0)],
    "window": lambda p, s: causal(p, s) + [mask(key(s), ir.map_(ir.MAX, ir.map_(ir.SUB, row(s), ir.const(40.0)), ir.const(0.0)), -1e30, 0.0)],
    "closing": lambda p, s: [mask(ir.map_(ir.SUB, ir.const(_half(s)), row(s)), key(s), -1e30, 0.0), mask(key(s), row(s), -1e30, 0.0)],
    "by a factor": lambda p, s: [mask(ir.map_(ir.MUL, row(s), p.input("position", (), ir.F32)), key(s), -1e30, 0.0)],
}


def _per_row(p, s):
    return ir.unsqueeze(p.input("bias", (s.shape[-2],), ir.F32), 1)


# Edges whose value at a row between two others these do not bound.
UNORDERED = {
    "stored per row": lambda p, s: [mask(_per_row(p, s), key(s), -1e30, 0.0)],
    "up and down": lambda p, s: [mask(ir.map_(ir.MIN, row(s), ir.map_(ir.SUB, ir.const(64.0), row(s))), key(s), -1e30, 0.0)],
    "two ways": lambda p, s: causal(p, s) + EDGES["falling"](p, s),
    # keys equal to a third of the row: no row between two multiples of 3 sees one
    "thirds": lambda p, s: [mask(ir.map_(ir.DIV, row(s), ir.const(3.0)), key(s), -1e30, 0.0),
                            mask(key(s), ir.map_(ir.DIV, row(s), ir.const(3.0)), -1e30, 0.0)],
}


def heads(NH, NKV, T, terms, HD=64):
    """One query row per head over NKV key/value heads, V as rows."""
    p = Program()
    q, k, v = p.input("Q", (NH, HD), ir.BF16), p.input("K", (NKV, T, HD), ir.BF16), p.input("V", (NKV, T, HD), ir.BF16)
    k, v = ir.expand_heads(k, 0, NH // NKV), ir.expand_heads(v, 0, NH // NKV)
    s = ir.map_(ir.MUL, ir.reduce(ir.map_(ir.MUL, ir.unsqueeze(q, 1), k), 2, ir.M_ADD), ir.const(HD ** -0.5))
    for t in terms(p, s):
        s = ir.map_(ir.ADD, s, t)
    p.fused("O", (NH, HD), T, [(s, (0, STREAM)), (v, (0, STREAM, 1))], C.online_softmax_weighted(), ir.F32)
    return p


def edge_per_head(p, s):
    """Each head with a last visible key of its own."""
    return [mask(ir.unsqueeze(p.input("edge", (s.shape[0],), ir.F32), 1), ir.iota(s.shape[1]), -1e30, 0.0)]
