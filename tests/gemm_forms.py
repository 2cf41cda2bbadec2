"""Projections y = x · W without a norm, for the lowering and GPU tests."""
from sanic_amd import carrier as C
from sanic_amd import ir
from sanic_amd.program import STREAM, Program


def projection(M, K, N, order, out=ir.BF16, residual=False):
    """`order`: how W is stored, "nk" or "kn"; " view" after it: read through a transpose of that.
    `residual`: y = R + x · W."""
    p = Program()
    x = p.input("x", (M, K), ir.BF16)
    nk = order.startswith("nk")
    w = p.input("W", (N, K) if nk else (K, N), ir.BF16)
    if order.endswith("view"):
        w, nk = ir.transpose(w, 0, 1), not nk
    p.fused("y", (M, N), K, [(x, (0, STREAM)), (w, (1, STREAM) if nk else (STREAM, 1))], C.dot(), out,
            epilogue=ir.map_(ir.ADD, p.input("R", (M, N), ir.BF16), ir.fold_value((M, N))) if residual else None)
    return p
