"""MFMA GEMM skeleton (configs B2 and D2, plus small ragged shapes) against the oracle."""
import numpy as np
import pytest

import oracle
from sanic_amd import configs, ir
from sanic_amd.backend import from_bf16_bits
from tests.test_gpu_skeletons import bf16_rel, _bf16_vals
from tests import attn_forms as A
from tests import gemm_forms as forms
from tests.util import run_on_gpu

pytestmark = pytest.mark.gpu


def _report(exe, got, want):
    got = np.asarray(got, np.float64).reshape(want.shape)
    rel = np.abs(got - want) / np.maximum(np.abs(want), 1e-3)
    bad = np.argwhere(rel > 2e-2)
    print(exe.stage_kernel(0), float(rel.max()), "bad", len(bad), bad[:8].tolist(), flush=True)


@pytest.mark.parametrize("variant", [0, 1])
@pytest.mark.parametrize("M,K,N,kmajor", [
    (512, 2048, 8192, True),      # config B2, W [K, N]
    (512, 2048, 8192, False),     # same with the reference's [out, in] layout
    (64, 256, 96, True),
    (192, 128, 160, False),
    (64, 512, 512, True),         # x·g built by the first launch (K % 512 == 0)
    (128, 256, 16384, True),      # 8-wave 128 × 64 tiles, x·g built in-kernel (K % 512 != 0)
    (256, 384, 8192, False),      # 8-wave tiles, [out, in] weights, in-kernel row slots
    (128, 1536, 2048, True),      # operand-building launch with 3 k chunks over 4 waves
])
def test_rmsnorm_gemm(dev, M, K, N, kmajor, variant):
    prog = configs.rmsnorm_projection(M=M, K=K, N=N, kmajor=kmajor).with_variants({0: variant})
    x = _bf16_vals(301, M * K).reshape(M, K)
    g = _bf16_vals(302, K, 1.0, 0.02)
    wbits = oracle.synth_bf16(303, N * K, "normal", 0.0, 0.02)
    wkn = wbits.reshape(K, N) if kmajor else np.ascontiguousarray(wbits.reshape(N, K).T)
    w = from_bf16_bits(wbits).astype(np.float64).reshape((K, N) if kmajor else (N, K))
    got, exe = run_on_gpu(dev, prog, {"x": x, "g": g, "W": w})
    want = oracle.rmsnorm_proj(x, g, np.ascontiguousarray(wkn), 1e-5)
    err = bf16_rel(got["y"], want)
    _report(exe, got["y"], want)
    assert exe.stage_kernel(0).startswith("skeleton:gemm")
    assert err < 2e-2


@pytest.mark.parametrize("M,K,N,kmajor", [(512, 2048, 8192, True), (64, 512, 512, False), (128, 1536, 2048, True)])
def test_rmsnorm_gemm_fragment_order_a(dev, M, K, N, kmajor, monkeypatch):
    """The first launch's x·g planes in MFMA fragment order (each wave loading its A fragments
    directly, 8 × 1 waves) against the row-major planes staged through LDS
    (SANIC_HIP_GEMM_ALDS): both within the bf16 bound of the oracle, and within one output
    rounding of each other (the row slots are summed per K slice in the first form)."""
    x = _bf16_vals(311, M * K).reshape(M, K)
    g = _bf16_vals(312, K, 1.0, 0.02)
    wbits = oracle.synth_bf16(313, N * K, "normal", 0.0, 0.02)
    wkn = wbits.reshape(K, N) if kmajor else np.ascontiguousarray(wbits.reshape(N, K).T)
    w = from_bf16_bits(wbits).astype(np.float64).reshape((K, N) if kmajor else (N, K))
    want = oracle.rmsnorm_proj(x, g, np.ascontiguousarray(wkn), 1e-5)
    outs = {}
    for form in ("fragment", "lds"):
        if form == "lds":
            monkeypatch.setenv("SANIC_HIP_GEMM_ALDS", "1")
        prog = configs.rmsnorm_projection(M=M, K=K, N=N, kmajor=kmajor)
        got, exe = run_on_gpu(dev, prog, {"x": x, "g": g, "W": w})
        kind = exe.stage_kernel(0)
        assert kind.startswith("skeleton:gemm") and ",pre" in kind, kind
        assert (",ad" in kind) == (form == "fragment"), kind
        assert bf16_rel(got["y"], want) < 2e-2
        outs[form] = np.asarray(got["y"], np.float64).reshape(want.shape)
    a, b = outs["fragment"], outs["lds"]
    assert np.max(np.abs(a - b) / np.maximum(np.abs(b), 1e-3)) <= 2.0 ** -7


@pytest.mark.parametrize("M,K,N,G,zk,variant", [
    (128, 2048, 8192, 64, "8s", 0),      # config D2: grouped tiles (q on the MFMA, s/z folded per tile)
    (128, 2048, 8192, 64, "8s", 1),      # the other load depth
    (64, 512, 256, 32, "8s", 0),         # groups narrower than a K tile: hi + lo dequantized B
    (256, 512, 8192, 64, "8s", 0),
    (128, 1024, 512, 128, "any", 0),     # groups of two K tiles, zero points unrelated to s
    (64, 512, 256, 64, "any", 1),
    (128, 2048, 8192, 64, "any", 2),
])
def test_int4_gemm(dev, M, K, N, G, zk, variant):
    """Config D2: packed uint4 [N, K], per-group scale and zero point, w = u·s − z."""
    prog = configs.int4_matmul(M=M, K=K, N=N, G=G).with_variants({0: variant})
    rng = np.random.default_rng(11)
    u = rng.integers(0, 16, size=(N, K))
    s = _bf16_vals(401, N * K // G, 0.001, 0.02, kind="uniform").reshape(N, K // G)
    if zk == "8s":
        z = np.array([oracle.round_bf16(8.0 * v) for v in s.reshape(-1)]).reshape(s.shape)
    else:
        z = _bf16_vals(403, N * K // G, -0.1, 0.1, kind="uniform").reshape(s.shape)
    x = _bf16_vals(402, M * K).reshape(M, K)
    got, exe = run_on_gpu(dev, prog, {"x": x, "Wq": u.reshape(N, K // G, G), "S": s, "Z": z})
    packed = (u[:, 0::2] | (u[:, 1::2] << 4)).astype(np.uint8)
    want = oracle.int4_matmul(x, packed, s, z, G)
    err = bf16_rel(got["y"], want)
    _report(exe, got["y"], want)
    assert exe.stage_kernel(0).startswith("skeleton:gemm")
    assert ("grp" in exe.stage_kernel(0)) == (G % 64 == 0)
    assert err < 2e-2


def _same_as_generic(dev, monkeypatch, prog, vals, scale):
    """The skeleton's bf16 output against the generic f32 fold of the same program: both sum the
    same exact products in f32, so before the store they differ by at most K · 2^-24 of Σ|terms|
    (`scale`), and the store adds one bf16 step; infinities and NaNs sit at the same points."""
    got, exe = run_on_gpu(dev, prog, vals)
    kind = exe.stage_kernel(0)
    monkeypatch.setenv("SANIC_HIP_GENERIC", "1")
    want, exe = run_on_gpu(dev, prog, vals)
    monkeypatch.delenv("SANIC_HIP_GENERIC")
    assert exe.stage_kernel(0).startswith("fold:")
    a, b = np.asarray(got["y"], np.float64), np.asarray(want["y"], np.float64)
    fin = np.isfinite(b)
    assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[~fin & ~np.isnan(b)], b[~fin & ~np.isnan(b)]), kind
    over = np.abs(a[fin] - b[fin]) - 2.0 ** -7 * np.abs(b)[fin]
    print(kind, float(over.max() / scale))
    assert over.max() <= 2.0 ** -13 * scale, kind
    return kind


# rows, k and columns off every tile: below one tile, one past it, K tiles odd in number and
# overlapping, columns not a multiple of 8; operand planes past the static scratch
RAGGED = [(2, 64, 32), (65, 128, 96), (200, 2048, 8192), (33, 200, 77), (100, 72, 1003), (129, 1000, 333),
          (256, 128, 8224), (127, 832, 5184), (8, 4160, 96), (20, 2200, 49), (40, 2048, 8192), (300, 2000, 1088), (250, 2056, 2000),
          (90, 1536, 2820), (4100, 2048, 136)]


@pytest.mark.parametrize("kmajor", [False, True])
@pytest.mark.parametrize("M,K,N", RAGGED)
def test_rmsnorm_gemm_any_size(dev, monkeypatch, M, K, N, kmajor):
    prog = configs.rmsnorm_projection(M=M, K=K, N=N, kmajor=kmajor)
    x = _bf16_vals(321, M * K).reshape(M, K)
    w = _bf16_vals(323, K * N, 0.0, 0.02).reshape((K, N) if kmajor else (N, K))
    vals = {"x": x, "g": _bf16_vals(322, K, 1.0, 0.02), "W": w}
    assert "skeleton" in _same_as_generic(dev, monkeypatch, prog, vals, scale=0.02 * K)
    # an infinite activation in the last row, a NaN weight in the last column's last k
    x[M - 1, K - 1] = np.inf
    w[(K - 1, N - 1) if kmajor else (N - 1, K - 1)] = np.nan
    w[(0, 0)] = np.inf
    _same_as_generic(dev, monkeypatch, prog, vals, scale=0.02 * K)


@pytest.mark.parametrize("M,K,N,G", [(40, 1056, 8192, 1056), (2, 64, 32, 64), (16, 2048, 8192, 64), (100, 1152, 777, 64), (65, 384, 1000, 128),
                                     (33, 192, 64, 64), (17, 256, 300, 32), (31, 8320, 48, 64),
                                     (16, 512, 16, 512), (100, 1920, 3270, 64), (103, 1920, 777, 32), (128, 512, 512, 32)])
def test_int4_gemm_any_size(dev, monkeypatch, M, K, N, G):
    prog = configs.int4_matmul(M=M, K=K, N=N, G=G)
    s = _bf16_vals(331, N * K // G, 0.001, 0.02, kind="uniform").reshape(N, K // G)
    z = _bf16_vals(332, N * K // G, -0.1, 0.1, kind="uniform").reshape(s.shape)
    x = _bf16_vals(333, M * K).reshape(M, K)
    vals = {"x": x, "Wq": np.random.default_rng(5).integers(0, 16, size=(N, K // G, G)), "S": s, "Z": z}
    _same_as_generic(dev, monkeypatch, prog, vals, scale=0.2 * K)
    x[0, 0] = -np.inf
    s[N - 1, 0] = np.nan
    _same_as_generic(dev, monkeypatch, prog, vals, scale=0.2 * K)


@pytest.mark.parametrize("M,K,N,order", [
    (500, 2040, 1000, "nk"), (130, 1000, 640, "nk"), (257, 72, 96, "nk"),       # GEMM tiles whose first K tile overlaps the second
    (8, 256, 64, "nk"), (40, 200, 300, "nk"), (200, 1968, 1088, "nk"), (20, 136, 100, "kn"), (5, 2048, 72, "kn"),   # few-row kernel, x as stored
    (40, 2048, 8192, "nk view"), (100, 1000, 2056, "kn view"), (500, 200, 1000, "nk view"), (300, 2048, 4104, "kn view"),
    (64, 64, 32, "nk view"), (128, 512, 2048, "kn view"),                       # whole tiles
])
def test_projection_without_a_norm(dev, monkeypatch, M, K, N, order):
    """y = x · W with both operands as stored; a view of W keeps what the stored order takes."""
    prog = forms.projection(M, K, N, order)
    x = _bf16_vals(351, M * K).reshape(M, K)
    w = _bf16_vals(352, K * N, 0.0, 0.02).reshape(prog.by_name["W"].shape)
    kind = _same_as_generic(dev, monkeypatch, prog, {"x": x, "W": w}, scale=0.02 * K)
    assert kind.startswith("skeleton:gemm") and (M < 500 or "any size" in kind), kind
    x[M - 1, K - 1] = np.inf
    w[-1, -1] = np.nan
    _same_as_generic(dev, monkeypatch, prog, {"x": x, "W": w}, scale=0.02 * K)


@pytest.mark.parametrize("prog", [forms.projection(500, 2040, 1000, "nk", residual=True), forms.projection(20, 200, 300, "nk", residual=True),
                                  A.attention(4, 2, 100, 300, A.causal, epilogue=A.residual), A.attention(4, 2, 200, 200, A.causal, dt=ir.F32, epilogue=A.residual)])
def test_residual_and_output_in_one_buffer(dev, prog):
    """y = R + f(x) bound to R itself, an infinity among the operands: every point is read and
    stored once, so the bits are those of two buffers."""
    out = prog.buffers[-1].name
    vals = {b.name: _bf16_vals(360 + i, int(np.prod(b.shape))) for i, b in enumerate(prog.buffers[:-1])}
    vals["V" if "V" in vals else "x"][10] = np.inf       # (a key that every row of its head sees)
    exe = dev.prepare(prog)
    print(exe.stage_kernel(0), flush=True)
    assert exe.stage_kernel(0).startswith("skeleton:")
    bufs = {n: dev.from_values(v, prog.by_name[n].dtype) for n, v in vals.items()}
    bufs[out] = dev.from_values(vals["R"], ir.BF16)
    exe.execute_static(bufs)
    want = bufs[out].download()
    assert not np.isfinite(from_bf16_bits(np.frombuffer(want, np.uint16))).all()
    bufs[out] = bufs["R"]
    exe.execute_static(bufs)
    assert bufs["R"].download() == want


@pytest.mark.parametrize("kmajor", [False, True])
@pytest.mark.parametrize("M,K,N", [(8, 256, 64), (100, 320, 4096 + 24)])
def test_rmsnorm_gemm_any_address(dev, M, K, N, kmajor):
    """Rows and weights bound one element off a 16-byte boundary (the sizes that the generic fold
    took at any address): the same bits as bound on one."""
    prog = configs.rmsnorm_projection(M=M, K=K, N=N, kmajor=kmajor)
    vals = {"x": _bf16_vals(341, M * K), "g": _bf16_vals(342, K, 1.0, 0.02), "W": _bf16_vals(343, K * N, 0.0, 0.02)}
    exe = dev.prepare(prog)
    assert exe.stage_kernel(0).startswith("skeleton:gemm")
    bufs = {n: dev.from_values(v, ir.BF16) for n, v in vals.items()}
    want = exe.execute(bufs)["y"].download()
    for n in ("x", "W"):
        raw = bufs[n].download()
        hold = dev.alloc(len(raw) + 16)
        hold.upload(b"\0\0" + raw)
        bufs["hold" + n], bufs[n] = hold, dev.wrap(hold.device_ptr + 2, len(raw))
    assert exe.execute({n: bufs[n] for n in vals})["y"].download() == want
