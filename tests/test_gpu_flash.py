"""FlashAttention prefill (MFMA skeleton) on the GPU against the oracle."""
import numpy as np
import pytest

import oracle
from sanic_amd import configs, ir
from sanic_amd.program import SCRATCH, Program
from tests import attn_forms as A
from tests.util import floored_rel_err, max_rel_err, run_on_gpu

pytestmark = pytest.mark.gpu


def _inputs(NH, NKV, S, HD=64, seed=400):
    return {"Q": oracle.synth(seed, NH * S * HD, dtype=ir.BF16).reshape(NH, S, HD),
            "K": oracle.synth(seed + 1, NKV * S * HD, dtype=ir.BF16).reshape(NKV, S, HD),
            "V": oracle.synth(seed + 2, NKV * S * HD, dtype=ir.BF16).reshape(NKV, S, HD)}


@pytest.mark.parametrize("window", [0, 64])
def test_flash_small_matches_interpreter_schedule(dev, window):
    """The whole schedule (RoPE stages + flash fold) against the interpreter, stage by stage."""
    NH, NKV, S = 4, 2, 256
    prog = configs.flash_prefill(NH, NKV, S, window=window)
    vals = _inputs(NH, NKV, S)
    got, exe = run_on_gpu(dev, prog, vals)
    assert exe.stage_kernel(2).startswith("skeleton:flash_prefill")
    want = oracle.run_program(prog, vals)
    # bf16 output: the reference's GPU metric |g − e| / (1 + |e|) (tests/metal.rs:99-105) at the
    # bf16 bound; attention outputs straddle zero, so a relative-to-|e| metric would not apply
    err = max_rel_err(got["O"], want["O"])
    print(exe.stage_kernel(2), window, err, floored_rel_err(got["O"], want["O"]))
    assert err < 2e-2


def _rope_bf16(x, invf):
    r = oracle.rope(x, 0, invf)
    return np.vectorize(oracle.round_bf16)(r) if r.size < 4096 else _round_bf16_array(r)


def _round_bf16_array(x):
    f = np.ascontiguousarray(x, dtype=np.float32)
    b = f.view(np.uint32)
    r = ((b + 0x7FFF + ((b >> 16) & 1)) >> 16).astype(np.uint32) << 16
    return r.view(np.float32).astype(np.float64)


@pytest.mark.parametrize("window", [0, 1024])
def test_flash_full_size_all_heads(dev, window):
    """Config C1 (causal) / C2 (1024-token window) at full size: all 32 query heads against the
    fused f64 attention over the same RoPE'd, bf16-rounded Q and K. Every head is checked, since
    the kernel remaps blockIdx to (KV head, query head, query block) for XCD locality and a
    mapping error would touch only some heads."""
    NH, NKV, S, HD = 32, 8, 4096, 64
    prog = configs.flash_prefill(NH, NKV, S, window=window)
    vals = _inputs(NH, NKV, S, seed=500)
    got, exe = run_on_gpu(dev, prog, vals)
    invf = oracle.inv_freq(500000.0, HD // 2)
    kr = _round_bf16_array(oracle.rope(vals["K"], 0, invf))
    qr = _round_bf16_array(oracle.rope(vals["Q"], 0, invf))
    want = oracle.attention(qr, kr, vals["V"], 1.0 / 8.0, mask=2 if window else 1, window=window)
    per_head = [max_rel_err(got["O"][h], want[h]) for h in range(NH)]
    floored = floored_rel_err(got["O"], want)
    print(exe.stage_kernel(2), window, f"max |g-e|/(1+|e|) {max(per_head):.3e}",
          f"max |g-e|/max(|e|,1e-3) {floored:.3e}")
    bad = [h for h, err in enumerate(per_head) if not err < 2e-2]
    assert not bad, [(h, per_head[h]) for h in bad]


@pytest.mark.parametrize("S,window", [(256, 0), (384, 100)])
def test_flash_transposed_values_layout(dev, S, window):
    """V stored [NKV, HD, S] (keys contiguous, as in the decode cache) and read through a
    transposed view: the skeleton loads those rows as they lie and reads its PV operand without
    the transposing LDS read — against the oracle, and bit for bit against the same values
    stored [NKV, S, HD] (the MFMAs see the same operands in the same order)."""
    NH, NKV = 4, 2
    vals = _inputs(NH, NKV, S, seed=430)
    outs = []
    for vt in (False, True):
        prog = configs.flash_prefill(NH, NKV, S, window=window, rope_stages=False, v_transposed=vt)
        v = {"Q": vals["Q"], "K": vals["K"], "V": vals["V"].transpose(0, 2, 1).copy() if vt else vals["V"]}
        got, exe = run_on_gpu(dev, prog, v)
        assert exe.stage_kernel(0).startswith("skeleton:flash_prefill"), exe.stage_kernel(0)
        outs.append(got["O"])
        if vt:
            want = oracle.run_program(prog, v)["O"]
            err = max_rel_err(got["O"], want)
            print(S, window, err, floored_rel_err(got["O"], want))
            assert err < 2e-2
    assert np.array_equal(outs[0], outs[1])


@pytest.mark.parametrize("NH,NKV", [(8, 8), (16, 2), (8, 1), (16, 16), (24, 8)])
def test_flash_head_groupings(dev, NH, NKV):
    """Query heads per KV head 1 (MHA), 8 and 3, and KV head counts on both sides of the
    XCD-aware block order (a multiple of 8 or not): every head against the oracle."""
    S = 128
    prog = configs.flash_prefill(NH, NKV, S, rope_stages=False)
    vals = _inputs(NH, NKV, S, seed=450 + NH + NKV)
    got, exe = run_on_gpu(dev, prog, vals)
    assert exe.stage_kernel(0).startswith("skeleton:flash_prefill"), exe.stage_kernel(0)
    want = oracle.run_program(prog, vals)["O"]
    err = max_rel_err(got["O"], want)
    print(NH, NKV, err, floored_rel_err(got["O"], want))
    assert err < 2e-2


@pytest.mark.parametrize("NH,NKV,S,window", [
    (4, 2, 40, 0),        # one query block, one key tile, both partly past the end
    (8, 8, 63, 0),
    (4, 2, 129, 0),       # one row into a third block, one key into a third tile
    (4, 2, 200, 100),     # a window ending inside a tile
    (2, 1, 321, 70),
    (6, 2, 512 + 64, 0),  # whole key tiles, rows not a multiple of 128
    (1, 1, 256, 0),       # a single head: no head dim in the grid
    (1, 1, 100, 30),
])
def test_flash_any_length(dev, monkeypatch, NH, NKV, S, window):
    """Lengths off the tiles against the generic f32 fold of the same program: the skeleton keeps
    q and the softmax weights to 16 significant bits (hi + lo), so the two differ by no more than
    the bf16 store of values 2^-16 · Σ p|v| ≤ 1e-4 apart — at most one bf16 step beside that.
    Once more with K and V bound one element off a 16-byte boundary: the same bits."""
    prog = configs.flash_prefill(NH, NKV, S, window=window)
    vals = _inputs(NH, NKV, S, seed=470 + S)
    got, exe = run_on_gpu(dev, prog, vals)
    assert exe.stage_kernel(2).startswith("skeleton:flash_prefill"), exe.stage_kernel(2)
    bufs = {n: dev.from_values(v, ir.BF16) for n, v in vals.items()}
    for n in ("K", "V"):
        raw = bufs[n].download()
        hold = dev.alloc(len(raw) + 16)
        hold.upload(b"\0\0" + raw + b"\0\0")
        bufs[n + "hold"], bufs[n] = hold, dev.wrap(hold.device_ptr + 2, len(raw))
    off = exe.execute({n: bufs[n] for n in ("Q", "K", "V")})["O"].read(ir.BF16, NH * S * 64).reshape(NH, S, 64)
    assert np.array_equal(off, got["O"])
    monkeypatch.setenv("SANIC_HIP_GENERIC", "1")
    want, exe = run_on_gpu(dev, prog, vals)
    assert exe.stage_kernel(2).startswith("fold:"), exe.stage_kernel(2)
    over = np.abs(got["O"] - want["O"]) - 2.0 ** -7 * np.abs(want["O"])
    print(S, window, float(over.max()), max_rel_err(got["O"], want["O"]))
    assert over.max() < 1e-4


def test_flash_any_length_keeps_infinities_and_nans(dev, monkeypatch):
    """A NaN value row, an infinite value and an infinite key late in the prompt: the rows before
    them see nothing of them, and every point is finite or not exactly where the generic fold's is."""
    NH, NKV, S = 2, 1, 100
    prog = configs.flash_prefill(NH, NKV, S, window=30)
    vals = _inputs(NH, NKV, S, seed=490)
    vals["V"][0, 50] = np.nan
    vals["V"][0, 90, 3] = -np.inf
    vals["K"][0, 75, 5] = np.inf
    got, _ = run_on_gpu(dev, prog, vals)
    monkeypatch.setenv("SANIC_HIP_GENERIC", "1")
    want, _ = run_on_gpu(dev, prog, vals)
    g, w = got["O"], want["O"]
    assert np.isfinite(w).any() and np.isnan(w).any()
    assert np.array_equal(np.isnan(g), np.isnan(w)) and np.array_equal(np.isinf(g), np.isinf(w))
    fin = np.isfinite(w)
    assert np.max(np.abs(g[fin] - w[fin]) - 2.0 ** -7 * np.abs(w[fin])) < 1e-4


def _attention_f32(NH, NKV, NQ, T, HD, E, causal, dtypes):
    """softmax(q·kᵀ/√HD + mask)·v with f32 output; NH = 0: no head dim."""
    from sanic_amd import carrier as C
    from sanic_amd.program import STREAM, Program
    p = Program()
    lead, klead = ((NH,), (NKV,)) if NH else ((), ())
    q, k, v = (p.input(n, shp, dt) for n, shp, dt in zip("QKV", (lead + (NQ, HD), klead + (T, HD), klead + (T, E)), dtypes))
    if NH:
        k, v = ir.expand_heads(k, 0, NH // NKV), ir.expand_heads(v, 0, NH // NKV)
        s = ir.reduce(ir.map_(ir.MUL, ir.unsqueeze(q, 2), ir.unsqueeze(k, 1)), 3, ir.M_ADD)
    else:
        s = ir.matmul(q, ir.transpose(k, 0, 1))
    s = ir.map_(ir.MUL, s, ir.const(HD ** -0.5))
    h = len(lead)
    if causal:
        s = ir.map_(ir.ADD, s, ir.causal_mask_like(s, h, h + 1))
    sb, vb = ((0, 1, STREAM), (0, STREAM, 2)) if NH else ((0, STREAM), (STREAM, 1))
    p.fused("O", lead + (NQ, E), T, [(s, sb), (v, vb)], C.online_softmax_weighted(), ir.F32)
    return p


F, B = ir.F32, ir.BF16


@pytest.mark.parametrize("NH,NKV,NQ,T,HD,E,causal,dtypes", [
    (0, 0, 129, 129, 64, 64, True, (F, F, F)),    # one row into a ninth block
    (0, 0, 400, 400, 32, 32, True, (F, F, F)),
    (0, 0, 1000, 1000, 64, 64, True, (F, F, F)),
    (0, 0, 65, 300, 16, 128, False, (F, F, F)),   # more keys than rows, value tiles of 8
    (6, 2, 60, 60, 128, 16, True, (F, F, F)),     # grouped heads, d above the value size
    (16, 16, 260, 5, 48, 32, False, (B, F, B)),   # fewer keys than a tile, stored types mixed
    (2, 1, 150, 150, 128, 128, True, (F, F, F)),  # the largest operands, whose registers are the most
])
def test_attention_f32_matches_generic(dev, monkeypatch, NH, NKV, NQ, T, HD, E, causal, dtypes):
    """Both evaluations are f32 throughout: scores within HD · 2^-24 of Σ|q·k| ≤ HD of each other,
    so the weights and outputs (|v| ≲ 4) within a few 1e-5 at most; and infinities and NaNs in the
    keys and values that some rows do not see sit at the same points."""
    prog = _attention_f32(NH, NKV, NQ, T, HD, E, causal, dtypes)
    vals = {n: oracle.synth(500 + i, int(np.prod(prog.by_name[n].shape)), dtype=prog.by_name[n].dtype).reshape(prog.by_name[n].shape)
            for i, n in enumerate("QKV")}
    for odd in (False, True):
        if odd:
            vals["V"][..., T - 1, 0] = np.nan
            vals["K"][..., T // 2, 1] = np.inf
        got, exe = run_on_gpu(dev, prog, vals)
        assert exe.stage_kernel(0).startswith("skeleton:attn_f32"), exe.stage_kernel(0)
        monkeypatch.setenv("SANIC_HIP_GENERIC", "1")
        want, _ = run_on_gpu(dev, prog, vals)
        monkeypatch.delenv("SANIC_HIP_GENERIC")
        g, w = got["O"], want["O"]
        fin = np.isfinite(w)
        assert np.array_equal(np.isnan(g), np.isnan(w)) and np.array_equal(fin, np.isfinite(g))
        if fin.any():
            err = max_rel_err(g[fin], w[fin])
            print(odd, err)
            assert err < 2e-5


@pytest.mark.parametrize("NH,NKV,S,window,teams", [
    (2, 1, 1024, 0, "+teams4"),      # whole tiles, 64-row blocks
    (12, 4, 1024 + 64, 0, "+teams4"),   # 17 tiles over 4 teams: teams of 4 and 5
    (1, 1, 800, 0, "+teams4"),       # a single head, 13 tiles, the last of them partial
    (32, 8, 600, 0, "+teams2"),      # 320 blocks: 2 teams
    (2, 1, 1024, 200, ""),           # a window of 5 tiles: one team
])
def test_flash_key_teams(dev, NH, NKV, S, window, teams):
    """Small launches: teams of waves over every 2nd or 4th key tile, merged at the end, against the
    fused f64 attention over the same RoPE'd, bf16-rounded K (and Q, where the kernel rounds it)."""
    prog = configs.flash_prefill(NH, NKV, S, window=window)
    vals = _inputs(NH, NKV, S, seed=520 + S)
    got, exe = run_on_gpu(dev, prog, vals)
    kind = exe.stage_kernel(2)
    assert kind.startswith("skeleton:flash_prefill") and kind.endswith("]" + teams), kind
    invf = oracle.inv_freq(500000.0, 32)
    kr = _round_bf16_array(oracle.rope(vals["K"], 0, invf))
    qr = oracle.rope(vals["Q"], 0, invf)
    if "any length" not in kind:
        qr = _round_bf16_array(qr)
    want = oracle.attention(qr, kr, vals["V"], 1.0 / 8.0, mask=2 if window else 1, window=window)
    err = max_rel_err(got["O"], want)
    print(kind, err)
    assert err < 2e-2


@pytest.mark.parametrize("S,H,F", [(1, 1, 8), (33, 1, 8), (128, 3, 32), (77, 2, 24)])
def test_rotation_table_and_keys_in_one_launch(dev, monkeypatch, S, H, F):
    """The rotation table and the keys rotated by it, formed in one launch, against the two generic
    stages: the table bit for bit, the keys within a bf16 step and what contracting the other of the
    two products changes in f32. Workgroups past the table's runs, partly filled ones, one run."""
    p = Program()
    k = p.input("K", (H, S, 2 * F), ir.BF16)
    invf = ir.map_(ir.EXP, ir.map_(ir.MUL, ir.iota(F), ir.const(-0.4)))
    table = p.pointwise("table", ir.rope_table(ir.iota(S), invf), ir.F32, role=SCRATCH)
    kr = p.pointwise("Kr", ir.rope_tabled(k, table), ir.BF16, role=SCRATCH)
    p.pointwise("Y", ir.map_(ir.MUL, kr, ir.const(1.0)), ir.F32)
    p.pointwise("T", ir.map_(ir.MUL, table, ir.const(1.0)), ir.F32)
    vals = {"K": np.random.default_rng(5).standard_normal((H, S, 2 * F))}
    got, exe = run_on_gpu(dev, p, vals)
    assert [exe.stage_kernel(i) for i in range(2)] == ["pointwise:runs8[2 stages]", "absorbed-into:0"]
    monkeypatch.setenv("SANIC_HIP_GENERIC", "1")
    want, exe = run_on_gpu(dev, p, vals)
    assert exe.stage_kernel(1) == "pointwise"
    np.testing.assert_array_equal(got["T"], want["T"])
    a, b = np.asarray(got["Y"], np.float64), np.asarray(want["Y"], np.float64)
    assert np.all(np.abs(a - b) <= 2.0 ** -7 * np.abs(b) + 2.0 ** -22 * np.abs(vals["K"]).max())


def _form_values(prog, seed):
    """Seeded inputs for every input buffer; `position` two thirds along the keys that K holds."""
    T = prog.by_name["K"].shape[-2]
    out = {}
    for i, b in enumerate(b for b in prog.buffers if b.role == 0):
        n = int(np.prod(b.shape)) if b.shape else 1
        out[b.name] = np.array(float(2 * T // 3)) if b.name == "position" else np.asarray(
            oracle.synth(seed + i, n, dtype=b.dtype), np.float64).reshape(b.shape)
    return out


@pytest.mark.parametrize("terms", [A.prefix, A.chunk, A.bias, lambda p, s: A.bias(p, s) + A.prefix(p, s)])
@pytest.mark.parametrize("NH,NKV,NQ,T,dt", [
    (4, 2, 128, 128, ir.BF16),      # whole tiles
    (4, 2, 100, 300, ir.BF16),      # any length
    (0, 0, 40, 1000, ir.BF16),      # no head dim
    (0, 0, 200, 200, ir.F32),
    (4, 2, 200, 200, ir.F32),
])
def test_masks_and_epilogues_that_read_buffers(dev, NH, NKV, NQ, T, dt, terms):
    """Masks and biases from buffers in the scores, a stored residual in the epilogue, against the
    f64 interpreter; the inputs come back as they were given."""
    prog = A.attention(NH, NKV, NQ, T, terms, dt=dt, out=ir.F32, epilogue=A.residual)
    vals = _form_values(prog, 540)
    exe = dev.prepare(prog)
    kind = exe.stage_kernel(0)
    print(kind, flush=True)
    assert kind.startswith("skeleton:flash_prefill" if dt == ir.BF16 else "skeleton:attn_f32"), kind
    bufs = {n: dev.from_values(v, prog.by_name[n].dtype) for n, v in vals.items()}
    held = {n: b.download() for n, b in bufs.items()}
    got = exe.execute(bufs)["O"].read(ir.F32, int(np.prod(prog.by_name["O"].shape))).reshape(prog.by_name["O"].shape)
    assert all(b.download() == held[n] for n, b in bufs.items())
    err = max_rel_err(got, oracle.run_program(prog, vals)["O"])
    print(err)
    # whole tiles round the softmax weights to bf16 (2^-9 of Σ p|v| ≲ 3); the others hold 16 bits or more
    assert err < (1e-2 if "any length" not in kind and dt == ir.BF16 else 1e-4)


def _against_interpreter(dev, prog, seed, bound, kind, **given):
    vals = dict(_form_values(prog, seed), **given)
    exe = dev.prepare(prog)
    print(exe.stage_kernel(0), flush=True)
    assert exe.stage_kernel(0).startswith(kind)
    bufs = {n: dev.from_values(v, prog.by_name[n].dtype) for n, v in vals.items()}
    got = exe.execute(bufs)["O"].read(ir.F32, int(np.prod(prog.by_name["O"].shape))).reshape(prog.by_name["O"].shape)
    err = max_rel_err(got, oracle.run_program(prog, vals)["O"])
    print(err)
    assert err < bound


@pytest.mark.parametrize("name", A.EDGES)
@pytest.mark.parametrize("NH,NKV,NQ,T,dt", [(4, 2, 128, 192, ir.BF16), (4, 2, 100, 300, ir.BF16), (0, 0, 200, 200, ir.F32)])
def test_windows_that_move_one_way(dev, NH, NKV, NQ, T, dt, name):
    """Falling, halved, clamped and iota-written window edges, rows without a visible key among
    them, against the f64 interpreter."""
    prog = A.attention(NH, NKV, NQ, T, A.EDGES[name], dt=dt, out=ir.F32)
    given = {"position": np.array(-1.0 if dt == ir.F32 else 0.75)} if "position" in prog.by_name else {}
    whole = NQ % 128 == 0 and T % 64 == 0 and dt == ir.BF16
    # as test_masks_and_epilogues_that_read_buffers
    _against_interpreter(dev, prog, 560, 1e-2 if whole else 1e-4, "skeleton:flash_prefill" if dt == ir.BF16 else "skeleton:attn_f32", **given)


@pytest.mark.parametrize("rows,T,terms,kind", [
    (2, 300, A.prefix, "skeleton:attn_decode"), (8, 300, A.prefix, "skeleton:attn_decode"),
    (5, 2049, A.prefix, "skeleton:attn_decode"), (8, 1000, A.bias, "skeleton:attn_decode"),
    (17, 1024, A.prefix, "skeleton:attn_f32"), (9, 4096, A.causal, "skeleton:attn_f32"), (8, 2050, A.chunk, "skeleton:attn_f32"),
    (8, 1000, A.chunk, "skeleton:flash_prefill"), (3, 300, A.causal, "skeleton:flash_prefill"),
])
def test_few_query_rows_without_heads(dev, rows, T, terms, kind):
    """Rows sharing a window, and rows each with a window of its own, over short and long caches."""
    _against_interpreter(dev, A.attention(0, 0, rows, T, terms, out=ir.F32), 580, 1e-5, kind)


@pytest.mark.parametrize("NH,NKV,kind", [(8, 2, "fold:"), (4, 4, "skeleton:attn_decode")])
def test_heads_each_with_a_window(dev, NH, NKV, kind):
    _against_interpreter(dev, A.heads(NH, NKV, 1000, A.edge_per_head), 590, 1e-5, kind, edge=np.linspace(5.0, 990.0, NH))


@pytest.mark.parametrize("out", [ir.F32, ir.F16, ir.BF16])
@pytest.mark.parametrize("NH,NKV,NQ,T,terms,qscale", [
    (4, 2, 100, 300, A.causal, False), (4, 2, 100, 300, A.EDGES["window"], True), (2, 1, 1000, 1000, A.causal, True), (0, 0, 200, 200, A.causal, True),
])
def test_any_length_is_no_further_from_64_bits_than_the_fold(dev, monkeypatch, NH, NKV, NQ, T, terms, qscale, out):
    """Softmax weights and a computed query side go to the matrix cores as bf16 terms: two where the
    output is bf16, else three (24 bits, what the f32 fold holds). Against the f64 value before the
    output's rounding."""
    forms = {o: A.attention(NH, NKV, NQ, T, terms, out=o, qscale=qscale) for o in (out, ir.F32)}
    vals = _form_values(forms[out], 600)
    want = oracle.run_program(forms[ir.F32], vals)["O"]
    errs, kinds = [], []
    for generic in (False, True):
        if generic:
            monkeypatch.setenv("SANIC_HIP_GENERIC", "1")
        exe = dev.prepare(forms[out])
        kinds.append(exe.stage_kernel(0))
        bufs = {n: dev.from_values(v, forms[out].by_name[n].dtype) for n, v in vals.items()}
        got = exe.execute(bufs)["O"].read(out, int(np.prod(want.shape))).reshape(want.shape)
        errs.append(float(np.sqrt(np.mean((got - want) ** 2))))
    print(kinds, errs, flush=True)
    assert kinds[0].startswith("skeleton:flash_prefill") and kinds[1].startswith("fold:")
    # f32: both are 24-bit sums, in different orders (within a quarter of each other); a narrower store's
    # rounding is the error of both
    assert errs[0] <= (1.25 if out == ir.F32 else 1.01) * errs[1]


@pytest.mark.parametrize("NH,NKV,S,window", [(4, 2, 512, 0), (2, 1, 2048, 0), (4, 1, 1024, 300), (8, 2, 4096, 0)])
def test_small_launches_are_no_further_from_64_bits_than_large_ones(dev, NH, NKV, S, window):
    """Whole tiles in 64-row blocks, and key teams that each keep a running maximum of their own, round
    the softmax weights to bf16 against other reference points than the 128-row form: other
    last bits of the output, the same distance from 64 bits."""
    def terms(p, s):
        low = [A.mask(A.key(s), ir.map_(ir.SUB, A.row(s), ir.const(window - 1.0)), -1e30, 0.0)]
        return A.causal(p, s) + (low if window else [])
    prog = A.attention(NH, NKV, S, S, terms, out=ir.F32)
    vals = _form_values(prog, 620)
    q, k, v = (np.asarray(vals[n], np.float64) for n in "QKV")
    i, j = np.arange(S)[:, None], np.arange(S)[None, :]
    hidden = (j > i) | ((j < i - (window - 1)) if window else False)
    want = np.empty_like(q)
    for h in range(NH):
        s = np.where(hidden, -np.inf, q[h] @ k[h // (NH // NKV)].T / 8.0)
        e = np.exp(s - s.max(axis=1, keepdims=True))
        want[h] = e @ v[h // (NH // NKV)] / e.sum(axis=1, keepdims=True)
    errs, kinds, outs = [], [], []
    for variant in (0, 1):
        exe = dev.prepare(prog.with_variants({0: variant}))
        kinds.append(exe.stage_kernel(0))
        bufs = {n: dev.from_values(x, prog.by_name[n].dtype) for n, x in vals.items()}
        outs.append(exe.execute(bufs)["O"].read(ir.F32, want.size).reshape(want.shape))
        errs.append(float(np.sqrt(np.mean((outs[-1] - want) ** 2))))
    apart = float(np.sqrt(np.mean((outs[0] - outs[1]) ** 2) / np.mean(want ** 2)))
    print(kinds, errs, "rms", float(np.sqrt(np.mean(want ** 2))), "apart", apart, flush=True)
    assert errs[0] <= 1.02 * errs[1]
