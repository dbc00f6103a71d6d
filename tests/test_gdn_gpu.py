"""GPU parity of the gated-delta-net ops (include/inl_gdn.h) through the C ABI
against the oracle (oracle/gdn.py, pinned by tests/test_oracle_gdn.py).

Bars:
- convolution, gated norm: the reference kernels' op sequence restated in
  numpy float32 (``*_ops``); every element within 4 ulps of it in f32 and
  equal or one bf16 ulp apart in bf16. The sources of difference are exp,
  whose device and numpy float32 results differ by an ulp for a good share
  of arguments, and, in the norm, the order of the 128-term f32 sum of
  squares (not fixed by the reference either: its Metal kernel and candle sum
  in other orders), which moves the f32 result by up to ~13 ulps: the norm's
  f32 bar is 16 ulps. At least 99% of bf16 results and half of the f32 ones
  are bit-equal;
- gates: within 1e-6 of the float32 restatement;
- unit-lower inverse: bit-equal to the float32 restatement (same products
  and sums in the same order, no transcendental);
- rule: against the f64 per-token recurrence, max-abs error within 1e-4 for
  the reference's own inputs in [-0.5, 0.5] (its chunked-vs-recurrent bar,
  qwen3_5.rs:1063-1160) and 2e-4 x max|ref| for N(0, 1) inputs; at the pplx
  shape (16 texts x 4096 tokens, 16 heads, dk = dv = 128) on sampled
  (text, head) pairs, plus linearity in v over the whole output;
- the tiny pplx-late tower with these ops on the GPU matches the HF golden
  vectors within the reference's 1e-4.
"""
import numpy as np
import pytest

from oracle import gdn as og

import tiny_encoders as te

pytestmark = pytest.mark.gpu


def _t(torch, x, dev, dtype):
    return torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).to(dev).to(dtype)


def _tdtype(torch, name):
    return torch.float32 if name == "f32" else torch.bfloat16


def _close_ulps(got, want, dtype, ulps=4):
    got, want = np.asarray(got, np.float32), np.asarray(want, np.float32)
    same = got == want
    if dtype == "f32":
        ok = np.abs(got - want) <= ulps * np.spacing(np.abs(want))
    else:
        ok = np.abs(got - want) <= np.abs(want) * 2.0 ** -7 + 1e-30
    return bool(ok.all()), float(same.mean())


def _min_equal(dtype):
    return 0.5 if dtype == "f32" else 0.99


CONV_CASES = [
    ("f32", 64, 4, [0, 1, 17, 3, 40, 0, 100]),
    ("bf16", 64, 4, [0, 1, 17, 3, 40, 0, 100]),
    ("f32", 37, 3, [5, 33, 16]),
    ("bf16", 40, 1, [2, 31]),
    ("bf16", 24, 8, [1, 2, 9, 70]),
]


@pytest.mark.parametrize("case", CONV_CASES, ids=[f"{c[0]}-c{c[1]}-k{c[2]}" for c in CONV_CASES])
def test_conv_matches_reference_op_sequence(case, cuda, inl):
    import torch
    dtype, ch, taps, lens = case
    print(f"case=gdn_conv {case}", flush=True)
    rng = np.random.default_rng(ch * 10 + taps)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    x = og._r(rng.standard_normal((cu[-1], ch)).astype(np.float32) * 2, dtype)
    w = og._r((rng.standard_normal((ch, taps)) * 0.6).astype(np.float32), dtype)
    td = _tdtype(torch, dtype)
    got = inl.gdn_conv(_t(torch, x, cuda, td), cu.tolist(), _t(torch, w, cuda, td)).float().cpu().numpy()
    want = og.causal_conv_ops(x, cu, w, dtype)
    ok, same = _close_ulps(got, want, dtype)
    print(f"gdn_conv {case}: bit-equal {same:.5f}", flush=True)
    assert ok and same >= _min_equal(dtype)


def test_conv_strided_input_and_output(cuda, inl):
    """x read as a column block of a wider projection output (row stride >
    channels): the projected tensor's q/k/v block."""
    import torch
    rng = np.random.default_rng(7)
    cu = np.array([0, 50, 90], np.int32)
    wide = rng.standard_normal((90, 96)).astype(np.float32)
    w = (rng.standard_normal((64, 4)) * 0.5).astype(np.float32)
    xd = torch.from_numpy(wide).to(cuda)[:, 16:80]
    got = inl.gdn_conv(xd, cu.tolist(), torch.from_numpy(w).to(cuda)).cpu().numpy()
    ok, same = _close_ulps(got, og.causal_conv_ops(wide[:, 16:80], cu, w), "f32")
    assert ok and same >= _min_equal("f32")


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_gates_match_f32_restatement(dtype, cuda, inl):
    import torch
    rng = np.random.default_rng(11)
    a = og._r(rng.standard_normal((300, 16)).astype(np.float32) * 3, dtype)
    b = og._r(rng.standard_normal((300, 16)).astype(np.float32) * 3, dtype)
    dt = rng.standard_normal(16).astype(np.float32)
    neg_a = -np.exp(np.log(rng.uniform(0.5, 4, 16))).astype(np.float32)
    td = _tdtype(torch, dtype)
    g, beta = inl.gdn_gates(_t(torch, a, cuda, td), _t(torch, b, cuda, td), _t(torch, dt, cuda, torch.float32),
                            _t(torch, neg_a, cuda, torch.float32))
    g32, b32 = og.gates_ops(a, b, dt, neg_a)
    assert np.abs(g.cpu().numpy() - g32).max() <= 1e-6 * max(1.0, np.abs(g32).max())
    assert np.abs(beta.cpu().numpy() - b32).max() <= 1e-6


@pytest.mark.parametrize("size", [1, 2, 8, 16, 33, 64])
def test_unit_lower_inverse_bit_equal(size, cuda, inl):
    import torch
    rng = np.random.default_rng(size)
    a = np.tril(rng.standard_normal((50, size, size)).astype(np.float32) * 0.4, -1)
    got = inl.unit_lower_inverse(torch.from_numpy(a).to(cuda)).cpu().numpy()
    want = og.unit_lower_inverse_ops(a)
    assert np.array_equal(got, want)
    eye = np.eye(size)
    assert np.abs((eye + a.astype(np.float64)) @ got - eye).max() < 1e-3


def _pseudo(n, seed):
    state = (seed * 2654435761 + 1) & 0xFFFFFFFF
    out = np.empty(n, np.float32)
    for i in range(n):
        state = (state * 1664525 + 1013904223) & 0xFFFFFFFF
        out[i] = np.float32(state >> 8) / np.float32(1 << 24) - np.float32(0.5)
    return out


RULE_CASES = [
    # dtype, nk, nv, dk, dv, lengths, inputs
    ("f32", 1, 3, 4, 3, [1, 7, 8, 63, 64, 65, 145], "pseudo"),
    ("f32", 2, 4, 8, 6, [145, 0, 17], "pseudo"),
    ("f32", 2, 4, 128, 128, [1, 15, 16, 17, 200], "normal"),
    ("bf16", 2, 4, 128, 128, [33, 0, 100], "normal"),
    ("bf16", 4, 8, 64, 96, [16, 40], "normal"),
    ("f32", 1, 1, 100, 37, [70], "normal"),
]


@pytest.mark.parametrize("case", RULE_CASES, ids=[f"{c[0]}-{c[1]}x{c[2]}-{c[3]}x{c[4]}-{c[6]}" for c in RULE_CASES])
def test_rule_matches_recurrence(case, cuda, inl):
    import torch
    dtype, nk, nv, dk, dv, lens, kind = case
    print(f"case=gdn_rule {case}", flush=True)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    n, ch = int(cu[-1]), 2 * nk * dk + nv * dv
    if kind == "pseudo":
        mixed = _pseudo(n * ch, 11).reshape(n, ch)
        g = -0.3 * (_pseudo(n * nv, 14).reshape(n, nv) + 0.5)
        beta = _pseudo(n * nv, 15).reshape(n, nv) + 0.5
    else:
        rng = np.random.default_rng(dk + dv)
        mixed = rng.standard_normal((n, ch)).astype(np.float32)
        g = -rng.uniform(0, 0.5, (n, nv)).astype(np.float32)
        beta = rng.uniform(0, 1, (n, nv)).astype(np.float32)
    mixed = og._r(mixed, dtype)
    td = _tdtype(torch, dtype)
    got = inl.gdn_rule(_t(torch, mixed, cuda, td), cu.tolist(), nk, nv, dk, dv,
                       _t(torch, g, cuda, torch.float32), _t(torch, beta, cuda, torch.float32)).cpu().numpy()
    ref = og.rule_packed(mixed, cu, nk, nv, dk, dv, g.astype(np.float64), beta.astype(np.float64))
    err = np.abs(got - ref).max()
    bar = 1e-4 if kind == "pseudo" else 2e-4 * max(1.0, np.abs(ref).max())
    print(f"gdn_rule {case[:5]}: max abs err {err:.3g} (bar {bar:.3g})", flush=True)
    assert err <= bar


def test_rule_full_size_sampled_and_linear_in_v(cuda, inl):
    """pplx shape: 16 texts x 4096 tokens, 16 key / 16 value heads, dk = dv =
    128, bf16 mixed. Two (text, head) pairs against the f64 recurrence over
    all 4096 tokens; linearity in v checked on the whole output."""
    import torch
    nk = nv = 16
    dk = dv = 128
    lens = [4096] * 16
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    n, ch = int(cu[-1]), 2 * nk * dk + nv * dv
    gen = torch.Generator(device=cuda).manual_seed(5)
    mixed = torch.randn(n, ch, generator=gen, device=cuda).to(torch.bfloat16)
    g = -torch.rand(n, nv, generator=gen, device=cuda) * 0.2
    beta = torch.rand(n, nv, generator=gen, device=cuda)
    print("case=gdn_rule full size 16x4096, 16 heads, 128x128", flush=True)
    out = inl.gdn_rule(mixed, cu.tolist(), nk, nv, dk, dv, g, beta)
    torch.cuda.synchronize()
    for b, h in [(0, 0), (13, 11)]:
        a, e = int(cu[b]), int(cu[b + 1])
        m = mixed[a:e].float().cpu().numpy().astype(np.float64)
        ref = og.recurrent_rule(m[:, h * dk:(h + 1) * dk], m[:, (nk + h) * dk:(nk + h + 1) * dk],
                                m[:, 2 * nk * dk + h * dv:2 * nk * dk + (h + 1) * dv],
                                g[a:e, h].cpu().numpy().astype(np.float64), beta[a:e, h].cpu().numpy().astype(np.float64))
        err = np.abs(out[a:e, h].cpu().numpy() - ref).max()
        print(f"text {b} head {h}: max abs err {err:.3g}, max |ref| {np.abs(ref).max():.3g}", flush=True)
        assert err <= 2e-4 * max(1.0, np.abs(ref).max())
    # linearity in v: split v over even and odd tokens (an exact split), then
    # out(v_even) + out(v_odd) == out(v) with q, k, g, beta fixed
    v0 = 2 * nk * dk
    odd = (torch.arange(n, device=cuda) % 2 == 1)[:, None]
    m_even, m_odd = mixed.clone(), mixed.clone()
    m_even[:, v0:] = torch.where(odd, torch.zeros_like(mixed[:, v0:]), mixed[:, v0:])
    m_odd[:, v0:] = torch.where(odd, mixed[:, v0:], torch.zeros_like(mixed[:, v0:]))
    o_even = inl.gdn_rule(m_even, cu.tolist(), nk, nv, dk, dv, g, beta)
    o_odd = inl.gdn_rule(m_odd, cu.tolist(), nk, nv, dk, dv, g, beta)
    torch.cuda.synchronize()
    diff = (o_even + o_odd - out).abs().max().item()
    scale = out.abs().max().item()
    print(f"linearity: max diff {diff:.3g} (scale {scale:.3g})", flush=True)
    assert diff <= 1e-4 * max(1.0, scale)


@pytest.mark.parametrize("dtype,core_f32", [("f32", True), ("bf16", True), ("bf16", False)])
def test_gated_norm_matches_reference_op_sequence(dtype, core_f32, cuda, inl):
    import torch
    rng = np.random.default_rng(21)
    n, heads, dv = 257, 4, 128
    core = rng.standard_normal((n, heads, dv)).astype(np.float32)
    if not core_f32:
        core = og._r(core, dtype)
    z = og._r(rng.standard_normal((n, heads, dv)).astype(np.float32) * 2, dtype)
    w = og._r((1 + 0.3 * rng.standard_normal(dv)).astype(np.float32), dtype)
    td = _tdtype(torch, dtype)
    cd = torch.float32 if core_f32 else td
    got = inl.gdn_gated_norm(_t(torch, core, cuda, cd), _t(torch, z, cuda, td), _t(torch, w, cuda, td),
                             1e-6).float().cpu().numpy()
    want = og.gated_norm_ops(core, z, w, 1e-6, dtype)
    ok, same = _close_ulps(got, want, dtype, ulps=16)
    print(f"gated_norm {dtype} core_f32={core_f32}: bit-equal {same:.5f}", flush=True)
    assert ok and same >= _min_equal(dtype)


def test_gated_norm_odd_width(cuda, inl):
    import torch
    rng = np.random.default_rng(22)
    core = rng.standard_normal((9, 3, 37)).astype(np.float32)
    z = rng.standard_normal((9, 3, 37)).astype(np.float32)
    w = rng.standard_normal(37).astype(np.float32)
    got = inl.gdn_gated_norm(torch.from_numpy(core).to(cuda), torch.from_numpy(z).to(cuda),
                             torch.from_numpy(w).to(cuda), 1e-6).cpu().numpy()
    ok, same = _close_ulps(got, og.gated_norm_ops(core, z, w, 1e-6), "f32", ulps=16)
    assert ok and same >= _min_equal("f32")


@pytest.mark.parametrize("task", ["query", "document"])
def test_tiny_late_tower_on_gpu_matches_golden(task, cuda, inl):
    import torch
    fx = te.load_late_fixture()
    g = fx[2]
    case = next(c for c in g["cases"] if c["task"] == task)
    out, lens = te.qwen35_late_encode(fx, g["texts"], task, te.HipOps(inl, torch, cuda))
    assert lens == case["lengths"]
    for key in ("alone", "batched"):
        worst = max(np.abs(a - np.asarray(r)).max() for a, r in zip(out, case[key]) if a.size)
        print(f"tiny late {task} {key}: {worst:.3g}", flush=True)
        assert worst < 1e-4


# The chunked rule (key and value dim 128, 40 tokens a text on average): text
# lengths at the edges of its 64-token (bf16) and 32-token (f32) chunks, empty
# texts, texts that start off a chunk's multiple, head counts that do not fill
# its workgroups of four, and gates from no decay to e^-30 (whose running sum
# must not lose the small decays that follow). Against the f64 recurrence on
# the same inputs: values are sums of order 1 over f32 products, so 2^-24 per
# rounding, some 40 roundings deep: 5e-6 of the largest value.
CHUNK_CASES = [
    ("bf16", 2, 2, [64], "small"), ("bf16", 2, 2, [65, 63, 128], "small"), ("f32", 2, 2, [32, 33, 95], "small"),
    ("f32", 1, 3, [97, 0, 31, 160], "mixed"), ("bf16", 1, 5, [1, 0, 200, 130, 0], "mixed"),
    ("bf16", 2, 4, [257, 1, 1, 64, 129], "zero"), ("f32", 2, 4, [257, 1, 64], "zero"),
]


@pytest.mark.parametrize("case", CHUNK_CASES, ids=[f"{c[0]}-{c[1]}x{c[2]}-{c[4]}-{sum(c[3])}" for c in CHUNK_CASES])
def test_chunked_rule_matches_recurrence(case, cuda, inl):
    import torch
    dtype, nk, nv, lens, gates = case
    print(f"case=gdn_chunked_rule {case}", flush=True)
    rng = np.random.default_rng(sum(lens))
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    n, dk = int(cu[-1]), 128
    mixed = og._r(rng.standard_normal((n, (2 * nk + nv) * dk)).astype(np.float32), dtype)
    u = rng.uniform(0, 1, (n, nv))
    g = {"small": -0.2 * u, "mixed": -np.where(u < 0.1, 30.0, 0.02 * u), "zero": 0 * u}[gates].astype(np.float32)
    beta = rng.uniform(0, 1, (n, nv)).astype(np.float32)
    got = inl.gdn_rule(_t(torch, mixed, cuda, _tdtype(torch, dtype)), cu.tolist(), nk, nv, dk, dk,
                       _t(torch, g, cuda, torch.float32), _t(torch, beta, cuda, torch.float32)).cpu().numpy()
    ref = og.rule_packed(mixed, cu, nk, nv, dk, dk, g.astype(np.float64), beta.astype(np.float64))
    err = np.abs(got - ref).max() / np.abs(ref).max()
    print(f"chunked rule: max error {err:.3g} of the largest value", flush=True)
    assert err <= 5e-6


# Gates that reset the state: e^g is 0 in f32 for all of these, whatever their
# size, at the first, an inner and the last token of a chunk (64 tokens in bf16,
# 32 in f32), twice in one chunk, and at a text's first token. What follows a
# reset depends on the small gates after it alone. The bound of the test above.
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("reset", [-200.0, -1e9, -1e12, -1e15, float(np.finfo(np.float32).min), -np.inf])
def test_chunked_rule_resets(reset, dtype, cuda, inl):
    import torch
    nk, nv, lens, dk = 1, 4, [150, 40, 97], 128
    rng = np.random.default_rng(9)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    n = int(cu[-1])
    mixed = og._r(rng.standard_normal((n, (2 * nk + nv) * dk)).astype(np.float32), dtype)
    g = (-0.05 * rng.uniform(0, 1, (n, nv))).astype(np.float32)
    g[[0, 31, 32, 63, 64, 80, 85, 127, 128, 150, 189, 190, 286], 0] = reset
    g[[20, 170, 200], 1] = reset
    g[149, 2] = reset   # head 3: none
    beta = rng.uniform(0, 1, (n, nv)).astype(np.float32)
    print(f"case=gdn_chunked_rule_resets {reset} {dtype}", flush=True)
    got = inl.gdn_rule(_t(torch, mixed, cuda, _tdtype(torch, dtype)), cu.tolist(), nk, nv, dk, dk,
                       _t(torch, g, cuda, torch.float32), _t(torch, beta, cuda, torch.float32)).cpu().numpy()
    ref = og.rule_packed(mixed, cu, nk, nv, dk, dk, g.astype(np.float64), beta.astype(np.float64))
    err = np.abs(got - ref).max(axis=(0, 2)) / np.abs(ref).max(axis=(0, 2))
    print(f"chunked rule: max error {err} of each head's largest value", flush=True)
    assert (err <= 5e-6).all()


# Values that the chunked form's products cannot take. Infinities and NaN reach
# what they reach in the recurrence (a value: its column from its token on; a
# key, gate or beta: all columns from its token on; a query: its token), earlier
# tokens and other texts not at all. Large finite values, gates above 0 and betas
# outside [0, 2] give the recurrence's results, within the bound above of the
# largest that a column's outputs, or a tenth of its values (what a query reads
# of the state: q . k / sqrt(dk)), have been so far.
_F32_MIN = float(np.finfo(np.float32).min)
ODD_CASES = [("v", np.nan), ("v", np.inf), ("v", _F32_MIN), ("v", 1e30), ("k", np.nan), ("k", -np.inf), ("k", 1e15),
             ("q", np.nan), ("q", np.inf), ("q", 1e15), ("g", np.nan), ("g", np.inf), ("g", 0.4), ("g", 2.0),
             ("beta", np.nan), ("beta", -np.inf), ("beta", 3.0), ("beta", -1.0)]


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("where,value", ODD_CASES)
def test_chunked_rule_odd_values(where, value, dtype, cuda, inl):
    import torch
    nk, nv, lens, dk = 1, 2, [150, 90, 70], 128
    rng = np.random.default_rng(10)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    n = int(cu[-1])
    mixed = rng.standard_normal((n, (2 * nk + nv) * dk)).astype(np.float32)
    g = (-0.05 * rng.uniform(0, 1, (n, nv))).astype(np.float32)
    beta = rng.uniform(0, 1, (n, nv)).astype(np.float32)
    col = {"q": 5, "k": dk + 5, "v": 2 * dk + 5}
    # inside a chunk, and the last token of two texts; text 2 has none (two lowest values would overflow the state)
    at = (17, 100, 149, 239) if value != _F32_MIN else (100, 239)
    for t in at:
        if where in col:
            mixed[t, col[where]] = value
        else:
            (g if where == "g" else beta)[t, 0] = value
    mixed = np.maximum(og._r(mixed, dtype), np.float32(_F32_MIN if dtype == "f32" else -3.3895e38))
    if value == -np.inf and where in col:
        mixed[at, col[where]] = value
    print(f"case=gdn_chunked_rule_odd {where}={value} {dtype}", flush=True)
    got = inl.gdn_rule(_t(torch, mixed, cuda, _tdtype(torch, dtype)), cu.tolist(), nk, nv, dk, dk,
                       _t(torch, g, cuda, torch.float32), _t(torch, beta, cuda, torch.float32)).cpu().numpy()
    with np.errstate(all="ignore"):
        ref = og.rule_packed(mixed, cu, nk, nv, dk, dk, g.astype(np.float64), beta.astype(np.float64))
    finite = np.isfinite(ref)
    assert (np.isfinite(got) == finite).all(), f"{(np.isfinite(got) != finite).sum()} values differ in being finite"
    ref, got = np.where(finite, ref, 0), np.where(finite, got, 0).astype(np.float64)
    v = np.abs(mixed[:, 2 * nk * dk:].reshape(n, nv, dk).astype(np.float64))
    size = np.maximum(np.abs(ref), 0.1 * np.where(np.isfinite(v), v, 0))
    for a, e in zip(cu[:-1], cu[1:]):
        held = np.maximum(np.maximum.accumulate(size[a:e], axis=0), 1.0)
        err = (np.abs(got[a:e] - ref[a:e]) / held).max()
        print(f"rows {a}-{e}: max error {err:.3g} of the largest value so far", flush=True)
        assert err <= 5e-6


# Positive gates: the state grows by e^0.2 a token, past the size up to which it
# enters products (10^20, after some 230 tokens). The bound of the test above.
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_chunked_rule_growing_state(dtype, cuda, inl):
    import torch
    n, dk = 330, 128
    rng = np.random.default_rng(11)
    mixed = og._r(rng.standard_normal((n, 3 * dk)).astype(np.float32), dtype)
    g = np.full((n, 1), 0.2, np.float32)
    beta = rng.uniform(0, 1, (n, 1)).astype(np.float32)
    print(f"case=gdn_chunked_rule_growing {dtype}", flush=True)
    got = inl.gdn_rule(_t(torch, mixed, cuda, _tdtype(torch, dtype)), [0, n], 1, 1, dk, dk,
                       _t(torch, g, cuda, torch.float32), _t(torch, beta, cuda, torch.float32)).cpu().numpy()
    ref = og.rule_packed(mixed, [0, n], 1, 1, dk, dk, g.astype(np.float64), beta.astype(np.float64))
    err = (np.abs(got - ref) / np.maximum(np.maximum.accumulate(np.abs(ref), axis=0), 1.0)).max()
    print(f"max error {err:.3g} of the largest value so far, largest {np.abs(ref).max():.3g}", flush=True)
    assert np.abs(ref).max() > 1e22 and err <= 5e-6


# Rows that start 8 (bf16) or 16 (f32) bytes past a multiple of 16 or 32, with
# NaN between them: the chunks load whole rows 16 bytes at a time. The bound of
# the test above.
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_chunked_rule_strided_rows(dtype, cuda, inl):
    import torch
    nk, nv, lens, dk = 1, 2, [63, 65, 7], 128
    rng = np.random.default_rng(5)
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    n, width = int(cu[-1]), (2 * nk + nv) * dk
    mixed = og._r(rng.standard_normal((n, width)).astype(np.float32), dtype)
    g = (-0.2 * rng.uniform(0, 1, (n, nv))).astype(np.float32)
    beta = rng.uniform(0, 1, (n, nv)).astype(np.float32)
    rows = torch.full((n, width + 12), float("nan"), dtype=_tdtype(torch, dtype), device=cuda)[:, 4:4 + width]
    rows.copy_(_t(torch, mixed, cuda, _tdtype(torch, dtype)))
    print(f"case=gdn_chunked_rule_strided {dtype}", flush=True)
    got = inl.gdn_rule(rows, cu.tolist(), nk, nv, dk, dk, _t(torch, g, cuda, torch.float32),
                       _t(torch, beta, cuda, torch.float32)).cpu().numpy()
    ref = og.rule_packed(mixed, cu, nk, nv, dk, dk, g.astype(np.float64), beta.astype(np.float64))
    assert np.abs(got - ref).max() / np.abs(ref).max() <= 5e-6
