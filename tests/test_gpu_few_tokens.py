"""GPU parity of the few-token GEMM (calls of at most 32 tokens) through the C ABI, at the sizes where
it can go wrong: every family, one to 32 tokens around its 16-token operand tiles, widths off its
16-row tiles, K around its units of 128 / 256 and its waves' K splits, rows too long for one tile's
LDS (two token tiles, then the tile GEMM), sizes whose rounds over the CUs leave it for the tile
GEMM, f32 inputs quantized in the kernel and by a launch of their own, code rows off dword boundaries,
groups of parts, outputs over the input, payloads that end at their last byte, the SwiGLU epilogue of
the prefill FFN, and a QuantAct scale whose products leave int64.

Tolerance: every 32-block (or super-block half) is one exact integer dot folded with at most four
f32 roundings, and the blocks' sums with one each, so an output is within (blocks + 8) * 2^-24 of the
sum of its terms' magnitudes; the min terms are summed apart from the dots, which at most doubles
that sum over sum|w * xhat| for these payloads.
"""
import numpy as np
import pytest

import oracle
from apeiron_amd import chart, synth

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

Q32 = 2.0 ** -32
Q5_0, Q8_0, Q2_K, Q3_K, Q4_K, Q6_K = 6, 8, 10, 11, 12, 14
ALL = [Q5_0, Q8_0, Q2_K, Q3_K, Q4_K, Q6_K]


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "GPU tests need the MI355X"
    d = chart.Device(0)
    yield d
    d.close()


def stream():
    return torch.cuda.current_stream().cuda_stream


def payload(t, rng, n_out, n_in):
    """Weights that average about zero, as trained ones do: no output is a near-cancellation."""
    return synth.q4_k_centered_payload(rng, n_out, n_in) if t == Q4_K else synth.payload(t, rng, n_out, n_in)


def close(t, raw, n_out, n_in, codes, scales, y, what):
    for c in range(codes.shape[0]):
        st, ref = oracle.matvec_q8act(t, raw, n_out, n_in, codes[c], scales[c])
        st2, absdot = oracle.row_absdot(t, raw, n_out, n_in, codes[c], scales[c])
        assert st == 0 and st2 == 0
        err = np.abs(y[c].astype(np.float64) - ref.astype(np.float64) * Q32)
        tol = 2 * (n_in / 32 + 8) * 2.0 ** -24 * absdot + Q32
        bad = np.nonzero(~(err <= tol))[0]
        assert bad.size == 0, f"{what} token {c}: rows {bad[:6]} err {err[bad[:6]]} tol {tol[bad[:6]]}"


@pytest.mark.parametrize("t", ALL)
@pytest.mark.parametrize("n_tok,n_out,n_in", [
    (1, 16, 32), (2, 17, 256), (8, 130, 300), (9, 48, 901), (16, 33, 1536), (17, 40, 1000), (32, 129, 520),
    (3, 20, 4864), (16, 18, 8960),   # waves of several units; two tiles of 8 tokens
    (2, 16, 32768),                  # the longest rows
])
def test_few_tokens_vs_oracle(dev, t, n_tok, n_out, n_in):
    rng = synth.rng_for(9, 1000 * t + n_in + n_tok)
    raw = payload(t, rng, n_out, n_in)
    x = synth.activations(rng, n_in, n_tok).reshape(n_tok, n_in)
    st, codes, scales = oracle.quant_act_f32_batch(x)
    assert st == 0
    # the weight in a buffer that ends with its payload
    dw = torch.from_numpy(raw).cuda()
    for w in (dev.upload(t, raw, n_out, n_in), dev.wrap(t, dw.data_ptr(), raw.nbytes, n_out, n_in)):
        y = torch.full((n_tok, n_out), float("nan"), device="cuda")
        dx = torch.from_numpy(x).cuda()
        w.gemm_f32_dev(dx.data_ptr(), n_tok, y.data_ptr(), stream())
        assert dev.sync_status(stream()) == 0
        close(t, raw, n_out, n_in, codes, scales, y.cpu().numpy(), "f32")
        # from codes, once at an odd address (rows off dword boundaries): the same outputs
        for off in (0, 1):
            dc = torch.zeros(n_tok * n_in + off, dtype=torch.int8, device="cuda")
            dc[off:] = torch.from_numpy(codes.reshape(-1)).cuda()
            ds = torch.from_numpy(scales).cuda()
            yq = torch.full((n_tok, n_out), float("nan"), device="cuda")
            w.gemm_q8_dev(dc.data_ptr() + off, ds.data_ptr(), n_tok, yq.data_ptr(), stream())
            assert dev.sync_status(stream()) == 0
            assert (yq == y).all(), (off, int((yq != y).sum()))
        w.free()


# The longest rows whose 16 (two tiles of 8) and 32 (two of 16) tokens fit a CU's LDS.
LDS_ROWS = {Q5_0: (14848, 7424), Q8_0: (13056, 6400), Q2_K: (12032, 5888), Q3_K: (14080, 6912), Q4_K: (12544, 6144), Q6_K: (11264, 5632)}


@pytest.mark.parametrize("t", ALL)
@pytest.mark.parametrize("n_tok", [16, 32])
def test_rows_at_the_lds_limit(dev, t, n_tok):
    """At the longest rows that fit the call runs on the few-token kernel, 256 columns further on the
    tile GEMM (the bits of the design that names it); both hold the oracle's bound."""
    n_out = 20
    for n_in, few in ((LDS_ROWS[t][n_tok > 16], True), (LDS_ROWS[t][n_tok > 16] + 256, False)):
        rng = synth.rng_for(16, n_in + t)
        raw = payload(t, rng, n_out, n_in)
        w = dev.upload(t, raw, n_out, n_in)
        x = synth.activations(rng, n_in, n_tok).reshape(n_tok, n_in)
        dx = torch.from_numpy(x).cuda()
        y, named = (torch.full((n_tok, n_out), float("nan"), device="cuda") for _ in range(2))
        w.gemm_f32_dev(dx.data_ptr(), n_tok, y.data_ptr(), stream())
        dev.set_gemm_design(t, 3 if t in (Q2_K, Q3_K) else 1)
        try:
            w.gemm_f32_dev(dx.data_ptr(), n_tok, named.data_ptr(), stream())
            assert dev.sync_status(stream()) == 0
        finally:
            dev.set_gemm_design(t, 0)
        assert torch.equal(y, named) != few, n_in
        st, codes, scales = oracle.quant_act_f32_batch(x)
        assert st == 0
        if few:
            close(t, raw, n_out, n_in, codes, scales, y.cpu().numpy(), f"K {n_in}")
        w.free()


GROUPS = {  # (type, n_out) of the parts
    "qkv": [(Q4_K, 1536), (Q4_K, 256), (Q6_K, 256)],
    "wide": [(Q4_K, 8960), (Q6_K, 300), (Q8_0, 0), (Q8_0, 64)],  # at 24 tokens its Q4_K part keeps the tile GEMM
    "six": [(Q8_0, 96), (Q8_0, 17), (Q8_0, 0), (Q8_0, 130), (Q8_0, 64), (Q8_0, 33), (Q8_0, 300)],  # two launches
    "types": [(Q3_K, 130), (Q5_0, 64), (Q2_K, 33), (Q3_K, 64), (Q6_K, 40)],
}


@pytest.mark.parametrize("group", sorted(GROUPS))
@pytest.mark.parametrize("n_tok", [9, 16, 24])
@pytest.mark.parametrize("src", ["f32", "codes"])
def test_grouped_parts_are_their_single_calls(dev, group, n_tok, src):
    """Parts of several types, an input quantized once for all of them, more parts of a type than a launch
    holds, parts without rows and parts of both routes: each is its single call's output bit for bit."""
    n_in = 1536
    rng = synth.rng_for(17, n_tok + len(group))
    ws = [dev.upload(t, payload(t, rng, o, n_in), o, n_in) for t, o in GROUPS[group]]
    dx = torch.from_numpy(synth.activations(rng, n_in, n_tok).reshape(n_tok, n_in)).cuda()
    dc = torch.zeros((n_tok, n_in), dtype=torch.int8, device="cuda")
    ds = torch.zeros((n_tok, n_in // 32), dtype=torch.int64, device="cuda")
    dev.quant_act_f32_dev(dx.data_ptr(), n_tok, n_in, dc.data_ptr(), ds.data_ptr(), stream())
    ys, y1 = ([torch.full((n_tok, max(w.n_out, 1)), float("nan"), device="cuda") for w in ws] for _ in range(2))
    if src == "f32":
        chart.gemm_group_f32_dev(dev, ws, dx.data_ptr(), n_tok, [y.data_ptr() for y in ys], stream())
    else:
        chart.gemm_group_q8_dev(dev, ws, dc.data_ptr(), ds.data_ptr(), n_tok, [y.data_ptr() for y in ys], stream())
    for w, y in zip(ws, y1):
        w.gemm_f32_dev(dx.data_ptr(), n_tok, y.data_ptr(), stream())
    assert dev.sync_status(stream()) == 0
    for w, y, one in zip(ws, ys, y1):
        if w.n_out:
            assert torch.isfinite(y).all() and torch.equal(y, one), (w.n_out, group)
        else:
            assert torch.isnan(y).all()
        w.free()


@pytest.mark.parametrize("gt,dt,n_embd,n_ff,n_tok", [
    (Q4_K, Q6_K, 1536, 333, 8), (Q8_0, Q8_0, 256, 300, 1), (Q6_K, Q5_0, 512, 1000, 17), (Q5_0, Q2_K, 96, 64, 5),
    (Q3_K, Q3_K, 901, 130, 16), (Q2_K, Q4_K, 1536, 96, 31),
    (Q4_K, Q4_K, 300, 4200, 19), (Q8_0, Q4_K, 2048, 100, 6),  # (the last: six K splits, two passes)
])
def test_few_tokens_ffn(dev, gt, dt, n_embd, n_ff, n_tok):
    """The SwiGLU epilogue: gate / up equal the projections' own calls, the hidden QuantAct is the
    oracle's of those values, and down is the projection of it."""
    rng = synth.rng_for(10, gt * 100 + n_ff)
    raws = [payload(t, rng, o, i) for t, o, i in ((gt, n_ff, n_embd), (gt, n_ff, n_embd), (dt, n_embd, n_ff))]
    G, U, D = (dev.upload(t, r, o, i) for r, (t, o, i) in zip(raws, ((gt, n_ff, n_embd), (gt, n_ff, n_embd), (dt, n_embd, n_ff))))
    x = (synth.activations(rng, n_embd, n_tok).reshape(n_tok, n_embd) * np.float32(2.0 ** -6))
    dx = torch.from_numpy(x).cuda()
    gy, uy, g1, u1 = (torch.full((n_tok, n_ff), float("nan"), device="cuda") for _ in range(4))
    hc = torch.zeros((n_tok, n_ff), dtype=torch.int8, device="cuda")
    hs = torch.zeros((n_tok, -(-n_ff // 32)), dtype=torch.int64, device="cuda")
    chart.ffn_gate_up_prefill_dev(dev, G, U, dx.data_ptr(), n_tok, hc.data_ptr(), hs.data_ptr(), gy.data_ptr(), uy.data_ptr(), stream())
    chart.gemm_group_f32_dev(dev, [G, U], dx.data_ptr(), n_tok, [g1.data_ptr(), u1.data_ptr()], stream())
    assert dev.sync_status(stream()) == 0
    assert (gy == g1).all() and (uy == u1).all()
    st, codes, scales = oracle.quant_act_f32_batch(x)
    close(gt, raws[0], n_ff, n_embd, codes, scales, gy.cpu().numpy(), "gate")
    HC, HS, g, u = hc.cpu().numpy(), hs.cpu().numpy(), gy.cpu().numpy(), uy.cpu().numpy()
    for t in range(n_tok):
        st, c, s, _ = oracle.swiglu_quant_f32(g[t], u[t])
        assert st == 0 and (HC[t] == c).all() and (HS[t] == s).all(), t
    y = torch.full((n_tok, n_embd), float("nan"), device="cuda")
    hc2, hs2 = torch.zeros_like(hc), torch.zeros_like(hs)
    chart.ffn_prefill_dev(dev, G, U, D, dx.data_ptr(), n_tok, y.data_ptr(), hc2.data_ptr(), hs2.data_ptr(), stream())
    assert dev.sync_status(stream()) == 0
    assert (hc2 == hc).all() and (hs2 == hs).all()
    close(dt, raws[2], n_embd, n_ff, HC, HS, y.cpu().numpy(), "down")
    for w in (G, U, D):
        w.free()


@pytest.mark.parametrize("t", ALL)
@pytest.mark.parametrize("n_tok", [17, 25, 32])
def test_one_token_tile_of_32_and_two_of_16_agree(dev, t, n_tok):
    """Past 16 tokens the tokens of a workgroup follow the run's size: the parts alone take two tiles of
    16, side by side in a group they fill the CUs and take one of 32.  The same bits, and the oracle's."""
    n_in, n_out = 520, 4200
    rng = synth.rng_for(12, 100 * t + n_tok)
    raws = [payload(t, rng, n_out, n_in) for _ in range(4)]
    ws = [dev.upload(t, raw, n_out, n_in) for raw in raws]
    x = synth.activations(rng, n_in, n_tok).reshape(n_tok, n_in)
    st, codes, scales = oracle.quant_act_f32_batch(x)
    assert st == 0
    dx = torch.from_numpy(x).cuda()
    ys, y1 = ([torch.full((n_tok, n_out), float("nan"), device="cuda") for _ in ws] for _ in range(2))
    chart.gemm_group_f32_dev(dev, ws, dx.data_ptr(), n_tok, [y.data_ptr() for y in ys], stream())
    for w, y in zip(ws, y1):
        w.gemm_f32_dev(dx.data_ptr(), n_tok, y.data_ptr(), stream())
    assert dev.sync_status(stream()) == 0
    for w, y, one in zip(ws, ys, y1):
        assert torch.equal(y, one)
        w.free()
    close(t, raws[0], n_out, n_in, codes, scales, ys[0].cpu().numpy(), "group")


@pytest.mark.parametrize("n_in", [256, 8960])
def test_few_tokens_refusals(dev, n_in):
    """Input refusals recorded by the in-kernel quantizer, the separate one (the longer rows) and the
    codes' own check, each the contract's first."""
    n_tok, n_out = 9, 32
    rng = synth.rng_for(11, n_in)
    raw = payload(Q4_K, rng, n_out, n_in)
    w = dev.upload(Q4_K, raw, n_out, n_in)
    y = torch.zeros((n_tok, n_out), device="cuda")
    x = synth.activations(rng, n_in, n_tok).reshape(n_tok, n_in)
    st, codes, scales = oracle.quant_act_f32_batch(x)
    x[7, 3], x[5, n_in - 1] = np.float32("nan"), np.float32(2.0 ** 40)
    w.gemm_f32_dev(torch.from_numpy(x).cuda().data_ptr(), n_tok, y.data_ptr(), stream())
    assert dev.sync_status(stream()) == 11  # token 5's range before token 7's NaN
    scales[6, -1] = 1 << 62
    codes[6, n_in - 32:] = 5
    w.gemm_q8_dev(torch.from_numpy(codes).cuda().data_ptr(), torch.from_numpy(scales).cuda().data_ptr(), n_tok, y.data_ptr(), stream())
    assert dev.sync_status(stream()) == 7
    w.free()


@pytest.mark.parametrize("t", [Q8_0, Q4_K, Q2_K])  # (no code sums, a block's, a 16-group's)
@pytest.mark.parametrize("n_in", [1, 15, 18, 31, 901, 1538, 4863])
def test_few_tokens_code_rows_at_any_byte(dev, t, n_in):
    """Code rows at every offset from the dword grid, other bytes around them, row ends inside and on a
    16-code chunk: the f32 call's outputs, whose codes these are, bit for bit."""
    n_out = 20
    rng = synth.rng_for(13, 10 * n_in + t)
    w = dev.upload(t, payload(t, rng, n_out, n_in), n_out, n_in)
    for n_tok in (1, 3, 17):
        dx = torch.from_numpy(synth.activations(rng, n_in, n_tok).reshape(n_tok, n_in)).cuda()
        ds = torch.zeros((n_tok, -(-n_in // 32)), dtype=torch.int64, device="cuda")
        y = torch.full((n_tok, n_out), float("nan"), device="cuda")
        w.gemm_f32_dev(dx.data_ptr(), n_tok, y.data_ptr(), stream())
        for off in range(4):
            dc = torch.full((off + n_tok * n_in + 7,), 77, dtype=torch.int8, device="cuda")
            dev.quant_act_f32_dev(dx.data_ptr(), n_tok, n_in, dc.data_ptr() + off, ds.data_ptr(), stream())
            yq = torch.full((n_tok, n_out), float("nan"), device="cuda")
            w.gemm_q8_dev(dc.data_ptr() + off, ds.data_ptr(), n_tok, yq.data_ptr(), stream())
            assert dev.sync_status(stream()) == 0
            assert torch.equal(yq, y), (n_tok, off)
    w.free()


@pytest.mark.parametrize("t,n_out,n_in,n_tok,route", [
    (Q4_K, 1536, 8960, 12, "few"), (Q4_K, 2560, 8960, 12, "tile"), (Q4_K, 4864, 6144, 12, "tile"), (Q4_K, 4864, 6144, 4, "few"),
    (Q2_K, 4200, 8960, 12, "tile"), (Q3_K, 4200, 4864, 24, "tile"), (Q3_K, 4200, 4864, 12, "few"), (Q8_0, 4400, 8960, 12, "tile"),
    (Q8_0, 4400, 8960, 8, "few"), (Q6_K, 9000, 4864, 24, "tile"), (Q6_K, 9000, 4864, 12, "few"), (Q5_0, 9000, 4864, 32, "tile"),
])
def test_wide_calls_keep_the_tile_gemm(dev, t, n_out, n_in, n_tok, route):
    """Where the few-token kernel's rounds over the CUs take longer than the tile GEMM, AUTO is the tile
    GEMM, from f32 and from codes: the outputs of the design that names it, bit for bit."""
    rng = synth.rng_for(14, n_out + n_in + t)
    w = dev.upload(t, payload(t, rng, n_out, n_in), n_out, n_in)
    dx = torch.from_numpy(synth.activations(rng, n_in, n_tok).reshape(n_tok, n_in)).cuda()
    dc = torch.zeros((n_tok, n_in), dtype=torch.int8, device="cuda")
    ds = torch.zeros((n_tok, n_in // 32), dtype=torch.int64, device="cuda")
    dev.quant_act_f32_dev(dx.data_ptr(), n_tok, n_in, dc.data_ptr(), ds.data_ptr(), stream())
    y, yq, named = (torch.full((n_tok, n_out), float("nan"), device="cuda") for _ in range(3))
    w.gemm_f32_dev(dx.data_ptr(), n_tok, y.data_ptr(), stream())
    w.gemm_q8_dev(dc.data_ptr(), ds.data_ptr(), n_tok, yq.data_ptr(), stream())
    dev.set_gemm_design(t, 3 if t in (Q2_K, Q3_K) else 1)
    try:
        w.gemm_f32_dev(dx.data_ptr(), n_tok, named.data_ptr(), stream())
        assert dev.sync_status(stream()) == 0
    finally:
        dev.set_gemm_design(t, 0)
    assert torch.equal(y, yq)
    assert torch.equal(y, named) == (route == "tile")
    w.free()


@pytest.mark.parametrize("t", ALL)
def test_outputs_over_the_input(dev, t):
    """An output that lies over the call's input: the input is read whole before anything is written, so
    the call gives what it gives with separate buffers on the tile GEMM."""
    n, n_tok, n_ff = 512, 9, 512
    rng = synth.rng_for(15, t)
    W = [dev.upload(t, payload(t, rng, n, n), n, n) for _ in range(3)]
    x = torch.from_numpy(synth.activations(rng, n, n_tok).reshape(n_tok, n)).cuda() * 2.0 ** -4
    codes, scales = torch.zeros((n_tok, n), dtype=torch.int8, device="cuda"), torch.zeros((n_tok, n // 32), dtype=torch.int64, device="cuda")
    dev.quant_act_f32_dev(x.data_ptr(), n_tok, n, codes.data_ptr(), scales.data_ptr(), stream())
    new = lambda: torch.full((n_tok, n), float("nan"), device="cuda")  # noqa: E731
    # one projection, then three of which the second's output is the input
    ref = [new() for _ in W]
    dev.set_gemm_design(t, 3 if t in (Q2_K, Q3_K) else 1)
    try:
        for w, y in zip(W, ref):
            w.gemm_f32_dev(x.data_ptr(), n_tok, y.data_ptr(), stream())
        assert dev.sync_status(stream()) == 0
    finally:
        dev.set_gemm_design(t, 0)
    y = x.clone()
    W[0].gemm_f32_dev(y.data_ptr(), n_tok, y.data_ptr(), stream())
    assert dev.sync_status(stream()) == 0 and torch.equal(y, ref[0])
    y0, y1, y2 = new(), x.clone(), new()
    chart.gemm_group_f32_dev(dev, W, y1.data_ptr(), n_tok, [q.data_ptr() for q in (y0, y1, y2)], stream())
    assert dev.sync_status(stream()) == 0
    assert all(torch.equal(q, r) for q, r in zip((y0, y1, y2), ref))
    # from codes inside the output's buffer
    y = new()
    held = y.view(torch.int8).reshape(-1)[:n_tok * n]
    held.copy_(codes.reshape(-1))
    W[0].gemm_q8_dev(held.data_ptr(), scales.data_ptr(), n_tok, y.data_ptr(), stream())
    assert dev.sync_status(stream()) == 0 and torch.equal(y, ref[0])
    # the FFN's hidden codes over its input, f32 and codes
    hc, hs = torch.zeros((n_tok, n_ff), dtype=torch.int8, device="cuda"), torch.zeros((n_tok, n_ff // 32), dtype=torch.int64, device="cuda")
    chart.ffn_gate_up_prefill_dev(dev, W[0], W[1], x.data_ptr(), n_tok, hc.data_ptr(), hs.data_ptr(), stream=stream())
    out, held, hs2 = new(), x.clone(), torch.zeros_like(hs)
    chart.ffn_gate_up_prefill_dev(dev, W[0], W[1], held.data_ptr(), n_tok, held.data_ptr(), hs2.data_ptr(), stream=stream())
    assert dev.sync_status(stream()) == 0
    assert torch.equal(held.view(torch.int8).reshape(-1)[:n_tok * n_ff], hc.reshape(-1)) and torch.equal(hs2, hs)
    c2, s2 = codes.clone(), scales.clone()
    chart.ffn_prefill_q8_dev(dev, W[0], W[1], W[2], c2.data_ptr(), s2.data_ptr(), n_tok, out.data_ptr(), c2.data_ptr(), s2.data_ptr(), stream())
    assert dev.sync_status(stream()) == 0
    assert torch.equal(c2, hc) and torch.equal(s2, hs)
    for w in W:
        w.free()
