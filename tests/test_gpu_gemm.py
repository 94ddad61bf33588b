"""GPU parity of the grouped GEMMs and the fused routed layer.

Tolerance: normwise max relative error
    rel = max|gpu - oracle| / max|oracle|
<= 1e-2 for the bf16 profile and <= 2e-2 for the a4w4 profile. Stage tests
feed the GPU kernel and the oracle the *same* quantised operands, so the only
difference is fp32 summation order and the bf16 roundings that follow it; they
must also meet a per-element bar (``_parity``). a4w4: the down GEMM bit for
bit (every product and partial sum is exact), h within one bf16 ulp (the
kernel's expf and numpy's exp may round apart). bf16 profile (E4M3 x E2M1 MFMA): each down
output within one bf16 ulp plus 2^-10 of its sum of absolute products (the
MFMA drops products far below the largest of their group), the gate/up
GEMM's h within one ulp plus that bound carried through SwiGLU from its gate
and up values. The end-to-end tests start from the same bf16 x and routing:
a4w4 bit for bit; bf16 per element within 3e-2 of max(|ref|, rms(ref)).
"""

import numpy as np
import pytest
import torch

from oracle import mxfp4 as Q
from oracle import moe as M
from _parity import check_bound, elementwise_rel, gemm_bound, swiglu_bound
from dsv4_hip import (ops, synth, AFMT_BF16, AFMT_E2M1, AFMT_E4M3, PROFILE_A4W4, PROFILE_BF16, PROFILE_BF16_PURE,
                      RULE_OCP_FLOOR, RULE_CEIL_DIV6)

pytestmark = pytest.mark.gpu

TOL = {"bf16": 1e-2, "a4w4": 2e-2, "bf16_pure": 1e-2}
# per-element relative error with a floor of rms(output) (_parity.elementwise_rel); a4w4: bit for bit;
# the pure-bf16 variant has no quantisation step for a 1-ulp difference to move
ELEM_TOL = {"bf16": 3e-2, "a4w4": 0.0, "bf16_pure": 2e-2}


def rel(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-30))


def _bits(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def _dev_bf16(bits, dev):
    return torch.from_numpy(np.ascontiguousarray(bits, np.uint16).view(np.int16)).view(torch.bfloat16).to(dev)


def _dev(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


def make_layer(E, D, I, experts_needed, dev):
    host = {e: synth.expert_weights(int(e), D, I) for e in experts_needed}
    devw = {e: {k: _dev(v, dev) for k, v in d.items()} for e, d in host.items()}
    return host, devw, ops.expert_table(devw, E, dev)


# rows of an expert around the edges of 64-row blocks, of the large tile's 128-row halves and their
# 32-row wave tiles, of 256-row blocks and of the layer's 64- and 128-row thresholds
EDGE_COUNTS = (1, 63, 64, 65, 127, 128, 129, 191, 192, 193, 255, 256, 257, 320)


def _edge_ids(T, K, seed):
    """ids [T, K] over 16 experts: expert 1 + i has exactly EDGE_COUNTS[i] rows, expert 0 the others."""
    flat = np.zeros(T * K, np.int64)
    at = np.random.default_rng(seed).permutation(T * K)
    o = 0
    for i, c in enumerate(EDGE_COUNTS):
        flat[at[o:o + c]] = i + 1
        o += c
    return flat.reshape(T, K)


def _case(T, K, E, D, I, seed, dev, ids=None):
    if ids is None:
        ids = synth.zipf_topk(T, K, E, synth.rank_permutation(E, 3), np.random.default_rng(seed))
    w = synth.routing_weights(T, K, seed + 1)
    x = synth.bf16_normal(np.random.default_rng(seed + 2), (T, D))
    xb = x.view(torch.int16).numpy().view(np.uint16)
    host, devw, table = make_layer(E, D, I, np.unique(ids), dev)
    return ids, w, xb, host, devw, table


@pytest.mark.parametrize("profile", ["bf16", "a4w4"])
@pytest.mark.parametrize("T,K,E,D,I,bm", [(24, 4, 16, 1024, 512, 16), (200, 8, 16, 512, 512, 16),
                                          (8, 8, 256, 4096, 2048, 16), (200, 8, 16, 512, 512, 64),
                                          (200, 8, 16, 1024, 512, 128), (300, 6, 24, 2048, 1024, 64),
                                          (200, 8, 16, 1024, 1024, 256), (300, 6, 24, 2048, 1024, 256),
                                          (640, 8, 8, 4096, 2048, 256)])
def test_grouped_gemm_stages(gpu, profile, T, K, E, D, I, bm):
    # bm 16 runs the single-wave decode kernel, 64/128 the LDS-tiled kernel, 256 the
    # large-tile kernel (32x32x64 MFMA) in workgroups of half a block each
    _stage_case(gpu, profile, T, K, E, D, I, bm)


@pytest.mark.parametrize("profile", ["bf16", "a4w4"])
@pytest.mark.parametrize("bm", [16, 64, 128, 256])
def test_grouped_gemm_stages_row_counts(gpu, profile, bm):
    # every element of both stages, the a4w4 down GEMM bit for bit; with 256-row blocks the
    # counts leave second halves without a row (they exit) and waves without one (loads and
    # barriers only)
    _stage_case(gpu, profile, 600, 4, 16, 1024, 1024, bm, _edge_ids(600, 4, bm))


def test_grouped_gemm_stages_many_blocks_a4w4(gpu):
    # 32,768 routed rows: more large-tile workgroups than the CUs hold at once
    _stage_case(gpu, "a4w4", 4096, 8, 16, 1024, 1024, 256)


def _stage_case(gpu, profile, T, K, E, D, I, bm, ids=None):
    ids, w, xb, host, devw, table = _case(T, K, E, D, I, 31 + T, gpu, ids)
    al = ops.moe_align(_dev(ids, gpu), _dev(w, gpu), E, bm)
    R = T * K
    if profile == "bf16":
        rt, codes, s, k = Q.act_quant(xb, 128)
        a_f = Q.bf16_bits_to_f32(rt)
        a = _dev(codes, gpu)
        a_s = _dev(np.repeat((k + 127).astype(np.uint8), 4, axis=-1), gpu)
        afmt = AFMT_E4M3
    else:
        _, packed, sc = Q.ocp_mx_quant(xb, 32)
        a_f = Q.fp4_codes_to_f32(packed, sc)
        a, a_s, afmt = _dev(packed, gpu), _dev(sc, gpu), AFMT_E2M1
    h = ops.gemm_gateup(afmt, a, a_s, K, al, table, D, I, _dev(w.reshape(-1), gpu), 10.0)
    torch.cuda.synchronize()
    # oracle gate/up + SwiGLU for each flat row on the same quantised x
    flat_e = ids.reshape(-1)
    h_ref = np.zeros((R, I), np.float32)
    g_all, u_all = np.zeros((R, I), np.float32), np.zeros((R, I), np.float32)
    g_abs, u_abs = np.zeros((R, I), np.float32), np.zeros((R, I), np.float32)
    for e in np.unique(flat_e):
        rows = np.nonzero(flat_e == e)[0]
        w1 = Q.dequant_fp4_weight_f32(host[e]["w1p"], host[e]["w1s"])
        w3 = Q.dequant_fp4_weight_f32(host[e]["w3p"], host[e]["w3s"])
        xa = a_f[rows // K]
        g = Q.f32_to_bf16_f32(M.matmul_nt(xa, w1))
        u = Q.f32_to_bf16_f32(M.matmul_nt(xa, w3))
        g_all[rows], u_all[rows] = g, u
        g_abs[rows], u_abs[rows] = M.matmul_nt(np.abs(xa), np.abs(w1)), M.matmul_nt(np.abs(xa), np.abs(w3))
        h_ref[rows] = M.swiglu(g, u, w.reshape(-1)[rows], 10.0)
    h_gpu = Q.bf16_bits_to_f32(_bits(h))
    h_want = Q.f32_to_bf16_f32(h_ref)
    print(f"gate/up {profile} T={T} bm={bm}: normwise rel {rel(h_gpu, h_want):.3e}")
    assert rel(h_gpu, h_want) <= TOL[profile]
    # a4w4: g and u are exact; h may still flip one ulp where the kernel's expf and
    # numpy's exp round differently, so both profiles take the SwiGLU bound
    check_bound(h_gpu, h_want, swiglu_bound(g_all, u_all, w.reshape(-1), 10.0, h_want,
                                            g_abs if profile == "bf16" else None,
                                            u_abs if profile == "bf16" else None),
                f"gate/up {profile} bm={bm}")
    # down GEMM on the oracle's quantised h
    hb = Q.f32_to_bf16_bits(h_ref)
    if profile == "bf16":
        hrt, hc, hs, hk = Q.act_quant(hb, 128)
        ha_f = Q.bf16_bits_to_f32(hrt)
        ha, has = _dev(hc, gpu), _dev(np.repeat((hk + 127).astype(np.uint8), 4, axis=-1), gpu)
    else:
        _, hp, hsc = Q.ocp_mx_quant(hb, 32)
        ha_f = Q.fp4_codes_to_f32(hp, hsc)
        ha, has = _dev(hp, gpu), _dev(hsc, gpu)
    out = ops.gemm_down(afmt, ha, has, al, table, I, D)
    torch.cuda.synchronize()
    out_ref = np.zeros((R, D), np.float32)
    out_abs = np.zeros((R, D), np.float32)
    for e in np.unique(flat_e):
        rows = np.nonzero(flat_e == e)[0]
        w2 = Q.dequant_fp4_weight_f32(host[e]["w2p"], host[e]["w2s"])
        out_ref[rows] = M.matmul_nt(ha_f[rows], w2)
        out_abs[rows] = M.matmul_nt(np.abs(ha_f[rows]), np.abs(w2))
    out_gpu, out_want = Q.bf16_bits_to_f32(_bits(out)), Q.f32_to_bf16_f32(out_ref)
    print(f"down {profile} T={T} bm={bm}: normwise rel {rel(out_gpu, out_want):.3e}")
    assert rel(out_gpu, out_want) <= TOL[profile]
    if profile == "a4w4":
        assert np.array_equal(out_gpu, out_want), "a4w4 down: not bit-exact"
    else:
        check_bound(out_gpu, out_want, gemm_bound(out_want, out_abs), f"down {profile} bm={bm}")


@pytest.mark.parametrize("afmt,bm", [(AFMT_E4M3, 16), (AFMT_E4M3, 64), (AFMT_E4M3, 128), (AFMT_E4M3, 256),
                                     (AFMT_E2M1, 16), (AFMT_E2M1, 64), (AFMT_E2M1, 128), (AFMT_E2M1, 256),
                                     (AFMT_BF16, 16), (AFMT_BF16, 64), (AFMT_BF16, 256)])
@pytest.mark.parametrize("shift", [1, 3, 4])
def test_grouped_gemm_outputs_need_element_alignment_only(gpu, afmt, bm, shift):
    """h_out and out `shift` elements past an aligned address (2, 6 and 8 bytes): the same bits as
    aligned ones, and nothing written around them. (out of 256-row blocks must be 16-byte aligned.)"""
    T, K, E, D, I = 37, 4, 4, 1024, 1024
    ids, w, xb, host, devw, table = _case(T, K, E, D, I, 5, gpu)
    al = ops.moe_align(_dev(ids, gpu), _dev(w, gpu), E, bm)
    g = torch.Generator(device=gpu).manual_seed(bm)

    def operand(rows, cols):
        if afmt == AFMT_BF16:
            return torch.randn(rows, cols, generator=g, device=gpu).to(torch.bfloat16), None
        a = torch.randn(rows, cols, generator=g, device=gpu).to(torch.bfloat16)
        if afmt == AFMT_E2M1:
            packed, scale, _ = ops.mxfp4_act_quant(a, RULE_OCP_FLOOR)
            return packed, scale
        q = ops.fp8_act_quant(a, 128, want_codes=True, want_e8m0x4=True)
        return q["codes"], q["e8m0x4"]

    def shifted(rows, cols):
        buf = torch.full((rows * cols + 16,), 7.0, dtype=torch.bfloat16, device=gpu)
        return buf, buf[shift:shift + rows * cols].view(rows, cols)

    a, a_s = operand(T, D)
    wf = _dev(w.reshape(-1), gpu)
    want = ops.gemm_gateup(afmt, a, a_s, K, al, table, D, I, wf, 10.0)
    buf, h = shifted(T * K, I)
    ops.gemm_gateup(afmt, a, a_s, K, al, table, D, I, wf, 10.0, out=h)
    torch.cuda.synchronize()
    assert torch.equal(h.view(torch.int16), want.view(torch.int16))
    assert (buf[:shift] == 7.0).all() and (buf[shift + h.numel():] == 7.0).all()
    a, a_s = operand(T * K, I)
    want = ops.gemm_down(afmt, a, a_s, al, table, I, D)
    buf, out = shifted(T * K, D)
    if bm == 256:
        with pytest.raises(ops._lib.Dsv4Error, match="16-byte aligned output"):
            ops.gemm_down(afmt, a, a_s, al, table, I, D, out=out)
        return
    ops.gemm_down(afmt, a, a_s, al, table, I, D, out=out)
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
    assert (buf[:shift] == 7.0).all() and (buf[shift + out.numel():] == 7.0).all()


@pytest.mark.parametrize("profile,rule", [("a4w4", RULE_OCP_FLOOR), ("a4w4", RULE_CEIL_DIV6),
                                          ("bf16", RULE_OCP_FLOOR), ("bf16_pure", RULE_OCP_FLOOR)])
def test_nan_rows_agree_between_kernels(gpu, profile, rule):
    """Weight scale bytes of 255 and no clamps: h and column 5 of the outputs hold NaN. Eight tokens'
    rows on an expert in 64-row blocks and the same rows on one in 256-row blocks (same weights) give
    the same h bits, and the same layer outputs: a4w4 bit for bit (its sums are exact), bf16 within
    the summation order of the E4M3 products (rel 1e-2, as the parity tests), pure bf16 NaN alike."""
    T, K, E, D, I, n = 8192 if profile == "bf16_pure" else 2048, 8, 16, 1024, 1024, 8
    host = synth.expert_weights(3, D, I)
    for row, block in ((0, 1), (37, 0), (I - 1, D // 32 - 1)):
        host["w1s"][row, block] = 255
    host["w3s"][100, 2] = 255
    host["w2s"][5, 3] = 255
    dev = {k: _dev(v, gpu) for k, v in host.items()}
    table = ops.expert_table({e: dev for e in range(E)}, E, gpu)
    ids = torch.zeros((T, K), dtype=torch.int32, device=gpu)      # expert 0: every row but
    ids[:n] = 15                                                  # the first n tokens' (64 rows)
    x = torch.randn(T, D, generator=torch.Generator(device=gpu).manual_seed(2), device=gpu).to(torch.bfloat16)
    x[n:2 * n] = x[:n]
    w = torch.rand(T, K, generator=torch.Generator(device=gpu).manual_seed(3), device=gpu)
    w[n:2 * n] = w[:n]

    def operand(v):
        if profile == "a4w4":
            return AFMT_E2M1, *ops.mxfp4_act_quant(v, rule)[:2]
        if profile == "bf16_pure":
            return AFMT_BF16, v, None
        q = ops.fp8_act_quant(v, 128, want_codes=True, want_e8m0x4=True)
        return AFMT_E4M3, q["codes"], q["e8m0x4"]

    al = {bm: ops.moe_align(ids, w, E, bm) for bm in (16, 64, 256)}
    afmt, a, a_s = operand(x)
    h = {bm: ops.gemm_gateup(afmt, a, a_s, K, al[bm], table, D, I, w.view(-1), 0.0) for bm in al}
    afmt, a, a_s = operand(x.repeat_interleave(K, 0)[:, :I].contiguous())
    out = {bm: ops.gemm_down(afmt, a, a_s, al[bm], table, I, D) for bm in al}
    y = ops.LayerRunner(gpu, E, D, I).forward(
        x, ids, w, table, profile={"bf16": PROFILE_BF16, "a4w4": PROFILE_A4W4, "bf16_pure": PROFILE_BF16_PURE}[profile],
        rule=rule, swiglu_limit=0.0)
    torch.cuda.synchronize()
    for bm in h:
        nan = torch.isnan(h[bm])
        assert nan[:, [0, 37, I - 1, 100]].all() and int(nan.sum()) == 4 * T * K
        assert (h[bm][nan].view(torch.int16) == 0x7fc0).all(), bm
        assert torch.isnan(out[bm][:, 5]).all() and int(torch.isnan(out[bm]).sum()) == T * K, bm
    y = y.float()
    assert torch.isnan(y[:, 5]).all()
    y = torch.cat((y[:, :5], y[:, 6:]), 1)
    if profile == "a4w4":
        assert torch.isfinite(y).all() and torch.equal(y[:n], y[n:2 * n])
    elif profile == "bf16":
        assert torch.isfinite(y).all() and (y[:n] - y[n:2 * n]).abs().max() <= 1e-2 * y[:n].abs().max()
    else:
        assert torch.isnan(y[:2 * n]).all()


def test_grouped_gemm_empty_group_pattern(gpu):
    # _bench_gmm.py:8-22: groups [2, 0, 3] -> expert 1 receives no rows
    E, D, I, K = 3, 512, 512, 1
    ids = np.array([[0], [0], [2], [2], [2]], np.int64)
    w = np.ones((5, 1), np.float32)
    xb = synth.bf16_normal(np.random.default_rng(0), (5, D)).view(torch.int16).numpy().view(np.uint16)
    host, devw, table = make_layer(E, D, I, [0, 2], gpu)
    al = ops.moe_align(_dev(ids, gpu), _dev(w, gpu), E, 16)
    rt, codes, s, k = Q.act_quant(xb, 128)
    h = ops.gemm_gateup(AFMT_E4M3, _dev(codes, gpu), _dev(np.repeat((k + 127).astype(np.uint8), 4, -1), gpu), K,
                        al, table, D, I, _dev(w.reshape(-1), gpu), 10.0)
    torch.cuda.synchronize()
    a_f = Q.bf16_bits_to_f32(rt)
    for e, rows in ((0, [0, 1]), (2, [2, 3, 4])):
        w1 = Q.dequant_fp4_weight_f32(host[e]["w1p"], host[e]["w1s"])
        w3 = Q.dequant_fp4_weight_f32(host[e]["w3p"], host[e]["w3s"])
        g = Q.f32_to_bf16_f32(M.matmul_nt(a_f[rows], w1))
        u = Q.f32_to_bf16_f32(M.matmul_nt(a_f[rows], w3))
        ref = M.swiglu(g, u, np.ones(len(rows), np.float32), 10.0)
        assert rel(Q.bf16_bits_to_f32(_bits(h))[rows], ref) <= 1e-2


@pytest.mark.parametrize("profile", ["bf16", "a4w4", "bf16_pure"])
@pytest.mark.parametrize("T,K,E,D,I", [(8, 8, 256, 4096, 2048), (64, 6, 32, 1024, 512), (100, 6, 32, 1024, 512),
                                       (256, 8, 32, 2048, 1024), (400, 8, 256, 1024, 512)])
def test_layer_forward_vs_oracle(gpu, profile, T, K, E, D, I):
    # 16-row blocks up to 2047 routed rows (h quantised in the gate/up epilogue for a4w4,
    # by a separate launch for FP8); 256 tokens x top-8 = 2048 routed rows: 64-row M blocks
    # (tiled kernel, h quantised in the epilogue in both profiles); 3200 routed rows: the
    # chunked two-launch align. The pure-bf16 variant takes the same block sizes (no h
    # quantisation: its down GEMM reads bf16 h).
    ids, w, xb, host, devw, table = _case(T, K, E, D, I, 77 + T, gpu)
    runner = ops.LayerRunner(gpu, E, D, I)
    x = _dev_bf16(xb, gpu)
    prof = {"bf16": PROFILE_BF16, "a4w4": PROFILE_A4W4, "bf16_pure": PROFILE_BF16_PURE}[profile]
    y = runner.forward(x, _dev(ids, gpu), _dev(w, gpu), table, profile=prof, rule=RULE_OCP_FLOOR)
    torch.cuda.synchronize()
    if profile == "bf16":
        ref = M.routed_bf16(xb, ids, w, host, n_experts=E)
    elif profile == "bf16_pure":
        ref = M.routed_bf16(xb, ids, w, host, n_experts=E, fp8_act=False)
    else:
        ref = M.routed_a4w4(xb, ids, w, host, n_experts=E, rule="ocp_floor")
    got = Q.bf16_bits_to_f32(_bits(y))
    want = Q.bf16_bits_to_f32(ref["y"])
    er = elementwise_rel(got, want)
    print(f"layer {profile} T={T} K={K} E={E} D={D} I={I}: normwise rel {rel(got, want):.3e}, "
          f"elementwise rel {er:.3e}")
    assert rel(got, want) <= TOL[profile], rel(got, want)
    assert er <= ELEM_TOL[profile], er
    if profile == "a4w4":
        assert np.array_equal(_bits(y), ref["y"])


def _largest_products(ref, host, n):
    """[n, D]: for each output of the oracle's layer, the sum over the token's rows of max_j |h_j w2_j|."""
    al = ref["align"]
    h = np.abs(Q.bf16_bits_to_f32(ref["hq"]))
    out = np.zeros((n, next(iter(host.values()))["w2p"].shape[0]))
    w2 = {}
    for r, (e, tok) in enumerate(zip(al["s_e"], al["row"])):
        if e not in w2:
            w2[e] = np.abs(Q.dequant_fp4_weight_f32(host[e]["w2p"], host[e]["w2s"]))
        out[tok] += (w2[e] * h[r]).max(1)
    return out


# the routed rows from which the layer splits, takes 64-row experts too, and (pure bf16) splits, and one fewer
@pytest.mark.parametrize("profile,T,K", [("bf16", 5461, 3), ("bf16", 2048, 8), ("bf16", 13333, 3), ("bf16", 5000, 8),
                                         ("a4w4", 5461, 3), ("a4w4", 2048, 8), ("a4w4", 13333, 3), ("a4w4", 5000, 8),
                                         ("bf16_pure", 21845, 3), ("bf16_pure", 8192, 8)])
def test_layer_split_edges_vs_oracle(gpu, profile, T, K):
    """Experts with row counts around the thresholds and block edges, h quantised in every kernel's
    epilogue: the tokens of each such expert's first and last rows, of the rows around its 32-row
    tiles, and of 32 rows of expert 0."""
    E, D, I = 16, 1024, 1024
    ids, w, xb, host, devw, table = _case(T, K, E, D, I, 91 + T, gpu, _edge_ids(T, K, T))
    prof = {"bf16": PROFILE_BF16, "a4w4": PROFILE_A4W4, "bf16_pure": PROFILE_BF16_PURE}[profile]
    y = ops.LayerRunner(gpu, E, D, I).forward(_dev_bf16(xb, gpu), _dev(ids, gpu), _dev(w, gpu), table, profile=prof,
                                              rule=RULE_OCP_FLOOR)
    torch.cuda.synchronize()
    picks = set()
    for e in range(E):
        tok = np.nonzero(ids.reshape(-1) == e)[0] // K
        if e == 0:
            picks.update(tok[:16].tolist() + tok[-16:].tolist())
            continue
        edges = np.arange(0, tok.size, 32)
        picks.update(tok[edges].tolist() + tok[edges - 1].tolist())  # (edge 0 - 1: the last row)
    t = np.array(sorted(picks))
    if profile == "a4w4":
        ref = M.routed_a4w4(xb[t], ids[t], w[t], host, n_experts=E, rule="ocp_floor", workers=16)
    else:
        ref = M.routed_bf16(xb[t], ids[t], w[t], host, n_experts=E, fp8_act=profile == "bf16", workers=16)
    got, want = Q.bf16_bits_to_f32(_bits(y)), Q.bf16_bits_to_f32(ref["y"])
    assert np.isfinite(got).all()
    er = elementwise_rel(got[t], want)
    print(f"split edges {profile} T={T} K={K}: {t.size} tokens, normwise rel {rel(got[t], want):.3e}, "
          f"elementwise rel {er:.3e}", flush=True)
    assert rel(got[t], want) <= TOL[profile]
    if profile == "bf16":
        # A bf16 ulp of a gate or up sum may move an E4M3 code of h by one step, at most 2^-3 of its
        # value. With three rows to a token instead of eight one such step in an output's largest
        # product can exceed the 3e-2: it may be off by such a step in each of the token's rows instead.
        step = _largest_products(ref, host, t.size) * 2.0 ** -3
        err, size = np.abs(got[t].astype(np.float64) - want), np.abs(want.astype(np.float64))
        floor = np.maximum(size, np.sqrt((size * size).mean()))
        assert (err <= np.maximum(ELEM_TOL[profile] * floor, step)).all()
    else:
        assert er <= ELEM_TOL[profile]
    if profile == "a4w4":
        assert np.array_equal(_bits(y)[t], ref["y"])


def test_layer_forward_ceil_rule_and_int32_ids(gpu):
    T, K, E, D, I = 16, 4, 16, 512, 512
    ids, w, xb, host, devw, table = _case(T, K, E, D, I, 5, gpu)
    runner = ops.LayerRunner(gpu, E, D, I)
    y = runner.forward(_dev_bf16(xb, gpu), _dev(ids.astype(np.int32), gpu), _dev(w, gpu), table,
                       profile=PROFILE_A4W4, rule=RULE_CEIL_DIV6)
    torch.cuda.synchronize()
    ref = M.routed_a4w4(xb, ids, w, host, n_experts=E, rule="ceil_div6")
    assert rel(Q.bf16_bits_to_f32(_bits(y)), Q.bf16_bits_to_f32(ref["y"])) <= TOL["a4w4"]


# ---- the pure-bf16 variant: bf16 activations as they are on the bf16 MFMA ----
# Products of a bf16 value and an exactly dequantised E2M1 weight are exact in fp32 and
# the MFMA accumulates in fp32, so each output is within one bf16 ulp of the float64
# oracle plus 2^-16 of its sum of absolute products (fp32 summation over K <= 4096).
PURE_ACC_REL = 2.0 ** -16


_PURE_SHAPES = [(24, 4, 16, 1024, 512), (8, 8, 256, 4096, 2048), (200, 8, 16, 512, 512), (300, 8, 8, 2048, 1024)]


@pytest.mark.parametrize("T,K,E,D,I,block_m", [s + (bm,) for bm in (16, 64) for s in _PURE_SHAPES] +
                         [(40, 4, 8, 1024, 384, 64)] +
                         [(8, 8, 256, 4096, 2048, 256), (300, 8, 8, 2048, 1024, 256), (1024, 8, 8, 1024, 1024, 256)])
def test_grouped_gemm_stages_bf16_pure(gpu, T, K, E, D, I, block_m):
    # 16-row blocks: the single-wave kernel; 64-row blocks: the LDS-tiled kernel
    # (bf16 A tile in LDS, weight fragments dequantised once per 32-k half, weight
    # scales through a per-wave LDS table; 8-wave workgroups where the columns
    # divide by 256 (gate/up) or 512 (down), 4-wave ones otherwise: I = 384 runs a
    # 4-wave gate/up, and no down, whose reduction length must be a multiple of 256); 256-row
    # blocks: the large-tile bf16 kernel (32x32x16 bf16 MFMAs, weight fragments
    # dequantised in registers per 16-k chunk; hidden and inter multiples of 1024)
    _pure_stage_case(gpu, T, K, E, D, I, block_m)


@pytest.mark.parametrize("block_m", [16, 64, 256])
def test_grouped_gemm_stages_bf16_pure_row_counts(gpu, block_m):
    _pure_stage_case(gpu, 600, 4, 16, 1024, 1024, block_m, _edge_ids(600, 4, block_m))


def _pure_stage_case(gpu, T, K, E, D, I, block_m, ids=None):
    ids, w, xb, host, devw, table = _case(T, K, E, D, I, 71 + T, gpu, ids)
    al = ops.moe_align(_dev(ids, gpu), _dev(w, gpu), E, block_m)
    R = T * K
    x = _dev_bf16(xb, gpu)
    h = ops.gemm_gateup(AFMT_BF16, x, None, K, al, table, D, I, _dev(w.reshape(-1), gpu), 10.0)
    torch.cuda.synchronize()
    a_f = Q.bf16_bits_to_f32(xb)
    flat_e = ids.reshape(-1)
    h_ref = np.zeros((R, I), np.float32)
    g_all, u_all = np.zeros((R, I), np.float32), np.zeros((R, I), np.float32)
    g_abs, u_abs = np.zeros((R, I), np.float32), np.zeros((R, I), np.float32)
    for e in np.unique(flat_e):
        rows = np.nonzero(flat_e == e)[0]
        w1 = Q.dequant_fp4_weight_f32(host[e]["w1p"], host[e]["w1s"])
        w3 = Q.dequant_fp4_weight_f32(host[e]["w3p"], host[e]["w3s"])
        xa = a_f[rows // K]
        g = Q.f32_to_bf16_f32(M.matmul_nt(xa, w1))
        u = Q.f32_to_bf16_f32(M.matmul_nt(xa, w3))
        g_all[rows], u_all[rows] = g, u
        g_abs[rows], u_abs[rows] = M.matmul_nt(np.abs(xa), np.abs(w1)), M.matmul_nt(np.abs(xa), np.abs(w3))
        h_ref[rows] = M.swiglu(g, u, w.reshape(-1)[rows], 10.0)
    h_gpu = Q.bf16_bits_to_f32(_bits(h))
    h_want = Q.f32_to_bf16_f32(h_ref)
    print(f"pure bf16 gate/up T={T} block_m={block_m}: normwise rel {rel(h_gpu, h_want):.3e}")
    check_bound(h_gpu, h_want, swiglu_bound(g_all, u_all, w.reshape(-1), 10.0, h_want, g_abs, u_abs,
                                            acc_rel=PURE_ACC_REL), f"pure bf16 gate/up T={T} block_m={block_m}")
    if I % 256:
        return
    # down on the oracle's bf16 h, as it is
    hb = Q.f32_to_bf16_bits(h_ref)
    out = ops.gemm_down(AFMT_BF16, _dev_bf16(hb, gpu), None, al, table, I, D)
    torch.cuda.synchronize()
    hf = Q.bf16_bits_to_f32(hb)
    out_ref = np.zeros((R, D), np.float32)
    out_abs = np.zeros((R, D), np.float32)
    for e in np.unique(flat_e):
        rows = np.nonzero(flat_e == e)[0]
        w2 = Q.dequant_fp4_weight_f32(host[e]["w2p"], host[e]["w2s"])
        out_ref[rows] = M.matmul_nt(hf[rows], w2)
        out_abs[rows] = M.matmul_nt(np.abs(hf[rows]), np.abs(w2))
    out_gpu, out_want = Q.bf16_bits_to_f32(_bits(out)), Q.f32_to_bf16_f32(out_ref)
    print(f"pure bf16 down T={T} block_m={block_m}: normwise rel {rel(out_gpu, out_want):.3e}")
    check_bound(out_gpu, out_want, gemm_bound(out_want, out_abs, acc_rel=PURE_ACC_REL),
                f"pure bf16 down T={T} block_m={block_m}")


@pytest.mark.parametrize("block_m", [16, 64, 256])
def test_dequant_in_the_bf16_gemm_every_byte_and_scale(gpu, block_m):
    # one-hot activations pick single weight elements: out[f][n] = W[n][k(f)] exactly, so
    # every packed byte value with every E8M0 byte 0..252 goes through the GEMM's
    # dequantisation and must equal the oracle's bf16 dequant (up to the sign of zero).
    # Above 252 some weights are infinite, and 0 x inf would turn whole output columns
    # into NaN, as it does in any dot product with them.
    from dsv4_hip import AFMT_BF16
    D, I, E = (1024, 1024, 1) if block_m == 256 else (512, 512, 1)  # the large-tile kernel: I % 1024 == 0
    rng = np.random.default_rng(5)
    w2p = rng.integers(0, 256, (D, I // 2), dtype=np.uint8)
    w2s = np.tile(np.arange(253, dtype=np.uint8), (D * (I // 32)) // 253 + 1)[:D * (I // 32)].reshape(D, I // 32)
    rng.shuffle(w2s.reshape(-1))
    ex = {k: torch.zeros(16, dtype=torch.uint8, device=gpu) for k in ("w1p", "w1s", "w3p", "w3s")}
    ex["w2p"], ex["w2s"] = _dev(w2p, gpu), _dev(w2s, gpu)
    table = ops.expert_table({0: ex}, E, gpu)
    R = I  # row f picks k = f
    ids = np.zeros((R, 1), np.int64)
    al = ops.moe_align(_dev(ids, gpu), None, E, block_m)
    one = np.zeros((R, I), np.float32)
    one[np.arange(R), np.arange(R)] = 1.0
    out = ops.gemm_down(AFMT_BF16, _dev_bf16(Q.f32_to_bf16_bits(one), gpu), None, al, table, I, D)
    torch.cuda.synchronize()
    want = Q.dequant_fp4_weight_f32(w2p, w2s).T   # [k, n]
    got = Q.bf16_bits_to_f32(_bits(out))
    assert np.isfinite(want).all()
    bad = got != want
    if bad.any():
        k, n = np.nonzero(bad)
        sb = w2s[n, k // 32]
        print(f"{int(bad.sum())} differ; scale bytes {np.unique(sb)[:20]}; |want| max {np.abs(want[bad]).max():.3e}; "
              f"got {got[bad][:8]} want {want[bad][:8]}")
    assert not bad.any(), "dequantised weights differ"
    print(f"{want.size} weight elements checked, scale bytes 0..252")
