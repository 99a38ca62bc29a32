"""GPU parity of every HIP kernel against the CPU oracle, through the C ABI.

Tolerances are the north star's: int4 unpack/dequant bit-exact; bf16 outputs atol 2e-2 /
rtol 1e-2 (reference harness/correctness.py:55-56 uses 1e-2/1e-2); the fp32 gated-delta
state within 1e-4. Inputs are the seeded synthetic configs of ``deltaforge_amd.synth``.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from deltaforge_amd import _native as N
from deltaforge_amd import ops, synth
from deltaforge_amd.config import qwen3_5_4b_config
from oracle import ops as oracle_ops
from oracle.int4 import dequant_gemv, dequantise_int4_k_major_np
from oracle.model import apply_partial_rope, causal_conv, gated_rms_norm, rms_norm

pytestmark = pytest.mark.gpu

ATOL, RTOL = 2e-2, 1e-2
STATE_TOL = 1e-4
DEV = "cuda"


def close(got: torch.Tensor, want: torch.Tensor, atol=ATOL, rtol=RTOL, what="", flip_frac=0.0):
    """Every element within atol + rtol*|want|. ``flip_frac`` > 0 admits that fraction of
    elements within twice the bar: a fused bf16 op downstream of a GEMV can land one ulp
    away when its bf16 inputs did (fp32 summation order), and its own rounding adds one more."""
    got = got.detach().float().cpu()
    want = want.detach().float().cpu()
    assert got.shape == want.shape, (what, got.shape, want.shape)
    err = (got - want).abs()
    bar = atol + rtol * want.abs()
    bad = err > bar
    msg = f"{what}: {int(bad.sum())}/{bad.numel()} outside atol={atol} rtol={rtol}; max_abs={float(err.max()):.4g}"
    if flip_frac:
        assert float(bad.float().mean()) <= flip_frac and not bool((err > 2 * bar).any()), msg
    else:
        assert not bool(bad.any()), msg


def repack(w: synth.CanonicalInt4) -> ops.Int4Weight:
    return ops.int4_repack(w.packed.to(DEV), w.scale.to(DEV))


@pytest.mark.parametrize("rows,n,shift", [
    (1, 8, 0), (3, 504, 0), (5, 520, 0), (1025, 1032, 0), (7, 2560, 0), (2, 4096, 0), (2, 4104, 0), (3, 30, 0),
    (3, 2560, 4)])
def test_rms_norm_edges(rows, n, shift):
    """Rows a wave holds (remainders of its 512-element chunks, its longest, a last workgroup
    that is not full) and rows it does not: too long, not a multiple of 8, not 16-byte aligned."""
    gen = torch.Generator().manual_seed(rows + n)
    rand = lambda *s: torch.randn(s, generator=gen).to(torch.bfloat16)
    x, r, w = rand(rows, n), rand(rows, n), rand(n) * 0.1

    def dev(t):
        return torch.zeros(t.numel() + shift, dtype=t.dtype, device=DEV)[shift:].copy_(t.flatten()).view(t.shape)

    close(ops.rms_norm(dev(x), dev(w), 1e-6), rms_norm(x, w, 1e-6), what="norm", flip_frac=1e-2)
    resid, got = ops.add_rms_norm(dev(x), dev(r), dev(w), 1e-6)
    assert torch.equal(resid.cpu(), x + r), "sum"
    close(got, rms_norm(x + r, w, 1e-6), what="sum's norm", flip_frac=1e-2)


# -- int4 ---------------------------------------------------------------------------------


@pytest.mark.parametrize("k,n", [(256, 64), (2560, 1024), (9216, 128)])
def test_int4_dequant_is_bit_exact(k, n):
    gen = torch.Generator().manual_seed(k + n)
    w = synth.draw_int4(gen, k, n)
    got = ops.int4_dequant(repack(w)).cpu().view(torch.int16).numpy().view(np.uint16)
    want = dequantise_int4_k_major_np(w.packed.numpy(), w.scale.view(torch.int16).numpy().view(np.uint16), 128)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("rows,k,n", [(1, 2560, 1024), (1, 9216, 2560), (3, 4096, 2560), (16, 2560, 18432),
                                      (1, 2560, 64), (16, 9216, 2560)])
def test_int4_gemv_matches_champion_expression(rows, k, n):
    gen = torch.Generator().manual_seed(rows * 7 + k + n)
    w = synth.draw_int4(gen, k, n)
    x = torch.randn((rows, k), generator=gen).to(torch.bfloat16)
    got = ops.int4_gemv(x.to(DEV), repack(w))
    close(got, dequant_gemv(x, w.packed, w.scale, 128), what=f"gemv {rows}x{k}x{n}")


@pytest.mark.parametrize("epilogue", [N.EPI_STORE, N.EPI_RESIDUAL, N.EPI_SWIGLU])
def test_int4_gemv_k_split_reuses_its_workspace(epilogue):
    """A K split across workgroups (partials in the workspace, summed in split order by the
    reduce kernel, which runs the epilogue): three calls in a row on one workspace, different
    inputs, row counts and split counts, each against the expression; a repeat of the first
    call is bit-identical."""
    gen = torch.Generator().manual_seed(31 + epilogue)
    k, n = 4608, 256
    w = synth.draw_int4(gen, k, n)
    weight = repack(w)
    plans = [ops.GemvPlan(2, 6, 6, int(N.lib().df_int4_gemv_workspace_bytes(16, n, 6))),
             ops.GemvPlan(4, 3, 12, int(N.lib().df_int4_gemv_workspace_bytes(16, n, 3)))]
    ws = torch.zeros(max(p.workspace_bytes for p in plans), dtype=torch.uint8, device=DEV)
    firsts = []
    for rows, plan in ((16, plans[0]), (5, plans[1]), (1, plans[0])):
        x = torch.randn((rows, k), generator=gen).to(torch.bfloat16)
        res = torch.randn((rows, n), generator=gen).to(torch.bfloat16)
        print(f"[k-split] epilogue {epilogue} rows {rows} ksplit {plan.ksplit}", flush=True)
        got = ops.int4_gemv(x.to(DEV), weight, epilogue=epilogue, plan=plan, ws=ws,
                            res=res.to(DEV) if epilogue == N.EPI_RESIDUAL else None)
        y = dequant_gemv(x, w.packed, w.scale, 128)
        if epilogue == N.EPI_RESIDUAL:
            want = (res.float() + y.float()).to(torch.bfloat16)
        elif epilogue == N.EPI_SWIGLU:  # 16-column gate / up tiles alternate
            yf = y.float().reshape(rows, n // 32, 2, 16)
            g, u = yf[:, :, 0].to(torch.bfloat16).float(), yf[:, :, 1].to(torch.bfloat16).float()
            want = (torch.nn.functional.silu(g).to(torch.bfloat16).float() * u).to(torch.bfloat16).reshape(rows, n // 2)
        else:
            want = y
        close(got, want, what=f"k-split gemv epilogue {epilogue} rows {rows}",
              flip_frac=2e-3 if epilogue == N.EPI_SWIGLU else 0.0)
        firsts.append((x, got.clone(), res))
    x0, got0, res0 = firsts[0]
    again = ops.int4_gemv(x0.to(DEV), weight, epilogue=epilogue, plan=plans[0], ws=ws,
                          res=res0.to(DEV) if epilogue == N.EPI_RESIDUAL else None)
    assert torch.equal(again, got0)


@pytest.mark.parametrize("prologue,epilogue,rows,k,nt", [
    (N.PRO_NONE, N.EPI_STORE, 1, 256, 1), (N.PRO_NONE, N.EPI_STORE, 6, 1280, 8), (N.PRO_NONE, N.EPI_STORE, 16, 1536, 8),
    (N.PRO_RMSNORM, N.EPI_STORE, 1, 256, 1), (N.PRO_RMSNORM, N.EPI_STORE, 3, 4096, 4),
    (N.PRO_RMSNORM, N.EPI_STORE, 2, 4352, 2), (N.PRO_RMSNORM, N.EPI_STORE, 9, 512, 8),
    (N.PRO_RMSNORM, N.EPI_LOGITS, 16, 2560, 8), (N.PRO_ADD_RMSNORM, N.EPI_LOGITS, 5, 2816, 8),
    (N.PRO_ADD_RMSNORM, N.EPI_STORE, 1, 4352, 1), (N.PRO_ADD_RMSNORM, N.EPI_STORE, 4, 2560, 4),
    (N.PRO_ADD_RMSNORM, N.EPI_STORE, 16, 2304, 2), (N.PRO_ADD_RMSNORM, N.EPI_STORE, 5, 4352, 8),
    (N.PRO_ADD_RMSNORM, N.EPI_STORE, 5, 256, 1), (N.PRO_ADD_RMSNORM, N.EPI_LOGITS, 16, 1024, 4),
    (N.PRO_RMSNORM, N.EPI_STORE, 9, 768, 2), (N.PRO_RMSNORM, N.EPI_STORE, 6, 1280, 2),
    (N.PRO_GATED_RMSNORM, N.EPI_STORE, 1, 256, 1), (N.PRO_GATED_RMSNORM, N.EPI_STORE, 3, 4096, 8),
    (N.PRO_GATED_RMSNORM, N.EPI_STORE, 7, 512, 4), (N.PRO_GATED_RMSNORM, N.EPI_STORE, 16, 2304, 2)])
def test_int4_gemv_prologue_forms(prologue, epilogue, rows, k, nt):
    """Rows and widths on both sides of what a prologue loads ahead of the weights, and from no
    group to several sets of groups in a wave. The norm's bf16 results may round the other way where
    the fp32 sum's order does (one in thousands, 2^-8 each), so the product is held normwise, like the
    MLP block."""
    print(f"gemv prologue {prologue} {rows} {k} {nt}", flush=True)
    gen = torch.Generator().manual_seed(rows + k)
    rand = lambda *s: torch.randn(s, generator=gen).to(torch.bfloat16)
    w = synth.draw_int4(gen, k, 128)
    x, x2 = rand(rows, k), rand(rows, k)
    nw = rand(128 if prologue == N.PRO_GATED_RMSNORM else k) * 0.1
    h_out = torch.zeros((rows, k), dtype=torch.bfloat16, device=DEV)
    kw = {} if prologue == N.PRO_NONE else {"norm_w": nw.to(DEV)}
    if prologue in (N.PRO_ADD_RMSNORM, N.PRO_GATED_RMSNORM):
        kw["x2"] = x2.to(DEV)
    if prologue == N.PRO_ADD_RMSNORM:
        kw["h_out"] = h_out
    got = ops.int4_gemv(x.to(DEV), repack(w), prologue=prologue, epilogue=epilogue,
                        plan=ops.GemvPlan(nt, 1, k // 128, 0), **kw)
    if prologue == N.PRO_RMSNORM:
        x = rms_norm(x, nw, 1e-6)
    elif prologue == N.PRO_ADD_RMSNORM:
        assert torch.equal(h_out.cpu(), x + x2)
        x = rms_norm(x + x2, nw, 1e-6)
    elif prologue == N.PRO_GATED_RMSNORM:
        x = gated_rms_norm(x.reshape(-1, 128), x2.reshape(-1, 128), nw, 1e-6).reshape(rows, k)
    want = dequant_gemv(x, w.packed, w.scale, 128).float()
    err = float((got.float().cpu() - want).abs().max())
    assert err <= ATOL + RTOL * float(want.abs().max()), f"max abs err {err:.4g}"


def test_int4_gemv_is_deterministic_across_runs():
    gen = torch.Generator().manual_seed(5)
    w = synth.draw_int4(gen, 9216, 2560)
    x = torch.randn((1, 9216), generator=gen).to(torch.bfloat16).to(DEV)
    weight = repack(w)
    first = ops.int4_gemv(x, weight)
    for _ in range(5):
        assert torch.equal(ops.int4_gemv(x, weight), first)


def test_config1_tied_head_with_residual_and_rmsnorm():
    inp = synth.head_inputs(seed=0)
    w = inp["weight"]
    weight = repack(w)
    x, r, nw = inp["x"], inp["residual"], inp["norm_w"]
    h_out = torch.empty((1, 2560), dtype=torch.bfloat16, device=DEV)
    got = ops.int4_gemv(x.to(DEV), weight, prologue=N.PRO_ADD_RMSNORM, x2=r.to(DEV), norm_w=nw.to(DEV),
                        eps=inp["eps"], h_out=h_out)
    want = oracle_ops.head(x, r, nw, w.packed, w.scale, 128, inp["eps"])
    close(got, want, what="head logits")
    assert torch.equal(h_out.cpu(), r + x)
    top2 = want.float().topk(2).values[0]
    if float(top2[0] - top2[1]) > 0.5:  # only a clear winner must agree exactly
        assert int(got.float().argmax()) == int(want.float().argmax())


@pytest.mark.parametrize("rows", [1, 16])
def test_config4_mlp_block(rows):
    inp = synth.mlp_inputs(seed=0, rows=rows)
    gate, up, down = inp["gate"], inp["up"], inp["down"]
    # gate / up tiles alternate so one workgroup holds both halves of SwiGLU.
    gp, gs = ops.interleave_gate_up(gate.packed, gate.scale, up.packed, up.scale)
    gu = ops.int4_repack(gp.to(DEV), gs.to(DEV))
    dn = repack(down)
    x = inp["x"].to(DEV)
    act = ops.int4_gemv(x, gu, prologue=N.PRO_RMSNORM, epilogue=N.EPI_SWIGLU, norm_w=inp["norm_w"].to(DEV))
    out = ops.int4_gemv(act, dn, epilogue=N.EPI_RESIDUAL, res=x)
    # Per op, on identical inputs (the north star's per-op bar): kernel 1 = RMSNorm + gate/up
    # GEMV + SwiGLU, kernel 2 = down GEMV + residual, each against the oracle's expression.
    n = rms_norm(inp["x"], inp["norm_w"], inp["eps"])
    want_act = torch.nn.functional.silu(dequant_gemv(n, gate.packed, gate.scale, 128)) * dequant_gemv(
        n, up.packed, up.scale, 128)
    close(act, want_act, what=f"gate/up+swiglu rows={rows}", flip_frac=1e-4)
    act_cpu = act.cpu()
    close(out, inp["x"] + dequant_gemv(act_cpu, down.packed, down.scale, 128), what=f"down+residual rows={rows}")
    # The whole block against the oracle's own chain: a 1-ulp flip of one bf16 intermediate
    # (different fp32 summation order) reaches every output through the 9216-term down
    # projection as an absolute error, so the composite is held normwise: max error within
    # 1e-2 of the output's largest magnitude (the per-op bars above are elementwise).
    want = oracle_ops.mlp_block(inp["x"], inp["norm_w"], (gate.packed, gate.scale), (up.packed, up.scale),
                                (down.packed, down.scale)).float()
    err = float((out.float().cpu() - want).abs().max())
    assert err <= ATOL + RTOL * float(want.abs().max()), f"mlp block rows={rows}: max abs err {err:.4g}"


@pytest.mark.parametrize("rows", [1, 8])
def test_gated_rmsnorm_out_proj_residual(rows):
    """GatedDeltaNet's tail as one GEMV launch: the per-head GatedRMSNorm prologue
    (``DF_PRO_GATED_RMSNORM``: norm over each 128-wide head, plain weight, SiLU(z) gate;
    reference.py:115-121, 546-550), the int4 out_proj 4096 -> 2560 and the residual epilogue
    (reference.py:730). Against the oracle's gated_rms_norm -> dequant_gemv -> bf16 add."""
    from oracle.model import gated_rms_norm

    gen = torch.Generator().manual_seed(40 + rows)
    w = synth.draw_int4(gen, 4096, 2560)
    core = torch.randn((rows, 4096), generator=gen).to(torch.bfloat16)
    z = torch.randn((rows, 4096), generator=gen).to(torch.bfloat16)
    gw = (1.0 + 0.02 * torch.randn(128, generator=gen)).to(torch.bfloat16)
    res = torch.randn((rows, 2560), generator=gen).to(torch.bfloat16)
    got = ops.int4_gemv(core.to(DEV), repack(w), prologue=N.PRO_GATED_RMSNORM, epilogue=N.EPI_RESIDUAL,
                        x2=z.to(DEV), norm_w=gw.to(DEV), res=res.to(DEV), eps=1e-6)
    normed = gated_rms_norm(core.reshape(-1, 128), z.reshape(-1, 128), gw, 1e-6).reshape(rows, 4096)
    y = dequant_gemv(normed, w.packed, w.scale, 128)
    close(got, res + y, what=f"gated norm + out_proj + residual rows={rows}")


# -- gated delta --------------------------------------------------------------------------


@pytest.mark.parametrize("batch", [1, 8])
def test_config2_gated_delta_step(batch):
    inp = synth.delta_inputs(seed=0, batch=batch)
    state = inp["state"].to(DEV).contiguous()
    conv_out = torch.empty_like(inp["conv_state"]).to(DEV)
    out = ops.gated_delta_step(inp["qkv"].to(DEV), inp["a"].to(DEV), inp["b"].to(DEV), inp["A_log"].to(DEV),
                               inp["dt_bias"].to(DEV), inp["conv_w"].to(DEV), state,
                               num_k_heads=inp["num_k_heads"], conv_in=inp["conv_state"].to(DEV), conv_out=conv_out)
    w_out, w_state, w_conv = oracle_ops.delta_step(inp["qkv"], inp["conv_state"], inp["conv_w"], inp["a"], inp["b"],
                                                   inp["A_log"], inp["dt_bias"], inp["state"], inp["num_k_heads"])
    close(out, w_out, what="delta out")
    close(state, w_state, atol=STATE_TOL, rtol=0, what="delta state")
    assert torch.equal(conv_out.cpu(), w_conv)


def test_gated_delta_ring_mode_matches_reference_layout():
    inp = synth.delta_inputs(seed=3, batch=2)
    pos = 5
    hist = inp["conv_state"]
    ring = torch.zeros((2, hist.shape[1], 4), dtype=torch.bfloat16)
    for j in range(3):  # oldest .. newest at positions pos-3 .. pos-1
        ring[:, :, (pos - 3 + j) % 4] = hist[:, :, j]
    ring = ring.to(DEV)
    position = torch.tensor([pos], dtype=torch.int32, device=DEV)
    state = inp["state"].to(DEV).contiguous()
    out = ops.gated_delta_step(inp["qkv"].to(DEV), inp["a"].to(DEV), inp["b"].to(DEV), inp["A_log"].to(DEV),
                               inp["dt_bias"].to(DEV), inp["conv_w"].to(DEV), state,
                               num_k_heads=16, conv_ring=ring, position=position)
    w_out, w_state, w_conv = oracle_ops.delta_step(inp["qkv"], hist, inp["conv_w"], inp["a"], inp["b"],
                                                   inp["A_log"], inp["dt_bias"], inp["state"], 16)
    close(out, w_out, what="ring out")
    ring = ring.cpu()
    got_hist = torch.stack([ring[:, :, (pos - 2 + j) % 4] for j in range(3)], dim=-1)
    assert torch.equal(got_hist, w_conv)


# -- attention ----------------------------------------------------------------------------


def _attention_case(batch, context, slack=64):
    cfg = qwen3_5_4b_config()
    inp = synth.attention_inputs(seed=0, batch=batch, context=context, slack=slack)
    kc, vc = inp["k_cache"].to(DEV), inp["v_cache"].to(DEV)
    position = torch.tensor([context], dtype=torch.int32, device=DEV)
    inv = synth.inv_freq(cfg).to(DEV)
    got = ops.attention_decode(inp["q"].to(DEV), inp["k"].to(DEV), inp["v"].to(DEV), inp["q_norm_w"].to(DEV),
                               inp["k_norm_w"].to(DEV), inv, kc, vc, position, num_q_heads=16)
    wk, wv = inp["k_cache"].clone(), inp["v_cache"].clone()
    want = oracle_ops.attention_decode(inp["q"], inp["k"], inp["v"], inp["q_norm_w"], inp["k_norm_w"], wk, wv,
                                       context, cfg)
    close(got, want, what=f"attention B={batch} L={context}")
    # The new key (normed, roped) and value were written at `position`.
    close(kc[:, :, context].cpu(), wk[:, :, context], what="k write")
    assert torch.equal(vc[:, :, context].cpu(), wv[:, :, context])


@pytest.mark.parametrize("batch,context", [(1, 4096), (8, 4096), (1, 32768), (8, 32768), (1, 131072), (8, 131072)])
def test_config3_split_kv_decode(batch, context):
    print(f"attention case B={batch} L={context}", flush=True)
    _attention_case(batch, context)


@pytest.mark.parametrize("context", [0, 2, 31, 63, 64, 65, 200])
def test_attention_edge_contexts(context):
    _attention_case(1, context)


# -- elementwise ops ----------------------------------------------------------------------


def test_rms_norm_and_add_rms_norm():
    gen = torch.Generator().manual_seed(1)
    x = torch.randn((3, 2560), generator=gen).to(torch.bfloat16)
    r = torch.randn((3, 2560), generator=gen).to(torch.bfloat16)
    w = (torch.randn(2560, generator=gen) * 0.1).to(torch.bfloat16)
    close(ops.rms_norm(x.to(DEV), w.to(DEV), 1e-6), rms_norm(x, w, 1e-6), what="rms_norm")
    s, n = ops.add_rms_norm(x.to(DEV), r.to(DEV), w.to(DEV), 1e-6)
    assert torch.equal(s.cpu(), r + x)
    close(n, rms_norm(r + x, w, 1e-6), what="add_rms_norm")


def test_silu_mul_matches_reference_rounding():
    gen = torch.Generator().manual_seed(2)
    g = (torch.randn(9216 * 3, generator=gen) * 4).to(torch.bfloat16)
    u = (torch.randn(9216 * 3, generator=gen) * 4).to(torch.bfloat16)
    close(ops.silu_mul(g.to(DEV), u.to(DEV)), torch.nn.functional.silu(g) * u, atol=0, rtol=1e-2, what="silu_mul")


def test_partial_rope_matches_reference():
    gen = torch.Generator().manual_seed(3)
    x = torch.randn((2, 4, 3, 256), generator=gen).to(torch.bfloat16)
    ang = torch.randn((2, 3, 32), generator=gen) * 100
    emb = torch.cat((ang, ang), -1)
    cos, sin = emb.cos().to(torch.bfloat16), emb.sin().to(torch.bfloat16)
    got = ops.partial_rope(x.to(DEV), cos.to(DEV), sin.to(DEV))
    assert torch.equal(got.cpu(), apply_partial_rope(x, cos, sin))


def test_causal_conv_step_matches_conv1d():
    gen = torch.Generator().manual_seed(4)
    x = torch.randn((2, 8192, 1), generator=gen).to(torch.bfloat16)
    hist = torch.randn((2, 8192, 3), generator=gen).to(torch.bfloat16)
    w = (torch.randn((8192, 1, 4), generator=gen) * 0.3).to(torch.bfloat16)
    cache = hist.clone().to(DEV)
    got = ops.causal_conv_step(x.to(DEV), cache, w.to(DEV))
    want, new_hist = causal_conv(x, hist, w)
    close(got, want, atol=0, rtol=1e-2, what="conv out")
    assert torch.equal(cache.cpu(), new_hist)


def test_embed_int4_is_the_dequantised_head_column():
    gen = torch.Generator().manual_seed(6)
    w = synth.draw_int4(gen, 2560, 4096)
    weight = repack(w)
    tokens = torch.tensor([0, 17, 4095], dtype=torch.int64, device=DEV)
    got = ops.embed_int4(tokens, weight)
    dense = ops.int4_dequant(weight)  # [K, N], bit-exact (tested above)
    assert torch.equal(got, dense[:, tokens].t())


def test_argmax_first_max_and_bookkeeping():
    logits = torch.randn((2, 248320)).to(torch.bfloat16)
    logits[0, 1000] = 50.0
    logits[0, 200000] = 50.0  # tie: the first index wins, as torch.argmax
    logits[1, 248319] = 60.0
    tokens = torch.zeros(2, dtype=torch.int64, device=DEV)
    log = torch.full((2, 4), -1, dtype=torch.int64, device=DEV)
    position = torch.tensor([10], dtype=torch.int32, device=DEV)
    step = torch.tensor([1], dtype=torch.int32, device=DEV)
    ops.argmax_tokens(logits.to(DEV), tokens, token_log=log, position=position, advance=1, step=step)
    assert tokens.tolist() == [1000, 248319]
    assert log[:, 1].tolist() == [1000, 248319]
    assert int(position) == 11 and int(step) == 2
