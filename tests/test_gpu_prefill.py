"""GPU parity of the prompt prefill (csrc/prefill.hip) against the CPU oracle's forward.

Kernel by kernel:
- the int4 GEMM against ``dequant_gemv``, the reference expression;
- the conv bit for bit against ``F.conv1d`` (the oracle's ``causal_conv``);
- the chunked delta rule against the token-by-token scan, at chunk edges (1, 63, 64, 65,
  200 tokens) and from a nonzero state.

Layer by layer, against ``OracleModel._delta_net`` / ``_attention`` with their caches. Then
the whole mid-config model against ``OracleModel.forward``:
- last-position KL and top-1;
- every cache;
- the greedy continuation of a ``PersistentDecoder`` filled by ``Prefiller.fill``.

Bars:
- bf16 outputs atol 2e-2 / rtol 1e-2, the kernel tests' bar;
- fp32 states 1e-4 of their scale for the kernel alone, 1e-3 for one layer, and 2e-2 deep in
  the model, where the inputs already differ by ulps.

The chunked scan reassociates fp32 sums, so nothing beyond the conv is bit-exact.
"""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from deltaforge_amd import _native as N
from deltaforge_amd import ops, synth
from deltaforge_amd.config import FULL_ATTENTION, LINEAR_ATTENTION, mid_config
from deltaforge_amd.harness.correctness import kl_and_agreement
from deltaforge_amd.persistent import PersistentDecoder
from deltaforge_amd.prefill import (Prefiller, causal_conv_prefill, delta_rule_prefill, gated_rms_norm_rows,
                                    int4_gemm)
from oracle.int4 import dequant_gemv
from oracle.model import causal_conv, gated_delta_rule, gated_rms_norm, rope_cos_sin

from .test_gpu_engine import oracle_for
from .test_gpu_kernels import close, repack

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rel_close(got, want, rel, what):
    got, want = got.float().cpu(), want.float().cpu()
    err = float((got - want).abs().max())
    scale = float(want.abs().max())
    assert err <= rel * max(scale, 1e-30), f"{what}: max err {err:.3g} vs scale {scale:.3g}"


# -- GEMM -----------------------------------------------------------------------------------


@pytest.mark.parametrize("m,k,n", [(1, 256, 64), (77, 512, 192), (300, 2560, 1088), (129, 9216, 256)])
def test_int4_gemm_is_the_dequantised_product(m, k, n):
    print(f"gemm {m}x{k}x{n}", flush=True)
    gen = torch.Generator().manual_seed(m + k + n)
    w = synth.draw_int4(gen, k, n)
    x = torch.randn((m, k), generator=gen).to(torch.bfloat16)
    got = int4_gemm(x.to(DEV), repack(w))
    close(got, dequant_gemv(x, w.packed, w.scale, 128), what=f"gemm {m}x{k}x{n}", flip_frac=1e-3)


def test_int4_gemm_strided_rows_and_swiglu_epilogue():
    gen = torch.Generator().manual_seed(3)
    m, k, inter = 150, 512, 320
    gate, up = synth.draw_int4(gen, k, inter), synth.draw_int4(gen, k, inter)
    wide = torch.randn((m, k + 64), generator=gen).to(torch.bfloat16)
    x = wide[:, 32:32 + k]  # row stride k + 64, 64-byte offset
    gp, gs = ops.interleave_gate_up(gate.packed, gate.scale, up.packed, up.scale)
    gu = ops.int4_repack(gp.to(DEV), gs.to(DEV))
    got = int4_gemm(wide.to(DEV)[:, 32:32 + k], gu, epilogue=N.EPI_SWIGLU)
    want = F.silu(dequant_gemv(x, gate.packed, gate.scale, 128)) * dequant_gemv(x, up.packed, up.scale, 128)
    close(got, want, what="gate|up + SwiGLU", flip_frac=2e-3)


# (M, K, N) that take each launch shape (128 x 256, 128 x 128, 96 x 256, 96 x 128, 64 x 128, 64 x 64,
# 32 x 64) with a partial last row block, a partial last column block and one or more rounds
@pytest.mark.parametrize("m,k,n,epilogue", [
    (700, 512, 8208, N.EPI_STORE), (300, 512, 8208, N.EPI_STORE), (641, 512, 6176, N.EPI_SWIGLU),
    (161, 512, 12304, N.EPI_STORE), (97, 512, 8208, N.EPI_STORE), (33, 768, 8224, N.EPI_SWIGLU),
    (31, 768, 1040, N.EPI_STORE), (2100, 256, 4128, N.EPI_SWIGLU)])
def test_int4_gemm_rows_do_not_depend_on_the_launch_shape(m, k, n, epilogue):
    """Each shape against the expression on its first, last and some middle rows, and bit for
    bit against the same rows as products of their own (other launch shapes); then with an output
    and scales that allow neither 16-byte stores nor 4-byte loads."""
    print(f"gemm shapes {m}x{k}x{n} epilogue {epilogue}", flush=True)
    gen = torch.Generator().manual_seed(m + n)
    w = synth.draw_int4(gen, k, -(-n // 64) * 64)
    x = torch.randn((m, k), generator=gen).to(torch.bfloat16)
    xd, whole = x.to(DEV), repack(w)
    tiles = n // 16 * (k // 128)  # the first n columns are the first n / 16 tiles
    weight = ops.Int4Weight(whole.w[:tiles * 1024], whole.s[:tiles * 16], k, n)
    got = int4_gemm(xd, weight, epilogue=epilogue)
    rows = torch.tensor(sorted({0, 1, min(31, m - 1), m // 2, m - 2, m - 1}))
    want = dequant_gemv(x[rows], w.packed, w.scale, 128)[:, :n]
    if epilogue == N.EPI_SWIGLU:  # 16-column gate / up tiles alternate
        gu = want.reshape(len(rows), n // 32, 2, 16)
        want = (F.silu(gu[:, :, 0]) * gu[:, :, 1]).reshape(len(rows), n // 2)
    close(got[rows.to(DEV)], want, what=f"gemm {m}x{k}x{n}", flip_frac=2e-3)
    for r0, r1 in ((0, 1), (0, min(m, 40)), (m // 2, m), (m - 1, m)):
        assert torch.equal(int4_gemm(xd[r0:r1], weight, epilogue=epilogue), got[r0:r1]), (r0, r1)
    cols = got.shape[1]
    odd = torch.zeros((m, cols + 3), dtype=torch.bfloat16, device=DEV)[:, 1:1 + cols]
    scales = torch.zeros(weight.s.numel() + 1, dtype=torch.bfloat16, device=DEV)[1:]
    scales.copy_(weight.s)
    int4_gemm(xd, ops.Int4Weight(weight.w, scales, k, n), epilogue=epilogue, out=odd)
    assert torch.equal(odd, got)


def test_int4_gemm_rejects_bad_shapes():
    gen = torch.Generator().manual_seed(4)
    w = repack(synth.draw_int4(gen, 256, 64))
    with pytest.raises(ValueError):
        int4_gemm(torch.zeros((4, 128), dtype=torch.bfloat16, device=DEV), w)
    with pytest.raises(RuntimeError):
        int4_gemm(torch.zeros((4, 256), dtype=torch.bfloat16), w)


# -- conv, delta rule, gated norm ----------------------------------------------------------


@pytest.mark.parametrize("tokens,pos0", [(1, 0), (2, 0), (37, 0), (37, 5)])
def test_causal_conv_prefill_is_conv1d(tokens, pos0):
    gen = torch.Generator().manual_seed(tokens + pos0)
    channels = 8192
    x = torch.randn((tokens, channels), generator=gen).to(torch.bfloat16)
    w = (torch.randn((channels, 1, 4), generator=gen) * 0.3).to(torch.bfloat16)
    hist = torch.zeros((1, channels, 3), dtype=torch.bfloat16)
    ring = torch.zeros((channels, 4), dtype=torch.bfloat16)
    if pos0:
        hist = torch.randn((1, channels, 3), generator=gen).to(torch.bfloat16)
        for j in range(3):  # positions pos0-3 .. pos0-1
            ring[:, (pos0 - 3 + j) % 4] = hist[0, :, j]
    ring_d = ring.to(DEV)
    got = causal_conv_prefill(x.to(DEV), w.reshape(channels, 4).to(DEV), ring_d, pos0=pos0)
    want, new_hist = causal_conv(x.t().unsqueeze(0), hist, w)
    assert torch.equal(got.cpu(), want[0].t()), "conv output"
    ring_h = ring_d.cpu()
    end = pos0 + tokens
    got_hist = torch.stack([ring_h[:, (end - 3 + j) % 4] for j in range(3)], dim=-1)
    assert torch.equal(got_hist, new_hist[0]), "history ring"


@pytest.mark.parametrize("tokens,pos0,channels,shift,pad", [
    (1, 2, 4, 0, 0), (3, 1, 1028, 0, 4), (4, 7, 1020, 0, 0), (5, 0, 6, 0, 2), (17, 3, 260, 4, 0), (17, 3, 260, 1, 0),
    (31, 6, 257, 0, 3), (2047, 5, 8, 0, 0), (2048, 0, 12, 0, 0), (2050, 9, 5, 0, 0), (1024, 2, 8191, 0, 1),
    (1025, 3, 8192, 0, 0), (2049, 3, 8194, 0, 0), (2049, 2, 8194, 1, 1)])
def test_causal_conv_prefill_edges(tokens, pos0, channels, shift, pad):
    """Remainders of the tokens a thread walks (4 below 2^23 elements, 16 from there) and of a workgroup's
    channels (two a thread from 2^24 elements), rows that allow only 2-byte loads, and the history ring read
    and written by one call; exact, as both sides take the taps in order in fp32."""
    print(f"conv edges {tokens} {pos0} {channels} {shift} {pad}", flush=True)
    gen = torch.Generator().manual_seed(tokens + channels)
    rand = lambda *s: torch.randn(s, generator=gen).to(torch.bfloat16)
    w, ring, x = rand(channels, 1, 4), rand(channels, 4), rand(tokens, channels)
    wide = torch.zeros((tokens, channels + shift + pad), dtype=torch.bfloat16, device=DEV)[:, shift:shift + channels]
    wide.copy_(x)
    ring_d = ring.to(DEV)
    got = causal_conv_prefill(wide, w.reshape(channels, 4).to(DEV), ring_d, pos0=pos0)
    hist = torch.stack([ring[:, (pos0 - 3 + j) % 4] for j in range(3)], dim=-1)
    want, new_hist = causal_conv(x.t().unsqueeze(0), hist.unsqueeze(0), w)
    assert torch.equal(got.cpu(), want[0].t()), "conv output"
    end = pos0 + tokens
    kept = torch.stack([ring_d.cpu()[:, (end - 3 + j) % 4] for j in range(3)], dim=-1)
    assert torch.equal(kept, new_hist[0]), "history ring"
    if tokens < 4:  # the slots that no token fell on
        same = [s for s in range(4) if s not in {(pos0 + t) % 4 for t in range(tokens)}]
        assert torch.equal(ring_d.cpu()[:, same], ring[:, same]), "other slots"


def test_conv_silu_rounds_every_bf16_like_64_bits():
    """One token whose channels are all the finite bf16 numbers, weight 1 on its own tap."""
    bits = torch.arange(1 << 16, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    x = bits[torch.isfinite(bits.float())]
    w = torch.zeros((x.numel(), 4), dtype=torch.bfloat16)
    w[:, 3] = 1
    ring = torch.zeros((x.numel(), 4), dtype=torch.bfloat16, device=DEV)
    got = causal_conv_prefill(x.unsqueeze(0).to(DEV), w.to(DEV), ring)[0].cpu()
    x64 = x.double()
    want = (x64 / (1 + torch.exp(-x64))).to(torch.bfloat16)
    # e^-x is past fp32's range below -88.7, where the quotient is under 2e-37 and may be zero
    far = x64 < -88.7
    assert torch.equal(got[~far], want[~far])
    assert float(got[far].double().abs().max()) < 2e-37


def _delta_case(tokens, seed, hk=16, hv=32):
    gen = torch.Generator().manual_seed(seed)
    mixed = (torch.randn((tokens, (2 * hk + hv) * 128), generator=gen)).to(torch.bfloat16)
    ab = torch.randn((tokens, 2 * hv + 8), generator=gen).to(torch.bfloat16)
    A_log = (torch.randn(hv, generator=gen) * 0.5).to(torch.bfloat16)
    dt_bias = (torch.randn(hv, generator=gen) * 0.5).to(torch.bfloat16)
    state = torch.randn((hv, 128, 128), generator=gen) * 0.1
    return mixed, ab, A_log, dt_bias, state


def _delta_oracle(mixed, ab, A_log, dt_bias, state, hk, hv):
    """The oracle's _delta_net between the conv and the gated norm (reference.py:518-545)."""
    tokens = mixed.shape[0]
    q, k, v = torch.split(mixed.unsqueeze(0), [hk * 128, hk * 128, hv * 128], dim=-1)
    q = q.reshape(1, tokens, hk, 128).repeat_interleave(hv // hk, dim=2)
    k = k.reshape(1, tokens, hk, 128).repeat_interleave(hv // hk, dim=2)
    v = v.reshape(1, tokens, hv, 128)
    a, b = ab[:, :hv].unsqueeze(0), ab[:, hv:2 * hv].unsqueeze(0)
    beta = b.sigmoid()
    g = -A_log.float().exp() * F.softplus(a.float() + dt_bias.float())
    out, new_state = gated_delta_rule(q, k, v, g, beta, state.unsqueeze(0))
    return out[0].reshape(tokens, hv * 128), new_state[0]


@pytest.mark.parametrize("tokens", [1, 63, 64, 65, 200])
def test_delta_rule_prefill_matches_the_scan(tokens):
    print(f"delta prefill {tokens}", flush=True)
    hk, hv = 16, 32
    mixed, ab, A_log, dt_bias, state = _delta_case(tokens, seed=tokens)
    st = state.to(DEV).contiguous()
    ab_d = ab.to(DEV)
    got = delta_rule_prefill(mixed.to(DEV), ab_d[:, :hv], ab_d[:, hv:], A_log.to(DEV), dt_bias.to(DEV), st,
                             num_k_heads=hk)
    want, want_state = _delta_oracle(mixed, ab, A_log, dt_bias, state, hk, hv)
    close(got, want, what=f"delta out P={tokens}", flip_frac=1e-3)
    _rel_close(st, want_state, 1e-4, f"delta state P={tokens}")


@pytest.mark.parametrize("tokens,hk,hv,shift,pad", [
    (15, 1, 1, 0, 0), (17, 2, 6, 2, 0), (64, 1, 4, 0, 2), (127, 2, 2, 2, 6), (128, 2, 4, 0, 8), (129, 1, 3, 8, 0),
    (191, 2, 8, 4, 4)])
def test_delta_rule_prefill_edges(tokens, hk, hv, shift, pad):
    """16-token blocks and 64-token chunks with remainders, head ratios, and rows that allow only
    4-byte loads (``shift`` and ``pad`` elements before and after each); an ``out`` inside ``mixed``'s
    own memory; and the same bits when the tokens come in two calls split at a chunk."""
    print(f"delta prefill edges {tokens} {hk} {hv} {shift} {pad}", flush=True)
    mixed, ab, A_log, dt_bias, state = _delta_case(tokens, seed=tokens, hk=hk, hv=hv)
    width = mixed.shape[1]
    wide = torch.zeros((tokens, width + shift + pad), dtype=torch.bfloat16, device=DEV)[:, shift:shift + width]
    wide.copy_(mixed)
    ab_d, al, dt = ab.to(DEV), A_log.to(DEV), dt_bias.to(DEV)

    def run(at, end, st, **kw):
        return delta_rule_prefill(wide[at:end], ab_d[at:end, :hv], ab_d[at:end, hv:], al, dt, st, num_k_heads=hk, **kw)

    st = state.to(DEV)
    got = run(0, tokens, st)
    want, want_state = _delta_oracle(mixed, ab, A_log, dt_bias, state, hk, hv)
    close(got, want, what=f"delta out P={tokens}", flip_frac=1e-3)
    _rel_close(st, want_state, 1e-4, f"delta state P={tokens}")
    if tokens > 64:
        st2 = state.to(DEV)
        parts = torch.cat([run(0, 64, st2), run(64, tokens, st2)])
        assert torch.equal(parts, got) and torch.equal(st2, st), "two calls"
    if (width + shift + pad) % 4 == 0 and shift % 4 == 0:
        st3 = state.to(DEV)
        assert torch.equal(run(0, tokens, st3, out=wide[:, :hv * 128]), got), "out within mixed"


@pytest.mark.parametrize("tokens,at,ld", [(1, 0, 0), (65, 1024, 0), (300, 128, 0), (300, 512, 1024), (65, 1536, 0)])
def test_delta_rule_prefill_out_over_mixed_by_address(tokens, at, ld):
    """``out`` as a tensor of another storage over ``mixed``'s memory: inside its columns, one row and
    several, with a stride of its own (``ld``), and beside it in a wider buffer."""
    hk, hv = 2, 4
    mixed, ab, A_log, dt_bias, state = _delta_case(tokens, seed=tokens + at, hk=hk, hv=hv)
    width = mixed.shape[1]
    buf = torch.zeros((tokens + 1, width + hv * 128), dtype=torch.bfloat16, device=DEV)
    rows = buf[:tokens, :width]
    rows.copy_(mixed)
    args = [t.to(DEV) for t in (ab, A_log, dt_bias)]

    def run(st, **kw):
        return delta_rule_prefill(rows, args[0][:, :hv], args[0][:, hv:], args[1], args[2], st, num_k_heads=hk, **kw)

    st, st2 = state.to(DEV), state.to(DEV)
    want = run(st)
    out = torch.as_strided(buf, (tokens, hv * 128), (ld or buf.stride(0), 1), at)
    out = torch.from_dlpack(out)
    assert out.untyped_storage().data_ptr() != buf.untyped_storage().data_ptr() or at == 0
    assert torch.equal(run(st2, out=out), want) and torch.equal(st2, st)


def test_gated_rms_norm_rows():
    gen = torch.Generator().manual_seed(9)
    tokens, heads = 70, 32
    x = torch.randn((tokens, heads * 128), generator=gen).to(torch.bfloat16)
    zw = torch.randn((tokens, heads * 128 + 64), generator=gen).to(torch.bfloat16)
    w = (1.0 + 0.02 * torch.randn(128, generator=gen)).to(torch.bfloat16)
    got = gated_rms_norm_rows(x.to(DEV), zw.to(DEV)[:, 64:], w.to(DEV), 1e-6)
    want = gated_rms_norm(x.reshape(-1, 128), zw[:, 64:].reshape(-1, 128), w, 1e-6).reshape(tokens, -1)
    close(got, want, what="gated norm rows")


@pytest.mark.parametrize("tokens,heads,shift,pad", [(1, 1, 0, 0), (3, 5, 0, 0), (5, 3, 2, 0), (16, 1, 0, 2), (17, 32, 8, 8)])
def test_gated_rms_norm_rows_edges(tokens, heads, shift, pad):
    """Heads that leave a workgroup's last groups empty, and rows that allow only 4-byte accesses."""
    gen = torch.Generator().manual_seed(tokens + heads)
    x, z = (torch.randn((tokens, heads * 128), generator=gen).to(torch.bfloat16) for _ in range(2))
    w = (1.0 + 0.02 * torch.randn(128, generator=gen)).to(torch.bfloat16)

    def wide(t):
        v = torch.zeros((tokens, t.shape[1] + shift + pad), dtype=t.dtype, device=DEV)[:, shift:shift + t.shape[1]]
        return v.copy_(t)

    got = gated_rms_norm_rows(wide(x), wide(z), w.to(DEV), 1e-6, out=wide(torch.zeros_like(x)))
    want = gated_rms_norm(x.reshape(-1, 128), z.reshape(-1, 128), w, 1e-6).reshape(tokens, -1)
    close(got, want, what="gated norm rows", flip_frac=1e-3)


def test_gated_rms_norm_rows_gate_is_fp32():
    """The gate's SiLU goes into the product unrounded, so results are compared with the product in 64
    bits, rounded once. x is +-1 and eps 0, so that the norm is x itself; a head has one z, all of a
    weight's mantissas. z is every bf16 from -80 to 1e38. The gate is off by 3 x 2^-23 at most (2 for e^-z,
    half for 1 + e^-z, half for the quotient), the product by 2^-24: a result may round the other way only
    that near to the middle of two bf16."""
    bits = torch.arange(1 << 16, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    z = bits[(bits.float() >= -80) & (bits.float() <= 1e38) & (bits.float().abs() > 1e-30)]
    z = torch.cat([z, z[:-z.numel() % 32]]).reshape(-1, 32, 1).expand(-1, 32, 128).reshape(-1, 32 * 128)
    x = torch.where(torch.arange(z.shape[1]) % 3 == 0, -1.0, 1.0).to(torch.bfloat16).expand(z.shape).contiguous()
    w = (1 + torch.arange(128) / 128).to(torch.bfloat16)
    got = gated_rms_norm_rows(x.to(DEV), z.to(DEV), w.to(DEV), 0.0).cpu()
    z64 = z.double()
    want = x.double() * w.double().repeat(32) * (z64 / (1 + torch.exp(-z64)))
    off = (got.double() - want).abs()
    spacing = 2.0 ** (torch.floor(torch.log2(want.abs())) - 7)  # of bf16 at want
    wrong = off > 0.5 * spacing + 3.5 * 2.0**-23 * want.abs()
    assert not wrong.any(), f"{int(wrong.sum())} results, z from {float(z[wrong].min())} to {float(z[wrong].max())}"


def test_gated_rms_norm_rows_gate_of_zeros_infinities_and_nan():
    """Each element's own: SiLU keeps a zero's sign and +inf, and has no value at -inf (0 times inf)."""
    inf, nan = float("inf"), float("nan")
    z = torch.tensor([0.0, -0.0, inf, -inf, nan, 3e38, -3e38, 1.0], dtype=torch.bfloat16).repeat(16).reshape(1, 128)
    ones = torch.ones((1, 128), dtype=torch.bfloat16, device=DEV)
    got = gated_rms_norm_rows(ones, z.to(DEV), ones[0].contiguous(), 0.0).cpu().float()[0, :8]
    assert got[0] == 0 and got[1] == 0 and torch.signbit(got[:2]).tolist() == [False, True]
    assert got[2] == inf and torch.isnan(got[3:5]).all()
    assert got[5] == z[0, 5].float() and abs(got[6]) < 2e-37 and got[7] == torch.tensor(0.7310586).bfloat16().float()


@pytest.mark.parametrize("tokens,hq,hkv,half,pos0,shift", [
    (1, 4, 1, 4, 0, 0), (3, 4, 1, 8, 5, 4), (7, 8, 2, 16, 30000, 0), (9, 4, 1, 32, 11, 0), (5, 12, 3, 128, 2, 4),
    (2047, 4, 1, 32, 0, 0), (2049, 4, 1, 32, 3, 0)])
def test_qk_norm_rope_prefill_edges(tokens, hq, hkv, half, pos0, shift):
    """Rotations from 8 dims to the whole head, tokens on both sides of the workgroup's change
    from one to four with a remainder, and rows that allow only 8-byte accesses."""
    from deltaforge_amd.prefill import qk_norm_rope_prefill
    print(f"qk edges {tokens} {hq} {hkv} {half} {pos0} {shift}", flush=True)
    gen = torch.Generator().manual_seed(tokens + half)
    kc, vc = hq * 512, hq * 512 + hkv * 256
    proj = torch.randn((tokens, vc + hkv * 256), generator=gen).to(torch.bfloat16)
    qn, kn = ((0.1 * torch.randn(256, generator=gen)).to(torch.bfloat16) for _ in range(2))
    inv = 10000.0 ** (-torch.arange(half) / half)
    wide = torch.zeros((tokens, proj.shape[1] + shift), dtype=torch.bfloat16, device=DEV)[:, shift:].copy_(proj)
    k_cache, v_cache = (torch.zeros((hkv, pos0 + tokens + 1, 256), dtype=torch.bfloat16, device=DEV) for _ in range(2))
    q = qk_norm_rope_prefill(wide, qn.to(DEV), kn.to(DEV), inv.to(DEV), k_cache, v_cache, num_q_heads=hq, k_col=kc,
                             v_col=vc, pos0=pos0)
    bf = lambda t: t.to(torch.bfloat16).float()
    ang = (pos0 + torch.arange(tokens, dtype=torch.float32)).unsqueeze(1) * inv
    c, s = (bf(f(torch.cat([ang, ang], -1))).unsqueeze(1) for f in (torch.cos, torch.sin))

    def want(x, w):
        x = x.float()
        n = bf(x * torch.rsqrt(x.double().pow(2).mean(-1, keepdim=True) + 1e-6).float() * (1 + w.float()))
        r = n[..., :2 * half]
        rotated = torch.cat([-r[..., half:], r[..., :half]], -1)
        return torch.cat([bf(bf(r * c) + bf(rotated * s)), n[..., 2 * half:]], -1)

    close(q, want(proj[:, :kc].reshape(tokens, hq, 512)[..., :256], qn), what="queries", flip_frac=1e-3)
    k = want(proj[:, kc:vc].reshape(tokens, hkv, 256), kn).transpose(0, 1)
    close(k_cache[:, pos0:-1], k, what="keys", flip_frac=1e-3)
    assert torch.equal(v_cache[:, pos0:-1].cpu(), proj[:, vc:].reshape(tokens, hkv, 256).transpose(0, 1)), "values"
    for cache in (k_cache, v_cache):
        assert not cache[:, :pos0].any() and not cache[:, -1].any(), "other rows"


def _attention_expression(q, k, v, gate, pos0, scale, swish):
    """The reference's rounding in fp32: bf16 scores, bf16 softmax, bf16 output, bf16 gate."""
    p, hq, _ = q.shape
    out = torch.empty((p, hq, 256))
    keep = torch.arange(pos0 + p)[None] <= pos0 + torch.arange(p)[:, None]
    for h in range(hq):
        kk, vv = k[h // 4, :pos0 + p].float(), v[h // 4, :pos0 + p].float()
        s = ((q[:, h].float() @ kk.t()).to(torch.bfloat16).float() * scale).to(torch.bfloat16).float()
        w = torch.softmax(s.masked_fill(~keep, float("-inf")), -1).to(torch.bfloat16).float()
        out[:, h] = (w @ vv).to(torch.bfloat16).float()
    g = gate.float()
    g = (g * torch.sigmoid(g) if swish else torch.sigmoid(g)).to(torch.bfloat16).float()
    return (out * g).to(torch.bfloat16).reshape(p, -1)


# row blocks of 32 positions, key blocks of 64 in two sets of 32, the first 32 positions, later
# chunks; a scale that is no power of two, zero or negative (a masked key stays masked); gate and output
# rows that allow no 8-byte access
@pytest.mark.parametrize("tokens,pos0,scale,swish,shift", [
    (1, 0, 1 / 16, False, 0), (31, 0, 1 / 16, True, 0), (33, 0, 0.07, False, 0), (64, 0, 1 / 16, False, 1),
    (97, 0, 0.05, True, 3), (1, 31, 1 / 16, False, 0), (2, 31, 1 / 16, False, 0), (40, 30, 1 / 16, False, 0),
    (1, 64, 1 / 16, False, 0), (70, 200, 1 / 16, False, 2), (130, 63, 0.3, False, 0), (97, 0, -0.05, False, 0),
    (40, 30, 0.0, False, 0), (130, 63, -1 / 16, True, 2)])
def test_attention_prefill_edges(tokens, pos0, scale, swish, shift):
    print(f"attention prefill {tokens} at {pos0}", flush=True)
    from deltaforge_amd import prefill as P

    gen = torch.Generator().manual_seed(1000 * tokens + pos0)
    max_len = pos0 + tokens + 5
    q = torch.randn((tokens, 8, 256), generator=gen).to(torch.bfloat16)
    k, v = (torch.randn((2, max_len, 256), generator=gen).to(torch.bfloat16) for _ in range(2))
    k[:, pos0 + tokens:], v[:, pos0 + tokens:] = float("nan"), float("nan")  # rows past the prompt are not read
    wide = torch.randn((tokens, shift + 8 * 512), generator=gen).to(torch.bfloat16)
    gate = wide[:, shift:]
    kd, vd, qd, gd = k.to(DEV), v.to(DEV), q.to(DEV), wide.to(DEV)[:, shift:]
    out = torch.zeros((tokens, 8 * 256 + 2 * shift), dtype=torch.bfloat16, device=DEV)[:, shift:shift + 8 * 256]
    got = P.attention_prefill(qd, kd, vd, gd, gate_head_stride=512, pos0=pos0, gate_kind=int(swish), scale=scale, out=out)
    heads = torch.stack([gate[:, h * 512:h * 512 + 256] for h in range(8)], 1)
    close(got, _attention_expression(q, k, v, heads, pos0, scale, swish), what="attention", flip_frac=5e-3)
    if tokens > 1:  # later rows as a chunk of their own
        at = tokens // 3
        part = P.attention_prefill(qd[at:].contiguous(), kd, vd, gd[at:], gate_head_stride=512, pos0=pos0 + at,
                                   gate_kind=int(swish), scale=scale)
        assert torch.equal(part, got[at:])


# -- layers and the model -------------------------------------------------------------------


@pytest.fixture(scope="module")
def mid():
    cfg = mid_config(4)
    model = synth.synth_model(cfg, seed=21, symmetric=True)
    return cfg, model, oracle_for(model), Prefiller(model)


def _caches(cfg, max_len):
    out = []
    for kind in cfg.layer_types:
        if kind == FULL_ATTENTION:
            k = torch.zeros((cfg.num_key_value_heads, max_len, cfg.head_dim), dtype=torch.bfloat16, device=DEV)
            out.append({"k_cache": k, "v_cache": torch.zeros_like(k)})
        else:
            out.append({"conv_ring": torch.zeros((cfg.linear_conv_dim, 4), dtype=torch.bfloat16, device=DEV),
                        "state": torch.zeros((cfg.linear_num_value_heads, 128, 128), dtype=torch.float32,
                                             device=DEV)})
    return out


@pytest.mark.parametrize("kind", [LINEAR_ATTENTION, FULL_ATTENTION])
def test_one_layer_against_the_oracle(mid, kind):
    """One token mixer over 150 tokens (two full chunks and a partial): its output and its
    cache, from the input-normed rows."""
    cfg, model, oracle, pre = mid
    i = cfg.layer_types.index(kind)
    tokens, max_len = 150, 192
    gen = torch.Generator().manual_seed(30 + i)
    x = torch.randn((1, tokens, cfg.hidden_size), generator=gen).to(torch.bfloat16)
    ocache = oracle.new_cache(1, max_len)
    caches = _caches(cfg, max_len)
    layer = pre.layers[i]
    xd = x[0].to(DEV)
    from deltaforge_amd import prefill as P

    if kind == LINEAR_ATTENTION:
        want = oracle._delta_net(i, x, ocache.layers[i])[0]
        c = cfg
        proj = int4_gemm(xd, layer["proj"])
        conv_c, vd, hv = c.linear_conv_dim, c.linear_value_dim, c.linear_num_value_heads
        mixed = causal_conv_prefill(proj[:, :conv_c], layer["conv_w"], caches[i]["conv_ring"])
        core = delta_rule_prefill(mixed, proj[:, conv_c + vd:], proj[:, conv_c + vd + hv:], layer["A_log"],
                                  layer["dt_bias"], caches[i]["state"], num_k_heads=c.linear_num_key_heads)
        y = gated_rms_norm_rows(core, proj[:, conv_c:conv_c + vd], layer["gnorm_w"], c.rms_norm_eps)
        got = int4_gemm(y, layer["out"])
        close(got, want, what="DeltaNet layer", flip_frac=5e-3)
        _rel_close(caches[i]["state"], ocache.layers[i]["recurrent"][0], 1e-3, "recurrent state")
        ring = caches[i]["conv_ring"].cpu()
        hist = torch.stack([ring[:, (tokens - 3 + j) % 4] for j in range(3)], dim=-1)
        close(hist, ocache.layers[i]["conv"][0], what="conv history", flip_frac=1e-3)
    else:
        positions = torch.arange(tokens).unsqueeze(0)
        cos, sin = rope_cos_sin(positions, cfg, torch.bfloat16, inv_freq_dtype=torch.bfloat16)
        want = oracle._attention(i, x, cos, sin, ocache.layers[i], 0)[0]
        qd, kvd = 2 * cfg.num_attention_heads * cfg.head_dim, cfg.num_key_value_heads * cfg.head_dim
        proj = int4_gemm(xd, layer["proj"])
        q = P.qk_norm_rope_prefill(proj, layer["q_norm"], layer["k_norm"], pre.inv_freq, caches[i]["k_cache"],
                                   caches[i]["v_cache"], num_q_heads=cfg.num_attention_heads, k_col=qd,
                                   v_col=qd + kvd)
        attn = P.attention_prefill(q, caches[i]["k_cache"], caches[i]["v_cache"], proj[:, cfg.head_dim:],
                                   gate_head_stride=2 * cfg.head_dim)
        got = int4_gemm(attn, layer["out"])
        close(got, want, what="attention layer", flip_frac=5e-3)
        close(caches[i]["k_cache"][:, :tokens].cpu(), ocache.layers[i]["keys"][0, :, :tokens], what="k cache",
              flip_frac=1e-3)
        close(caches[i]["v_cache"][:, :tokens].cpu(), ocache.layers[i]["values"][0, :, :tokens], what="v cache",
              flip_frac=1e-3)


@pytest.mark.parametrize("tokens", [1, 100])
def test_prefill_logits_and_caches_match_the_oracle_forward(mid, tokens):
    cfg, model, oracle, pre = mid
    prompt = synth.prompt_ids(cfg.vocab_size, tokens, seed=40 + tokens)
    ocache = oracle.new_cache(1, 128)
    with torch.no_grad():
        want = oracle.forward(prompt, ocache)[:, -1]
    caches = _caches(cfg, 128)
    got = pre.forward(prompt[0].to(DEV), caches)
    kl, agree = kl_and_agreement(want.float().unsqueeze(1), got.float().cpu().unsqueeze(1))
    print(f"prefill P={tokens}: KL {float(kl.mean()):.3e}, top-1 agrees {bool(agree.all())}", flush=True)
    assert float(kl.mean()) < 1e-3 and bool(agree.all())
    for i, kind in enumerate(cfg.layer_types):
        # a deeper layer's input has passed through earlier layers whose bf16 outputs differ
        # from the oracle's by summation-order ulps, so its caches are held normwise (the largest
        # error against the largest value); the single-layer test holds them elementwise
        if kind == FULL_ATTENTION:
            _rel_close(caches[i]["k_cache"][:, :tokens], ocache.layers[i]["keys"][0, :, :tokens], 2e-2,
                       f"layer {i} keys")
            _rel_close(caches[i]["v_cache"][:, :tokens], ocache.layers[i]["values"][0, :, :tokens], 2e-2,
                       f"layer {i} values")
        else:
            _rel_close(caches[i]["state"], ocache.layers[i]["recurrent"][0], 2e-2, f"layer {i} state")


def _teacher_forced(dec, ref_tokens):
    got = [dec.logits.float().cpu().clone()]
    for t in range(ref_tokens.shape[1] - 1):
        dec.tokens.copy_(ref_tokens[:, t].to(DEV))  # teacher forcing with the oracle's continuation
        dec.decode(1)
        dec.check()
        got.append(dec.logits.float().cpu().clone())
    return torch.stack(got, dim=1)


def test_filled_persistent_decoder_continues_like_the_oracle(mid):
    """The same decoder, prefilled token by token (its own launch) and by ``Prefiller.fill``,
    teacher-forced through the oracle's greedy continuation. The filled one must agree on top-1
    and stay within twice the own-prefill decoder's KL (this symmetric-weight model's noise
    floor against the oracle), or 1e-3 if that is larger."""
    cfg, model, oracle, pre = mid
    prompt = synth.prompt_ids(cfg.vocab_size, 90, seed=50)
    with torch.no_grad():
        ref_tokens, ref_logits = oracle.greedy(prompt, 8)
    own = PersistentDecoder(model, max_seq_len=128, max_new_tokens=16)
    own.prefill(prompt.to(DEV))
    own.check()
    kl_own, agree_own = kl_and_agreement(ref_logits.float(), _teacher_forced(own, ref_tokens))
    dec = PersistentDecoder(model, max_seq_len=128, max_new_tokens=16)
    pre.fill(dec, prompt.to(DEV))
    kl, agree = kl_and_agreement(ref_logits.float(), _teacher_forced(dec, ref_tokens))
    print(f"own prefill: agreement {float(agree_own.float().mean()):.4f}, KL {float(kl_own.mean()):.3e}; "
          f"filled: agreement {float(agree.float().mean()):.4f}, KL {float(kl.mean()):.3e}", flush=True)
    assert float(kl.mean()) < max(1e-3, 2 * float(kl_own.mean()))
    assert float(agree.float().mean()) >= min(7 / 8, float(agree_own.float().mean()))


def test_fill_in_chunks_equals_one_pass(mid):
    """``Prefiller.fill`` runs a long prompt in chunks (positions continuing from the caches).
    With chunk boundaries on the delta rule's 64-token chunks the arithmetic is the single
    pass's, so 200 tokens filled 64 at a time must leave bit-identical caches, logits and first
    token; chunk sizes off that grid are refused."""
    cfg, model, oracle, pre = mid
    prompt = synth.prompt_ids(cfg.vocab_size, 200, seed=60).to(DEV)
    one = PersistentDecoder(model, max_seq_len=256, max_new_tokens=16)
    pre.fill(one, prompt)
    parts = PersistentDecoder(model, max_seq_len=256, max_new_tokens=16)
    pre.fill(parts, prompt, chunk=64)
    torch.cuda.synchronize()
    for i, (a, b) in enumerate(zip(one.layer_state, parts.layer_state)):
        for name in a:
            assert torch.equal(a[name], b[name]), f"layer {i} {name}"
    assert torch.equal(one.logits, parts.logits) and torch.equal(one.tokens, parts.tokens)
    assert int(parts.position.item()) == 200
    for bad in (32, 100, 65536):
        with pytest.raises(ValueError):
            pre.fill(parts, prompt, chunk=bad)
